// Scores off the grid, with their gradients, for refining docked poses.  The reference
// has no counterpart; these kernels extend its score (src/fft_process.cpp:333-446).
//
// 1. Spectral score at a continuous translation.  With Q the Hermitian fold of
//    conj(R^) L^ for one rotation (kz <= nf/2 stored), signed frequencies k' (k' = k for
//    k < nf/2, else k - nf) and phase phi = 2 pi k'.t / nf,
//        s(t) = 1/nf^3 sum_{kz <= nf/2} w(kz) Re[Q(k) e^{i phi}],  w = 1 at kz = 0, nf/2, else 2,
//    which equals the reported score value/nf^3 at every grid point t, and
//        ds/dt_a = 1/nf^3 sum w(kz) (-2 pi k'_a / nf) Im[Q(k) e^{i phi}].
// 2. Companion score of a pose with trilinear interpolation of the receptor grids: with
//    the ligand atom a rotated about the ligand centre, X_a = R (a - c), placed at
//    P_a = X_a - gw t' (t' the signed translation in voxels, as decoygen places poses),
//        s = sum_a [ w_a Rr(P_a) + q_a Ri(P_a) ],   w_a = (4/3) pi r_a^3 / gw^3,
//    where Rr, Ri are the receptor's shape and electrostatic grids (voxel i at
//    gw (i + 1/2 - ng/2), zero outside).  The atom adjoint is g_a = ds/dP_a; from it
//    ds/dt' = -gw sum_a g_a and, for a rotation R -> exp([w]x) R, ds/dw = sum_a X_a x g_a.
//    This spreads each atom trilinearly instead of over its voxel sphere: a smooth
//    companion of the hard voxelizer, recomputed per call, never stored.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "mdk_internal.h"

namespace {

__device__ __forceinline__ int signed_freq(int k, int nf) { return k < nf / 2 ? k : k - nf; }

// phases e^{2 pi i k' t_a / nf} of pose b: ph[b][a][k]
__global__ void __launch_bounds__(256) k_spec_phase(const float *__restrict__ tq, float2 *__restrict__ ph, int nf) {
    const int b = blockIdx.x;
    for (int q = threadIdx.x; q < 3 * nf; q += 256) {
        const int a = q / nf, k = q - a * nf;
        double sn, cs;
        sincos(2.0 * M_PI * signed_freq(k, nf) / nf * tq[3 * b + a], &sn, &cs);
        ph[(size_t)b * 3 * nf + q] = make_float2((float)cs, (float)sn);
    }
}

// trilinear value and gradient (per unit of u) of the two receptor grids at voxel
// coordinate u; corners outside the grid count as 0, and all is NaN where u has a NaN
__device__ __forceinline__ void trilinear(const float2 *__restrict__ rg, int ng, float ux, float uy, float uz,
                                          float2 &val, float2 &dx, float2 &dy, float2 &dz) {
    // a position with no corner in the grid counts as one just outside it; one that is not a number
    // does too, for its loads, and makes the weights NaN (0 would be the score of a ligand outside)
    const float hi = (float)ng + 1.0f, nan = ux != ux || uy != uy || uz != uz ? NAN : 0.0f;
    if (!(ux > -2.0f && ux < hi && uy > -2.0f && uy < hi && uz > -2.0f && uz < hi)) ux = uy = uz = -2.0f;
    const float fx0 = floorf(ux), fy0 = floorf(uy), fz0 = floorf(uz);
    const int i0 = (int)fx0, j0 = (int)fy0, k0 = (int)fz0;
    const float fx = ux - fx0 + nan, fy = uy - fy0 + nan, fz = uz - fz0 + nan;
    val = dx = dy = dz = make_float2(0.f, 0.f);
    // the corners' loads are issued together (a corner outside the grid loads a voxel inside and
    // counts as 0); with a branch around each, they came one after another
    float2 corner[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int i = i0 + (c >> 2), j = j0 + ((c >> 1) & 1), k = k0 + (c & 1);
        const bool in = i >= 0 && i < ng && j >= 0 && j < ng && k >= 0 && k < ng;
        const int at = in ? (i * ng + j) * ng + k : 0;
        const float2 g = rg[at];
        corner[c] = in ? g : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int di = c >> 2, dj = (c >> 1) & 1, dk = c & 1;
        const float2 g = corner[c];
        const float wx = di ? fx : 1.f - fx, wy = dj ? fy : 1.f - fy, wz = dk ? fz : 1.f - fz;
        const float sx = di ? 1.f : -1.f, sy = dj ? 1.f : -1.f, sz = dk ? 1.f : -1.f;
        const float w = wx * wy * wz, ax = sx * wy * wz, ay = wx * sy * wz, az = wx * wy * sz;
        val.x += w * g.x;
        val.y += w * g.y;
        dx.x += ax * g.x;
        dx.y += ax * g.y;
        dy.x += ay * g.x;
        dy.y += ay * g.y;
        dz.x += az * g.x;
        dz.y += az * g.y;
    }
}

// Sums v[0..K) over a workgroup of NT threads in a fixed order: within each wavefront by halving
// strides, then over the wavefronts; the result is in thread 0.
template <int K, int NT> __device__ __forceinline__ void block_sum(double *v) {
    __shared__ double part[NT / 64][K];
#pragma unroll
    for (int a = 0; a < K; a++)
        for (int h = 32; h >= 1; h >>= 1) v[a] += __shfl_down(v[a], h, 64);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int a = 0; a < K; a++) part[threadIdx.x >> 6][a] = v[a];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < NT / 64; w++)
#pragma unroll
            for (int a = 0; a < K; a++) v[a] += part[w][a];
}

// out[b][0..3] = (s, ds/dtx, ds/dty, ds/dtz) from the n partial sums of kp_x_spec, one workgroup a
// pose; added in a fixed order
__global__ void __launch_bounds__(256) k_spec_finish(const double *__restrict__ part, float *__restrict__ out, int n,
                                                     int nf) {
    const double *p = part + (size_t)blockIdx.x * n * 4;
    double s[4] = {0, 0, 0, 0};
    for (int k = threadIdx.x; k < n; k += 256)
#pragma unroll
        for (int a = 0; a < 4; a++) s[a] += p[4 * k + a];
    block_sum<4, 256>(s);
    if (threadIdx.x == 0) {
        const double n3 = (double)nf * nf * nf, g = -2.0 * M_PI / nf / n3;
        float *o = out + 4 * (size_t)blockIdx.x;
        o[0] = (float)(s[0] / n3);
        for (int a = 1; a < 4; a++) o[a] = (float)(s[a] * g);
    }
}

// Sums of a pose, out[b][7] = (s, ds/dt'(3), ds/dw(3)), one workgroup a pose and one launch a call (with
// eight workgroups a pose, their partial sums and a second kernel, in batches of the context's size, 2000
// poses of 2081 atoms took 16 times two copies in, two kernels (13 and 4 us) and a copy out).  The atoms
// of a large ligand go to a workgroup by parts, and k_companion_finish adds these in their order.
__global__ void __launch_bounds__(256) k_companion(LigandDev L, const float *__restrict__ wshape,
                                                   const float2 *__restrict__ rg, const float *__restrict__ rot,
                                                   const float *__restrict__ tq, int nf, int parts,
                                                   double *__restrict__ part, float *__restrict__ out) {
    const int b = blockIdx.x, tid = threadIdx.x;
    float r[9];
    for (int q = 0; q < 9; q++) r[q] = rot[9 * b + q];
    float t3[3];
    for (int a = 0; a < 3; a++) {
        const float t = tq[3 * b + a];
        t3[a] = t < 0.5f * nf ? t : t - nf;  // signed translation (voxels)
    }
    const int ng = L.ng, len = ((L.na + parts - 1) / parts + 255) / 256 * 256;
    const float gw = L.gw, h = 0.5f * ng - 0.5f;
    const int p = blockIdx.y;
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int a = p * len + tid; a < min(L.na, (p + 1) * len); a += 256) {
        const float x = L.xyz[3 * a] - L.cx, y = L.xyz[3 * a + 1] - L.cy, z = L.xyz[3 * a + 2] - L.cz;
        const float X = r[0] * x + r[1] * y + r[2] * z;
        const float Y = r[3] * x + r[4] * y + r[5] * z;
        const float Z = r[6] * x + r[7] * y + r[8] * z;
        const float Px = X - gw * t3[0], Py = Y - gw * t3[1], Pz = Z - gw * t3[2];
        float2 val, dx, dy, dz;
        trilinear(rg, ng, Px / gw + h, Py / gw + h, Pz / gw + h, val, dx, dy, dz);
        const float ws = wshape[a], q = L.charge[a];
        const float s = ws * val.x + q * val.y;
        // g = ds/dP (per Angstrom)
        const float gx = (ws * dx.x + q * dx.y) / gw, gy = (ws * dy.x + q * dy.y) / gw, gz = (ws * dz.x + q * dz.y) / gw;
        acc[0] += s;
        acc[1] += -gw * gx;
        acc[2] += -gw * gy;
        acc[3] += -gw * gz;
        acc[4] += Y * gz - Z * gy;
        acc[5] += Z * gx - X * gz;
        acc[6] += X * gy - Y * gx;
    }
    block_sum<7, 256>(acc);
    if (tid == 0)
        for (int a = 0; a < 7; a++) {
            if (parts > 1)
                part[((size_t)b * parts + p) * 7 + a] = acc[a];
            else
                out[7 * (size_t)b + a] = (float)acc[a];
        }
}

__global__ void k_companion_finish(const double *__restrict__ part, float *__restrict__ out, int n, int parts) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x, b = q / 7, a = q - 7 * b;
    if (q >= n) return;
    double sum = 0;
    for (int p = 0; p < parts; p++) sum += part[((size_t)b * parts + p) * 7 + a];
    out[q] = (float)sum;
}

// Parts of a ligand's sums: up to sixteen of about 1024 atoms or more, from 2560 atoms on.  A call of
// one pose takes 28, 38, 48, 73 and 197 us with one workgroup and 336, 2081, 4000, 8000 and 30000
// atoms, and 34, 36 and 43 us with the last three in parts.
int companion_parts(int na) { return na < 2560 ? 1 : std::min(16, (na + 1023) / 1024); }
// Partial sums of one launch, and so poses times parts.  With one workgroup going through all parts of a pose
// instead, 300 poses of 4000, 8000 and 30000 atoms (the last at 256^3) take 65, 102 and 625 us in
// place of 56, 86 and 418, 1000 poses 131, 223 and 1356 in place of 131, 220 and 1310, 10000 poses of 2600
// atoms 671 in place of 658.
constexpr int kParts = 65536;

}  // namespace

hipError_t launch_spec_phase(const float *t_dev, int B, int nf, float2 *ph, hipStream_t s) {
    k_spec_phase<<<B, 256, 0, s>>>(t_dev, ph, nf);
    return hipGetLastError();
}

hipError_t launch_spec_finish(const double *part, int B, int n, int nf, float *out_dev, hipStream_t s) {
    k_spec_finish<<<B, 256, 0, s>>>(part, out_dev, n, nf);
    return hipGetLastError();
}

size_t companion_scratch_doubles(int na) { return companion_parts(na) > 1 ? (size_t)kParts * 7 : 0; }

hipError_t launch_companion(const LigandDev &lig, const float *wshape, const float2 *recgrid, const float *rot_dev,
                            const float *t_dev, int B, int nf, double *part, float *out_dev, hipStream_t s) {
    const int parts = companion_parts(lig.na), most = parts > 1 ? kParts / parts : B;
    for (int b0 = 0; b0 < B; b0 += most) {
        const int n = std::min(most, B - b0);
        float *o = out_dev + 7 * (size_t)b0;
        k_companion<<<dim3(n, parts), 256, 0, s>>>(lig, wshape, recgrid, rot_dev + 9 * (size_t)b0, t_dev + 3 * (size_t)b0, nf,
                                                   parts, part, o);
        if (parts > 1) k_companion_finish<<<(7 * n + 255) / 256, 256, 0, s>>>(part, o, 7 * n, parts);
    }
    return hipGetLastError();
}
