// Ligand voxelization on the device, bit-exact with the reference's CPU voxelizer
// (src/ligand.cpp:20-261, src/docking.cpp:368-396).
//
// Built with -ffp-contract=off: every float expression rounds after each operation in
// the same order as the reference's x86-64 build (no FMA), so rotated coordinates,
// squared distances and voxel indices are identical.
//
// The reference's sequential sweeps are restated as order-free rules:
//   core[v]   = some atom has (xd+yd)+zd < 1.5 r^2 in its 5^3 box      (ligand.cpp:68-101)
//   scraped   = interior(v) & core[v] & some 6-neighbour not core      (ligand.cpp:110-134;
//               the sweep tests ==0 on values it never turns into 0, so it does not cascade)
//   grid_r[v] = core & !scraped ? delta : (surf[v] ? 1 : 0)             (ligand.cpp:140-173)
//   delta != 1: interior delta voxels with a 0 neighbour become 1       (ligand.cpp:176-195;
//               again non-cascading because delta != 0 and 1 != 0)
//   grid_i[v] = charges of the atoms nearest to v, summed in atom order (ligand.cpp:212-235)
// delta == 0 makes the last rule order-dependent; the host rejects it.
//
// Representation handed to the FFT passes (VoxGrid): per rotation, a bit mask of the
// voxels whose shape value is delta (D) and of those whose value is 1 (O), each row
// (i, j) of ng voxels in its own rw = ceil(ng/32) words, and a dense float charge grid.
// The rules above become word-wide bit operations over rows; the charge grid and the
// per-voxel atom counts are kept all-zero between batches (their consumers clear what
// they read), so a batch writes only the voxels its atoms touch.
#pragma clang fp contract(off)

#include <algorithm>

#include "mdk_internal.h"

namespace {

__device__ __forceinline__ void rotate_atom(const LigandDev &L, const float *r, int l, float &X,
                                            float &Y, float &Z) {
    const float x = L.xyz[3 * l] - L.cx;
    const float y = L.xyz[3 * l + 1] - L.cy;
    const float z = L.xyz[3 * l + 2] - L.cz;
    X = r[0] * x + r[1] * y + r[2] * z;
    Y = r[3] * x + r[4] * y + r[5] * z;
    Z = r[6] * x + r[7] * y + r[8] * z;
}

// Planes (atom's voxel) + d0 .. + d1 - 1 of atom l's box, -2 <= d0 < d1 <= 3: its core/surface bits
// into cb/sb (LDS masks of the grid's planes i0 .. i1 - 1); gc: the grid's coordinates.  Bound by its
// vector instructions (the LDS form has one workgroup's waves on one CU): the box's ten squared
// coordinate differences are formed once, the tests of a row gather into five bits, and a row's
// run is those bits shifted into the word of the box's first column.
__device__ __forceinline__ void vox_planes(const LigandDev &L, const float *gc, float X, float Y, float Z, int l, int d0,
                                           int d1, uint32_t *cb, uint32_t *sb, int i0, int i1) {
    const int ng = L.ng, rw = row_words(ng);
    const float h = (float)(ng / 2);
    // (a voxel far outside has the same empty box as one 3 outside)
    const int i2 = min(max((int)(X / L.gw + h), -3), ng + 2);
    const int j2 = min(max((int)(Y / L.gw + h), -3), ng + 2);
    const int k2 = min(max((int)(Z / L.gw + h), -3), ng + 2);
    const int ka = max(k2 - 2, 0), kn = min(k2 + 3, ng) - ka;  // the box's columns: ka .. ka + kn - 1
    const uint32_t inside = kn > 0 ? (1u << kn) - 1u : 0u;
    const float rc2 = L.rc2[l], rs2 = L.rs2[l];
    float y2[5], z2[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {  // outside the grid: any coordinate, not used below
        const int j = min(max(j2 - 2 + q, 0), ng - 1), k = min(ka + q, ng - 1);
        const float dy = Y - gc[j], dz = Z - gc[k];
        y2[q] = dy * dy;
        z2[q] = dz * dz;
    }
    const int w = ka >> 5, sh = ka & 31;
    for (int di = d0; di < d1; di++) {
        const int i = i2 + di;
        if (i < i0 || i >= i1) continue;
        const float dx = X - gc[i];
        const float xd = dx * dx;
        if (xd > rc2) continue;  // rs2 <= rc2, so neither sphere reaches this plane
        const int row0 = ((i - i0) * ng + j2 - 2) * rw + w;
#pragma unroll
        for (int p = 0; p < 5; p++) {
            const int j = j2 - 2 + p;
            const float d2 = xd + y2[p];
            if (j < 0 || j >= ng || d2 > rc2) continue;
            // each voxel is tested exactly as the reference does; the hits along k form one run
            // per sphere (d3 grows away from the atom)
            uint32_t c = 0, s = 0;
#pragma unroll
            for (int q = 4; q >= 0; q--) {
                const float d3 = d2 + z2[q];
                c = c + c + (d3 < rc2 ? 1u : 0u);
                s = s + s + (d3 < rs2 ? 1u : 0u);
            }
            c &= inside;
            s &= inside;
            if (c == 0) continue;  // rs2 <= rc2
            c = (c | (0u - c)) & (0xffffffffu >> __clz(c));
            atomicOr(&cb[row0 + p * rw], c << sh);
            if (sh > 27 && c >> (32 - sh)) atomicOr(&cb[row0 + p * rw + 1], c >> (32 - sh));
            if (s == 0) continue;
            s = (s | (0u - s)) & (0xffffffffu >> __clz(s));
            atomicOr(&sb[row0 + p * rw], s << sh);
            if (sh > 27 && s >> (32 - sh)) atomicOr(&sb[row0 + p * rw + 1], s >> (32 - sh));
        }
    }
}

// the voxel that holds an atom's charge
__device__ __forceinline__ int charge_row(const LigandDev &L, float X) {
    return max(0, min(L.ng - 1, (int)((X + L.pad) / L.gw)));
}
__device__ __forceinline__ int charge_voxel(const LigandDev &L, float X, float Y, float Z) {
    return (charge_row(L, X) * L.ng + charge_row(L, Y)) * L.ng + charge_row(L, Z);
}

// bits k = 32 w + s of word w with lo <= k <= hi
__device__ __forceinline__ uint32_t range_bits(int w, int lo, int hi) {
    const int a = max(lo - 32 * w, 0), e = min(hi - 32 * w, 31);
    if (a > e) return 0u;
    const uint32_t upto = (e == 31) ? 0xffffffffu : ((1u << (e + 1)) - 1u);
    return upto & (0xffffffffu << a);
}

struct MaskRows {
    const uint32_t *m;  // from plane i0 on
    int ng, rw, i0;
    // word w of row (i, j); zero outside the grid
    __device__ __forceinline__ uint32_t at(int i, int j, int w) const {
        if (i < 0 || i >= ng || j < 0 || j >= ng || w < 0 || w >= rw) return 0u;
        return m[((i - i0) * ng + j) * rw + w];
    }
};

// core after the scrape step, word w of row (i, j)
__device__ __forceinline__ uint32_t core2_word(const MaskRows &C, int i, int j, int w) {
    const int ng = C.ng;
    const uint32_t c = C.at(i, j, w);
    if (i < 1 || i > ng - 2 || j < 1 || j > ng - 2 || c == 0u) return c;
    const uint32_t zm = (c << 1) | (C.at(i, j, w - 1) >> 31);  // bit k: voxel k-1 is core
    const uint32_t zp = (c >> 1) | (C.at(i, j, w + 1) << 31);  // bit k: voxel k+1 is core
    const uint32_t closed = zm & zp & C.at(i, j - 1, w) & C.at(i, j + 1, w) & C.at(i - 1, j, w) & C.at(i + 1, j, w);
    return c & ~(range_bits(w, 1, ng - 2) & ~closed);
}

// word q of the delta mask D and the value-1 mask O of one rotation from its core (C) and
// surface (S) bits
__device__ __forceinline__ void vox_mask_word(const MaskRows &C, const MaskRows &S, int q, int ng, float delta,
                                              uint32_t &dq, uint32_t &oq) {
    const int rw = C.rw;
    const int w = q % rw, row = q / rw, i = row / ng, j = row - i * ng;
    uint32_t d = core2_word(C, i, j, w);
    uint32_t o = ~d & S.at(i, j, w);
    if (delta != 1.0f && i >= 1 && i <= ng - 2 && j >= 1 && j <= ng - 2) {
        // interior delta voxels next to a voxel of value 0 (neither core nor surface) become 1
        auto zero = [&](int ii, int jj, int ww) { return ~core2_word(C, ii, jj, ww) & ~S.at(ii, jj, ww); };
        const uint32_t z0 = zero(i, j, w);
        const uint32_t zm = (z0 << 1) | (zero(i, j, w - 1) >> 31);
        const uint32_t zp = (z0 >> 1) | (zero(i, j, w + 1) << 31);
        const uint32_t nb = zm | zp | zero(i, j - 1, w) | zero(i, j + 1, w) | zero(i - 1, j, w) | zero(i + 1, j, w);
        const uint32_t to1 = d & range_bits(w, 1, ng - 2) & nb;
        d &= ~to1;
        o |= to1;
    }
    dq = d;
    oq = o;
}

// Charges of the atoms nearest to each voxel, summed in atom order from +0.0f
// (src/ligand.cpp:216-234).  One workgroup per rotation.  With one or two atoms in a
// voxel the float sum does not depend on the order (0 + a = a and a + b = b + a
// exactly), so those are added atomically; atoms of voxels holding three or more are
// listed in LDS and each such voxel is summed in atom order by its lowest-index atom.
// Leaves the rotation's atom counts zero again.
constexpr int kChargeThreads = 1024;
constexpr int kCrowdCap = 2048;  // listed atoms of crowded voxels (beyond: global scan)

// Voxels with three or more atoms (count(v): how many of them lie in v), whose atoms are listed in
// list[0 .. *nlist), or any atoms if *nlist is above kCrowdCap: the sum in atom order
template <class Count>
__device__ __forceinline__ void vox_crowded(const int *vi, const float *__restrict__ charge, float *g, int na,
                                            const int2 *list, const int *nlist, Count count) {
    const int tid = threadIdx.x;
    const int m = *nlist;  // uniform
    if (m <= kCrowdCap) {
        for (int e = tid; e < m; e += kChargeThreads) {
            const int v = list[e].x, l = list[e].y;
            bool owner = true;
            for (int f = 0; f < m; f++)
                if (list[f].x == v && list[f].y < l) owner = false;
            if (!owner) continue;
            float sum = 0.0f;
            for (int cur = -1;;) {  // next atom of the voxel in index order
                int nxt = 0x7fffffff;
                for (int f = 0; f < m; f++)
                    if (list[f].x == v && list[f].y > cur && list[f].y < nxt) nxt = list[f].y;
                if (nxt == 0x7fffffff) break;
                sum += charge[nxt];
                cur = nxt;
            }
            g[v] = sum;
        }
    } else {
        for (int l = tid; l < na; l += kChargeThreads) {
            const int v = vi[l];
            if (count(v) <= 2) continue;
            bool owner = true;
            for (int q = 0; q < l; q++)
                if (vi[q] == v) owner = false;
            if (!owner) continue;
            float sum = 0.0f;
            for (int q = l; q < na; q++)
                if (vi[q] == v) sum += charge[q];
            g[v] = sum;
        }
    }
}

// the counts are global words of two 16-bit counts, left zero again
__global__ void __launch_bounds__(kChargeThreads)
    k_vox_charge(const int *__restrict__ vidx, uint32_t *cnt, const float *__restrict__ charge, float *chg, int na, int ng3, int cw) {
    __shared__ int nlist;
    __shared__ int2 list[kCrowdCap];  // (voxel, atom)
    const int b = blockIdx.x, tid = threadIdx.x;
    const int *vi = vidx + (size_t)b * na;
    uint32_t *cb = cnt + (size_t)b * cw;
    float *g = chg + (size_t)b * ng3;
    auto count = [&](int v) { return (cb[v >> 1] >> (16 * (v & 1))) & 0xffffu; };
    if (tid == 0) nlist = 0;
    __syncthreads();
    for (int l = tid; l < na; l += kChargeThreads) {
        const int v = vi[l];
        if (count(v) <= 2) {
            atomicAdd(&g[v], charge[l]);
        } else {
            const int k = atomicAdd(&nlist, 1);
            if (k < kCrowdCap) list[k] = make_int2(v, l);
        }
    }
    __syncthreads();
    vox_crowded(vi, charge, g, na, list, &nlist, count);
    __syncthreads();  // every count read above is done
    for (int l = tid; l < na; l += kChargeThreads) cb[vi[l] >> 1] = 0u;
}

// The same with the voxels' counts and sums in an LDS table of nt entries (a power of two, three
// times na where there is room, never less than 1.6 times): tab holds
// (voxel + 1) << 13 | atoms, 0 if free, linear probing.  One workgroup.  The global counts cost an
// atomic and a read on a line of their own for every atom, the sums another: 20 us of the 52 that
// a batch of 128 rotations of 2081 atoms took; the table takes 9.
// The slot is the leading bits of a product.  An atom's probes depend on how the factor takes to the grid's
// rows and planes: for balls of 50 to 5120 atoms on every grid from 24 to 75 they were 1.33 on average, the
// longest chain 12 on average and 48 at worst; with 2654435761 1.52, 16 and 131 (grid 75, where one
// rotation of 5100 atoms took 184 us, 171 with the counts in memory; now 121).
constexpr int kCountBits = 13, kTableMax = 8192;
__device__ __forceinline__ uint32_t table_slot(int v, int nt) { return (uint32_t)v * 0xcc9e2d51u >> (__clz(nt) + 1); }

__device__ __forceinline__ void vox_charges_lds(const int *vi, const float *__restrict__ charge, float *g, int na,
                                                uint32_t *tab, float *sum, int nt, int2 *list) {
    __shared__ int nlist;
    const int tid = threadIdx.x;
    if (tid == 0) nlist = 0;
    for (int q = tid; q < nt; q += kChargeThreads) {
        tab[q] = 0u;
        sum[q] = 0.0f;
    }
    __syncthreads();
    for (int l = tid; l < na; l += kChargeThreads) {
        const int v = vi[l];
        const uint32_t first = (uint32_t)(v + 1) << kCountBits | 1u;
        uint32_t q = table_slot(v, nt);
        for (;; q = (q + 1) & (nt - 1)) {  // a free entry is met: nt > na
            const uint32_t was = atomicCAS(&tab[q], 0u, first);
            if (was == 0u) break;
            if ((was ^ first) >> kCountBits == 0u) {
                atomicAdd(&tab[q], 1u);
                break;
            }
        }
        atomicAdd(&sum[q], charge[l]);
    }
    __syncthreads();
    bool crowd = false;
    for (int q = tid; q < nt; q += kChargeThreads) {
        const uint32_t w = tab[q], n = w & ((1u << kCountBits) - 1u);
        if (n > 2)
            crowd = true;
        else if (sum[q] != 0.0f)  // the grid is zero
            g[(w >> kCountBits) - 1] = sum[q];
    }
    if (!__syncthreads_or(crowd)) return;
    auto count = [&](int v) {
        uint32_t q = table_slot(v, nt);
        while (tab[q] >> kCountBits != (uint32_t)(v + 1)) q = (q + 1) & (nt - 1);  // v is in the table
        return tab[q] & ((1u << kCountBits) - 1u);
    };
    for (int l = tid; l < na; l += kChargeThreads) {
        const int v = vi[l];
        if (count(v) <= 2) continue;
        const int k = atomicAdd(&nlist, 1);
        if (k < kCrowdCap) list[k] = make_int2(v, l);
    }
    __syncthreads();
    vox_crowded(vi, charge, g, na, list, &nlist, count);
}

// One workgroup per rotation with its core and surface bits in LDS (grids whose masks
// fit): atom runs by LDS atomics, then the D and O words straight to dmo and, if nt > 0, the
// charges by a table of nt entries (else k_vox_charge follows).  For one rotation it is a chain of dependent steps in
// one workgroup: with a thread per atom walking five planes, the grid's coordinates loaded from
// memory inside its loops, a ligand of 336 atoms took 21.6 us and its charges a launch of 4.2 us.  Now
// 14 together.
constexpr int kVoxLdsThreads = kChargeThreads;
// Atoms up to which an atom's planes go to five threads.  One rotation of 200, 336, 512, 800 and 2081 atoms at 80^3
// takes 16.0, 21.9, 26.5, 37.0 and 88.5 us with five threads an atom, 18.6, 22.8, 25.4, 33.4 and 76.9
// with one (with the events that time it); 128 rotations 24.9, 33.0, 38.4, 56.7, 119 and 26.6, 34.4, 38.0, 54.3, 107.
constexpr int kVoxSplitAtoms = 512;
__global__ void __launch_bounds__(kVoxLdsThreads)
    k_vox_lds(LigandDev L, const float *__restrict__ rot, const int *__restrict__ boff, uint32_t *dmo, uint32_t *cnt,
              int *vidx, int mw, int cw, float *chg, int nt) {
    // [2][mw]: core, surface; then the grid's coordinates.  After the masks: the charges' table
    extern __shared__ uint32_t msk[];
    const int b = blockIdx.x, tid = threadIdx.x, ng = L.ng;
    float *gc = reinterpret_cast<float *>(msk + 2 * mw);
    for (int q = tid; q < 2 * mw; q += kVoxLdsThreads) msk[q] = 0u;
    for (int q = tid; q < ng; q += kVoxLdsThreads) gc[q] = L.gc[q];
    __shared__ float coef[9];  // read once (rot may lie in host memory)
    if (tid < 9) coef[tid] = rot[9 * ((size_t)(boff ? *boff : 0) + b) + tid];
    __syncthreads();
    float r[9];
#pragma unroll
    for (int q = 0; q < 9; q++) r[q] = coef[q];
    // an atom's five planes in one thread share its box; a small ligand's go to five threads, so
    // that the CU's four SIMDs have waves enough
    const int split = L.na <= kVoxSplitAtoms ? 5 : 1;
    for (int q = tid; q < split * L.na; q += kVoxLdsThreads) {
        const int l = q / split, d = q - split * l;
        float X, Y, Z;
        rotate_atom(L, r, l, X, Y, Z);
        vox_planes(L, gc, X, Y, Z, l, d - 2, split == 1 ? 3 : d - 1, msk, msk + mw, 0, ng);
        if (d == 0) {
            const int v = charge_voxel(L, X, Y, Z);
            vidx[(size_t)b * L.na + l] = v;
            if (nt == 0) atomicAdd(&cnt[(size_t)b * cw + (v >> 1)], 1u << (16 * (v & 1)));
        }
    }
    __syncthreads();
    const MaskRows C{msk, ng, row_words(ng), 0}, S{msk + mw, ng, row_words(ng), 0};
    uint32_t *db = dmo + (size_t)b * 2 * mw;
    for (int q = tid; q < mw; q += kVoxLdsThreads) {
        uint32_t d, o;
        vox_mask_word(C, S, q, ng, L.delta, d, o);
        db[q] = d;
        db[mw + q] = o;
    }
    if (nt == 0) return;
    __syncthreads();  // the masks are read
    vox_charges_lds(vidx + (size_t)b * L.na, L.charge, chg + (size_t)b * ng * ng * ng, L.na, msk,
                    reinterpret_cast<float *>(msk + nt), nt, reinterpret_cast<int2 *>(msk + 2 * nt));
}

// Larger grids: a workgroup takes `planes` planes of a rotation's D and O words, with the core and surface
// bits of two planes more on each side (what the rules reach) in LDS, and goes through the ligand for the
// atoms that touch them: every kSlabAtoms atoms it lists those whose box or charge lies there, then sets
// their bits.  Masks in memory (cleared, set by up to 55 atomics an atom, read back with their
// neighbours) made 768 rotations take 76.5 ms at 256^3 and 82.0 at 216^3; with slabs 71.6 and 79.0.
constexpr int kSlabAtoms = 4096;
__global__ void __launch_bounds__(kVoxLdsThreads)
    k_vox_slab(LigandDev L, const float *__restrict__ rot, const int *__restrict__ boff, uint32_t *dmo, uint32_t *cnt,
               int *vidx, int mw, int cw, int planes) {
    extern __shared__ uint32_t msk[];
    __shared__ uint16_t list[kSlabAtoms];
    __shared__ int nlist;
    const int b = blockIdx.y, tid = threadIdx.x, ng = L.ng, rw = row_words(ng);
    const int p0 = blockIdx.x * planes, p1 = min(p0 + planes, ng);
    const int i0 = max(p0 - 2, 0), i1 = min(p1 + 2, ng), nw = (i1 - i0) * ng * rw;
    uint32_t *core = msk, *surf = msk + nw;
    float *gc = reinterpret_cast<float *>(msk + 2 * nw);
    __shared__ float coef[9];  // read once (rot may lie in host memory)
    if (tid < 9) coef[tid] = rot[9 * ((size_t)(boff ? *boff : 0) + b) + tid];
    for (int q = tid; q < 2 * nw; q += kVoxLdsThreads) msk[q] = 0u;
    for (int q = tid; q < ng; q += kVoxLdsThreads) gc[q] = L.gc[q];
    if (tid == 0) nlist = 0;
    __syncthreads();
    float r[9];
#pragma unroll
    for (int q = 0; q < 9; q++) r[q] = coef[q];
    const float h = (float)(ng / 2);
    for (int l0 = 0; l0 < L.na; l0 += kSlabAtoms) {
        for (int l = l0 + tid; l < min(l0 + kSlabAtoms, L.na); l += kVoxLdsThreads) {
            float X, Y, Z;
            rotate_atom(L, r, l, X, Y, Z);
            const int i2 = min(max((int)(X / L.gw + h), -3), ng + 2), ci = charge_row(L, X);
            if ((i2 + 2 >= i0 && i2 - 2 < i1) || (ci >= p0 && ci < p1)) list[atomicAdd(&nlist, 1)] = (uint16_t)(l - l0);
        }
        __syncthreads();
        const int n = nlist;
        for (int q = tid; q < n; q += kVoxLdsThreads) {
            const int l = l0 + list[q];
            float X, Y, Z;
            rotate_atom(L, r, l, X, Y, Z);
            vox_planes(L, gc, X, Y, Z, l, -2, 3, core, surf, i0, i1);
            const int ci = charge_row(L, X);
            if (ci >= p0 && ci < p1) {
                const int v = charge_voxel(L, X, Y, Z);
                vidx[(size_t)b * L.na + l] = v;
                atomicAdd(&cnt[(size_t)b * cw + (v >> 1)], 1u << (16 * (v & 1)));
            }
        }
        __syncthreads();  // the list is read; its count too
        if (tid == 0) nlist = 0;
        __syncthreads();
    }
    const MaskRows C{core, ng, rw, i0}, S{surf, ng, rw, i0};
    uint32_t *db = dmo + (size_t)b * 2 * mw;
    for (int q = p0 * ng * rw + tid; q < p1 * ng * rw; q += kVoxLdsThreads) {
        uint32_t d, o;
        vox_mask_word(C, S, q, ng, L.delta, d, o);
        db[q] = d;
        db[mw + q] = o;
    }
}

// The same with the core and surface bits in memory, for few rotations: a thread per atom and plane, so that
// one rotation of a large ligand fills the chip, where its slabs are a workgroup each.
__global__ void k_vox_clear(uint32_t *p, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

__global__ void __launch_bounds__(128) k_vox_atoms(LigandDev L, const float *__restrict__ rot, const int *__restrict__ boff,
                                                   uint32_t *cs, uint32_t *cnt, int *vidx, int mw, int cw) {
    const int b = blockIdx.y, q = blockIdx.x * blockDim.x + threadIdx.x, l = q / 5, d = q - 5 * l;
    __shared__ float coef[9];  // read once (rot may lie in host memory)
    if (threadIdx.x < 9) coef[threadIdx.x] = rot[9 * ((size_t)(boff ? *boff : 0) + b) + threadIdx.x];
    __syncthreads();
    if (l >= L.na) return;
    float r[9], X, Y, Z;
#pragma unroll
    for (int k = 0; k < 9; k++) r[k] = coef[k];
    rotate_atom(L, r, l, X, Y, Z);
    uint32_t *cb = cs + (size_t)b * 2 * mw;
    vox_planes(L, L.gc, X, Y, Z, l, d - 2, d - 1, cb, cb + mw, 0, L.ng);
    if (d == 0) {
        const int v = charge_voxel(L, X, Y, Z);
        vidx[(size_t)b * L.na + l] = v;
        atomicAdd(&cnt[(size_t)b * cw + (v >> 1)], 1u << (16 * (v & 1)));
    }
}

__global__ void __launch_bounds__(256) k_vox_masks(const uint32_t *__restrict__ cs, uint32_t *dmo, int ng, int mw, float delta) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
    if (q >= mw) return;
    const uint32_t *cb = cs + (size_t)b * 2 * mw;
    uint32_t *db = dmo + (size_t)b * 2 * mw;
    const MaskRows C{cb, ng, row_words(ng), 0}, S{cb + mw, ng, row_words(ng), 0};
    vox_mask_word(C, S, q, ng, delta, db[q], db[mw + q]);
}

// Rotations of a larger grid up to which their bits lie in memory.  One, 4, 8 and 16 rotations at 256^3 (with
// their charges): 2081 atoms 73, 82, 110, 123 us in memory, 87, 93, 114, 116 in slabs; 8000 atoms 213,
// 249, 290, 350 and 248, 270, 290, 303; at 216^3 8 rotations 112 and 107, 296 and 283.
constexpr int kFewRotations = 4;

// grids as (grid_r, grid_i) pairs; clears the charge grid it reads
__global__ void k_vox_expand(VoxGrid vg, float2 *lg, int ng3) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    const int b = blockIdx.y;
    if (v >= ng3) return;
    lg[(size_t)b * ng3 + v] = vox_take(vg, b, v / vg.ng, v % vg.ng);
}

}  // namespace

hipError_t launch_voxelize(const LigandDev &lig, const float *rot, int B, const VoxScratch &vs, int *vidx,
                           float *chg, hipStream_t s, const int *boff) {
    const int ng = lig.ng, mw = mask_words(ng), cw = count_words(ng);
    const int ng3 = ng * ng * ng;
    const size_t masks = mask_bytes(ng);
    if (masks_in_lds(ng)) {  // one workgroup per rotation, bits in LDS
        // the charges' table beside their list, where it fits into the masks' LDS (or little enough
        // for two workgroups a CU); more atoms than that are counted in memory
        const size_t most = std::max(masks + sizeof(float) * ng, (size_t)64 * 1024);
        auto table = [](int n) { return 2 * sizeof(uint32_t) * (size_t)n + sizeof(int2) * kCrowdCap; };
        int nt = kTableMax;
        while (nt > 256 && (nt / 2 >= 3 * lig.na || table(nt) > most)) nt /= 2;
        if (nt / 8 * 5 < lig.na) nt = 0;
        const size_t lds = std::max(masks + sizeof(float) * ng, nt ? table(nt) : 0);
        k_vox_lds<<<B, kVoxLdsThreads, lds, s>>>(lig, rot, boff, vs.dmo, vs.cnt, vidx, mw, cw, chg, nt);
        if (!nt) k_vox_charge<<<B, kChargeThreads, 0, s>>>(vidx, vs.cnt, lig.charge, chg, lig.na, ng3, cw);
    } else if (B <= kFewRotations) {
        const size_t words = 2 * (size_t)B * mw;
        k_vox_clear<<<(unsigned)std::min((words + 255) / 256, (size_t)65535), 256, 0, s>>>(vs.cs, words);
        k_vox_atoms<<<dim3((5 * lig.na + 127) / 128, B), 128, 0, s>>>(lig, rot, boff, vs.cs, vs.cnt, vidx, mw, cw);
        k_vox_masks<<<dim3((mw + 255) / 256, B), 256, 0, s>>>(vs.cs, vs.dmo, ng, mw, lig.delta);
        k_vox_charge<<<B, kChargeThreads, 0, s>>>(vidx, vs.cnt, lig.charge, chg, lig.na, ng3, cw);
    } else {
        // Slabs of 64 KB of masks (two workgroups a CU), or up to 132 KB where that is fewer than 12 planes.
        // Always 132 KB: 3-12% more time for 8 and 32 rotations at 160^3 to 320^3, 5% less for 64 at 216^3 and
        // 256^3.  Always 64 KB: within 4% of this either way, above 137 planes (where they differ) as well.
        const size_t plane = 2 * sizeof(uint32_t) * (size_t)ng * row_words(ng);
        const int with_halo = (int)std::max((size_t)64 * 1024 / plane, std::min((size_t)12, kVoxLdsBytes / plane));
        const int planes = with_halo - 4;
        if (planes < 1) return hipErrorInvalidValue;  // above ng = 320, which no context has
        const size_t lds = plane * std::min(with_halo, ng) + sizeof(float) * ng;
        k_vox_slab<<<dim3((ng + planes - 1) / planes, B), kVoxLdsThreads, lds, s>>>(lig, rot, boff, vs.dmo, vs.cnt, vidx, mw, cw,
                                                                                   planes);
        k_vox_charge<<<B, kChargeThreads, 0, s>>>(vidx, vs.cnt, lig.charge, chg, lig.na, ng3, cw);
    }
    return hipGetLastError();
}

hipError_t launch_vox_expand(const VoxGrid &vg, int B, float2 *lg, hipStream_t s) {
    const int ng3 = vg.ng * vg.ng * vg.ng;
    k_vox_expand<<<dim3((ng3 + 255) / 256, B), 256, 0, s>>>(vg, lg, ng3);
    return hipGetLastError();
}
