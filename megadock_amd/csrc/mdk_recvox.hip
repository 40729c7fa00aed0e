// Receptor grids on the device, bit-exact with the reference's producer (Receptor::rpscace
// and Receptor::electro, src/receptor.cpp:20-346; the host restatement is
// host/receptor.cpp).  Compiled with -ffp-contract=off; division and square root are
// the correctly rounded ones.
//
//   core fill        one workgroup per atom over its box: voxels with d^2 < 1.5 r^2 set
//                    their core bit (order-free);
//   open space       six rays per line of the grid, each until the first core voxel, 32
//                    voxels of a row at a time;
//   two sweeps       the reference's in-place propagation in increasing linear order
//                    (src/receptor.cpp:159-189).  A voxel is open when the sweep reaches it
//                    if it was open, or was zero with an in-range predecessor (-z, -y, -x)
//                    that was open when reached.  On rows of bits that is a recurrence over
//                    the rows i + j = d, run by one workgroup with a thread per i, the +z
//                    direction a carry through a row's zero voxels; every zero neighbour of
//                    an in-range voxel open when reached ends the sweep open;
//   cavities         zero becomes core, open becomes zero;
//   surface, charge  one thread per voxel, summing over the atoms in index order (the
//                    atoms whose boxes meet the workgroup's tile, compacted in LDS chunk by
//                    chunk), exactly the reference's per-voxel sequence of roundings.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mdk_internal.h"

namespace {

struct RecAtoms {
    const float *xyz, *radius, *charge, *ace, *gc;
    int na, ng;
    float gw;
};

// the voxel holding coordinate p along one axis (src/receptor.cpp:73-83)
__device__ __forceinline__ int cell_of(float p, float gw, int ng) { return (int)(p / gw + ng / 2); }

__device__ __forceinline__ float sq_dist(float p, float g) {
    const float d = p - g;
    return d * d;
}

__global__ void k_rec_clear(uint32_t *p, size_t n) {
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x) p[q] = 0u;
}

// bits of word w that are voxels lo <= k <= hi of a row
__device__ __forceinline__ uint32_t row_range(int w, int lo, int hi) {
    const int a = max(lo - 32 * w, 0), e = min(hi - 32 * w, 31);
    if (a > e) return 0u;
    return (e == 31 ? 0xffffffffu : (1u << (e + 1)) - 1u) & (0xffffffffu << a);
}

// core bits, rows (i, j) of row_words(ng) words
__global__ void __launch_bounds__(128) k_rec_core(RecAtoms A, uint32_t *core, int range) {
    const int l = blockIdx.x, ng = A.ng, rw = row_words(ng);
    const float x = A.xyz[3 * l], y = A.xyz[3 * l + 1], z = A.xyz[3 * l + 2];
    const float r = A.radius[l], rc2 = r * r * 1.5f;
    int lo[3], n[3];
    const float p[3] = {x, y, z};
    for (int a = 0; a < 3; a++) {
        // kept away from the ends of the integers, where an infinite coordinate's box would wrap to a size
        // above 0 far outside the arrays
        const int c = min(max(cell_of(p[a], A.gw, ng), -(1 << 24)), 1 << 24);
        lo[a] = max(c - range, 0);
        n[a] = max(min(c + range + 1, ng) - lo[a], 0);
    }
    for (int t = threadIdx.x; t < n[0] * n[1] * n[2]; t += blockDim.x) {
        const int i = lo[0] + t / (n[1] * n[2]), j = lo[1] + (t / n[2]) % n[1], k = lo[2] + t % n[2];
        const float ax = sq_dist(x, A.gc[i]), ay = sq_dist(y, A.gc[j]), az = sq_dist(z, A.gc[k]);
        if (ax > rc2 || ax + ay > rc2) continue;
        if (ax + ay + az < rc2) atomicOr(&core[(i * ng + j) * rw + (k >> 5)], 1u << (k & 31));
    }
}

// the word of open voxels along a row from its low (first set bit stops) end, `open` = nothing
// met so far; and from the high end
__device__ __forceinline__ uint32_t below_first(uint32_t c) { return c ? (c & (0u - c)) - 1u : 0xffffffffu; }
__device__ __forceinline__ uint32_t above_last(uint32_t c) {
    return c ? (__clz((int)c) ? 0xffffffffu << (32 - __clz((int)c)) : 0u) : 0xffffffffu;
}

// Rays of the three axes: one thread per row (z), per (i, word) (y) and per (j, word) (x), both
// directions.  The words met are independent loads, so the walks cost their count, not their
// latency.
__global__ void __launch_bounds__(64) k_rec_rays(const uint32_t *__restrict__ core, uint32_t *open, int ng) {
    const int rw = row_words(ng), nr = ng * ng, nw = ng * rw, t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < nr) {  // along the row t
        const uint32_t *c = core + t * rw;
        uint32_t *o = open + t * rw;
        for (int w = 0; w < rw; w++) {
            atomicOr(&o[w], below_first(c[w]) & row_range(w, 0, ng - 1));
            if (c[w]) break;
        }
        for (int w = rw - 1; w >= 0; w--) {
            atomicOr(&o[w], above_last(c[w]) & row_range(w, 0, ng - 1));
            if (c[w]) break;
        }
        return;
    }
    const int q = t - nr;
    if (q >= 2 * nw) return;
    const bool alongx = q >= nw;
    const int p = alongx ? q - nw : q, a = p / rw, w = p - a * rw;
    const int base = alongx ? a * rw + w : a * ng * rw + w, step = alongx ? ng * rw : rw;
    const uint32_t in = row_range(w, 0, ng - 1);
    uint32_t run = in;
#pragma unroll 8
    for (int s = 0; s < ng; s++) {
        run &= ~core[base + s * step];
        if (run) atomicOr(&open[base + s * step], run);
    }
    run = in;
#pragma unroll 8
    for (int s = ng - 1; s >= 0; s--) {
        run &= ~core[base + s * step];
        if (run) atomicOr(&open[base + s * step], run);
    }
}

// One sweep: reached[row] = the voxels of a row that are visited (src/receptor.cpp:161-165: i
// in [1, ng - 2], j and k in [2, ng - 2]) and open when the sweep reaches them.  Thread i walks
// j = d - i; its row's predecessors are its own previous row and thread i - 1's, both of step
// d - 1, in LDS; within a row the flags run upwards through zero voxels.  The next row's words
// are loaded a step ahead.  One workgroup: 2 ng steps of a few dozen instructions
// (ng = 72: 2 x 605 us with a thread per voxel of the planes i + j + k = s, 214 steps of up to
// 5184 voxels each, every voxel's value loaded inside its step).  RW: words a row, at least
// row_words(ng).
template <int RW>
__global__ void __launch_bounds__(512) k_rec_sweep(const uint32_t *__restrict__ core, const uint32_t *__restrict__ open,
                                                  uint32_t *__restrict__ reached, int ng) {
    extern __shared__ uint32_t flags[];  // [2][ng + 1][RW], row 0 stays zero
    const int rw = row_words(ng), i = threadIdx.x, plane = (ng + 1) * RW;
    for (int q = threadIdx.x; q < 2 * plane; q += blockDim.x) flags[q] = 0u;
    const bool on = i >= 1 && i <= ng - 2;
    uint32_t o[RW], z[RW];
    auto load = [&](int j) {
#pragma unroll
        for (int w = 0; w < RW; w++) {
            o[w] = z[w] = 0u;
            if (on && j >= 2 && j <= ng - 2 && w < rw) {
                const int q = (i * ng + j) * rw + w;
                const uint32_t in = row_range(w, 2, ng - 2), c = core[q], v = open[q];
                o[w] = v & in;
                z[w] = ~c & ~v & in;
            }
        }
    };
    load(0 - i);
    __syncthreads();
    for (int d = 0; d <= 2 * (ng - 1); d++) {
        const uint32_t *prev = flags + (d & 1 ? 0 : plane);
        uint32_t *cur = flags + (d & 1 ? plane : 0);
        const int j = d - i;
        if (i < ng) {
            uint32_t f[RW], carry = 0u;
#pragma unroll
            for (int w = 0; w < RW; w++) {
                uint32_t p = z[w];
                uint32_t s = o[w] | (p & (prev[(i + 1) * RW + w] | prev[i * RW + w])) | (p & carry);
                s |= p & (s << 1);
                p &= p << 1;
                s |= p & (s << 2);
                p &= p << 2;
                s |= p & (s << 4);
                p &= p << 4;
                s |= p & (s << 8);
                p &= p << 8;
                s |= p & (s << 16);
                f[w] = s;
                carry = s >> 31;
            }
            load(j + 1);
#pragma unroll
            for (int w = 0; w < RW; w++) {
                cur[(i + 1) * RW + w] = f[w];
                if (j >= 0 && j < ng && w < rw) reached[(i * ng + j) * rw + w] = f[w];
            }
        }
        __syncthreads();
    }
}

// end of a sweep: a zero voxel next to a voxel open when reached is open
__global__ void __launch_bounds__(256) k_rec_sweep_apply(const uint32_t *__restrict__ core, uint32_t *open,
                                                        const uint32_t *__restrict__ reached, int ng) {
    const int rw = row_words(ng), q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= ng * ng * rw) return;
    const int w = q % rw, row = q / rw, i = row / ng, j = row - i * ng;
    const uint32_t c = reached[q];
    uint32_t nb = (c << 1) | (c >> 1);
    if (w > 0) nb |= reached[q - 1] >> 31;
    if (w + 1 < rw) nb |= reached[q + 1] << 31;
    if (j > 0) nb |= reached[q - rw];
    if (j + 1 < ng) nb |= reached[q + rw];
    if (i > 0) nb |= reached[q - ng * rw];
    if (i + 1 < ng) nb |= reached[q + ng * rw];
    open[q] |= nb & ~core[q] & row_range(w, 0, ng - 1);
}

// Surface score and electrostatics, one thread per voxel of a 4 x 8 x 8 tile.
constexpr int kTI = 4, kTJ = 8, kTK = 8, kSumThreads = kTI * kTJ * kTK;
// an atom as the tile sees it: its box relative to the tile's origin, whether the box covers
// the tile; surface: squared reach and the double term; charge: eratio beta q divided by the
// dielectric's two constants
struct TileAtom {
    float x, y, z, rj, q, q4, q80;
    int whole;
    double add;
    int lo[3], hi[3];
};

// (An infinite coordinate's box wraps to lo far above the grid or hi below it, so it meets no tile; a clamp
// here, for every atom in every tile, cost the sums 8 of 479 us.)
__device__ __forceinline__ void atom_box(const float *p, float gw, int ng, int range, int *lo, int *hi) {
    for (int a = 0; a < 3; a++) {
        const unsigned c = (unsigned)cell_of(p[a], gw, ng);
        lo[a] = max((int)(c - (unsigned)range), 0);
        hi[a] = min((int)(c + (unsigned)range + 1u), ng);
    }
}

__global__ void __launch_bounds__(kSumThreads)
    k_rec_sums(RecAtoms A, const uint32_t *__restrict__ core, const uint32_t *__restrict__ open, float2 *out, float eps,
               int surf_range, bool regular, float aceratio, float eratio, float gwl, float charge_per_grid) {
    __shared__ TileAtom list[kSumThreads];
    __shared__ int wave_count[kSumThreads / 64];
    const int ng = A.ng, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0[3] = {(int)blockIdx.z * kTI, (int)blockIdx.y * kTJ, (int)blockIdx.x * kTK};
    const int i = t0[0] + tid / (kTJ * kTK), j = t0[1] + (tid / kTK) % kTJ, k = t0[2] + tid % kTK;
    const bool mine = i < ng && j < ng && k < ng;
    const size_t v = mine ? ((size_t)i * ng + j) * ng + k : 0;
    const float gci = A.gc[mine ? i : 0], gcj = A.gc[mine ? j : 0], gck = A.gc[mine ? k : 0];
    const int t1[3] = {min(t0[0] + kTI, ng), min(t0[1] + kTJ, ng), min(t0[2] + kTK, ng)};
    const float beta = -2800.0f;
    // the atoms of the next chunk whose boxes meet this tile, in index order
    auto gather = [&](int base, bool elec) -> int {
        const int l = base + tid;
        bool keep = false;
        TileAtom a;
        if (l < A.na) {
            a.x = A.xyz[3 * l];
            a.y = A.xyz[3 * l + 1];
            a.z = A.xyz[3 * l + 2];
            const float p[3] = {a.x, a.y, a.z};
            if (!elec) {
                const float r = A.radius[l];
                a.rj = (r + 3.6f) * (r + 3.6f);
                a.add = 1.0 + (double)A.ace[l] * (-0.8) * (double)aceratio;
                // voxels further than r + 3.6 are never hit: where the grid's coordinates are the
                // voxel centres (regular), the box need not reach past that
                const float reach = fabsf(r + 3.6f) / A.gw;
                atom_box(p, A.gw, ng, regular && reach < (float)surf_range - 3.0f ? (int)reach + 3 : surf_range, a.lo, a.hi);
                keep = true;
            } else {
                a.q = A.charge[l];
                const float aq = fabsf(a.q);
                if (aq > 1.0e-6f) {
                    const int range = (double)aq < 0.07 ? 4 : ((double)aq < 0.21 ? 5 : (int)(aq / charge_per_grid));
                    atom_box(p, gwl, ng, range, a.lo, a.hi);
                    keep = true;
                    a.q = eratio * beta * a.q;
                    a.q4 = a.q / 4.0f;
                    a.q80 = a.q / 80.0f;
                }
            }
            a.whole = 1;
            if (keep)
                for (int d = 0; d < 3; d++) {
                    keep = keep && a.lo[d] < t1[d] && a.hi[d] > t0[d];
                    a.whole = a.whole && a.lo[d] <= t0[d] && a.hi[d] >= t1[d];
                }
        }
        const unsigned long long bal = __ballot(keep);
        if (lane == 0) wave_count[wave] = __popcll(bal);
        __syncthreads();
        int off = 0, total = 0;
        for (int w = 0; w < kSumThreads / 64; w++) {
            if (w < wave) off += wave_count[w];
            total += wave_count[w];
        }
        if (keep) list[off + __popcll(bal & ((1ull << lane) - 1ull))] = a;
        __syncthreads();
        return total;
    };
    // surface: sum over atoms of 1 + ACE * (-0.8) * aceratio, in double, rounded per term
    float surf = 0.0f;
    for (int base = 0; base < A.na; base += kSumThreads) {
        const int n = gather(base, false);
        if (mine)
            for (int m = 0; m < n; m++) {
                const TileAtom &a = list[m];
                if (i < a.lo[0] || i >= a.hi[0] || j < a.lo[1] || j >= a.hi[1] || k < a.lo[2] || k >= a.hi[2]) continue;
                const float ax = sq_dist(a.x, gci), ay = sq_dist(a.y, gcj), az = sq_dist(a.z, gck);
                if (ax > a.rj || ax + ay > a.rj) continue;
                if (ax + ay + az < a.rj) surf = (float)((double)surf + a.add);
            }
        __syncthreads();  // the list is rewritten by the next chunk
    }
    // core and enclosed cavities hold the core value
    const int word = (i * ng + j) * row_words(ng) + (k >> 5);
    const bool inner = mine && (((core[word] | ~open[word]) >> (k & 31)) & 1u);
    const float g = inner ? eps : surf;
    // electrostatics on the voxels that are not core (src/receptor.cpp:258-346); the quotient
    // (eratio beta q / er) / d with er = 4 or 80 divides the atom's constants
    float e = 0.0f;
    const bool field = mine && !(g < 0.0);
    for (int base = 0; base < A.na; base += kSumThreads) {
        const int n = gather(base, true);
        if (field)
            for (int m = 0; m < n; m++) {
                const TileAtom &a = list[m];
                if (!a.whole &&
                    (i < a.lo[0] || i >= a.hi[0] || j < a.lo[1] || j >= a.hi[1] || k < a.lo[2] || k >= a.hi[2]))
                    continue;
                const float dij = sq_dist(a.x, gci) + sq_dist(a.y, gcj);
                const float d = sqrtf(dij + sq_dist(a.z, gck));
                float t = d >= 8.0f ? a.q80 : a.q4;
                if (d > 6.0f && d < 8.0f) t = a.q / (38.0f * d + -224.0f);
                e += t / d;
            }
        __syncthreads();
    }
    if (mine) out[v] = make_float2(g, e);
}

}  // namespace

size_t receptor_voxel_scratch_bytes(int ng) { return 3 * sizeof(uint32_t) * (size_t)mask_words(ng); }

// atoms (centred coordinates xyz, radius, charge, ace: device, na each; gc: device, ng);
// scratch: core, open and reached bits; regular: gc holds the voxel centres of pitch gw
hipError_t launch_receptor_voxel(const float *xyz, const float *radius, const float *charge, const float *ace,
                                 const float *gc, int na, int ng, float gw, float aceratio, float rec_core, float eratio,
                                 float gc0, float gc1, bool regular, void *scratch, float2 *out, hipStream_t s) {
    const int mw = mask_words(ng), rw = row_words(ng);
    uint32_t *core = (uint32_t *)scratch, *open = core + mw, *reached = open + mw;
    const RecAtoms A{xyz, radius, charge, ace, gc, na, ng, gw};
    k_rec_clear<<<(2 * mw + 255) / 256, 256, 0, s>>>(core, 2 * (size_t)mw);
    const int core_range = (int)((2.4 + (double)gw - 0.01) / (double)gw);
    // a core value that no voxel compares equal to (not a number) stops no ray and keeps no
    // voxel: as without core voxels; with the core value 0 every voxel is core from the start
    const bool none = rec_core != rec_core, all = rec_core == 0.0f;
    if (na > 0 && !none && !all) k_rec_core<<<na, 128, 0, s>>>(A, core, core_range);
    if (!all) {
        k_rec_rays<<<(ng * ng + 2 * ng * rw + 63) / 64, 64, 0, s>>>(core, open, ng);
        const unsigned apply = (unsigned)((mw + 255) / 256), nt = (unsigned)((ng + 63) / 64 * 64);
        for (int sweep = 0; sweep < 2; sweep++) {
            const size_t lds = 2 * sizeof(uint32_t) * (size_t)(ng + 1);
            if (rw <= 1) k_rec_sweep<1><<<1, nt, lds, s>>>(core, open, reached, ng);
            else if (rw <= 2) k_rec_sweep<2><<<1, nt, 2 * lds, s>>>(core, open, reached, ng);
            else if (rw <= 3) k_rec_sweep<3><<<1, nt, 3 * lds, s>>>(core, open, reached, ng);
            else if (rw <= 4) k_rec_sweep<4><<<1, nt, 4 * lds, s>>>(core, open, reached, ng);
            else if (rw <= 6) k_rec_sweep<6><<<1, nt, 6 * lds, s>>>(core, open, reached, ng);
            else if (rw <= 10) k_rec_sweep<10><<<1, nt, 10 * lds, s>>>(core, open, reached, ng);
            else return hipErrorInvalidValue;  // ng > 320: beyond the FFT passes' own limit
            k_rec_sweep_apply<<<apply, 256, 0, s>>>(core, open, reached, ng);
        }
    }
    const int surf_range = (int)((12 + (double)gw - 0.01) / (double)gw);
    const float beta = -2800.0f, gwl = gc1 - gc0;
    const float charge_per_grid = -1 * gwl * 80.0f / (beta * eratio);
    const dim3 tiles((ng + kTK - 1) / kTK, (ng + kTJ - 1) / kTJ, (ng + kTI - 1) / kTI);
    k_rec_sums<<<tiles, kSumThreads, 0, s>>>(A, core, open, out, rec_core, surf_range, regular, aceratio, eratio, gwl,
                                             charge_per_grid);
    return hipGetLastError();
}
