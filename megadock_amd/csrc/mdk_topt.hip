// Per-rotation top-t for t above the register lists of the fused inverse passes
// (t > MDK_MAXT).  The inverse passes write the batch's real score maps; this selects each
// rotation's t best entries with the order of the reference's insertion top-t for t > 1
// (src/fft_process.cpp:407-431): key fl(value / nf^3) descending, ties to the lower linear
// grid index, only keys above the starting value -99999 kept.
//
// Each map entry i of a rotation gets the 64-bit key
//   K = sortable(fl(v / nf^3)) << 32 | (2^32 - 1 - i)
// (sortable() maps float order to unsigned order after -0 -> +0, so equal keys tie and the
// lower index wins), all distinct, so the wanted entries are the t largest K:
//   1. radix select per rotation, 8 bits a level from the top, every workgroup of a level
//      adding its histogram of one chunk of one rotation; a level whose chosen bucket
//      holds exactly the entries still wanted ends the select early (the threshold is
//      then that bucket's lowest key);
//   2. compaction of the entries with K >= threshold (exactly min(t, nf^3) of them);
//   3. one workgroup per rotation sorts them (bitonic, in LDS up to 8192 keys, else in
//      global memory) and writes the rotation's t SortScore entries.
// For t up to kWideT two passes over the maps do instead of the levels' up to eight and the
// compaction's one (112^3, t = 64, 128 rotations: 1.25 -> 0.4 ms):
//   1. one histogram of the raw scores' leading 13 bits (sign, exponent, four bits of the
//      fraction: 8192 buckets in LDS, 6% wide) gives the bucket that holds the t-th largest
//      score, and with its lower edge a score below which no key can reach the top t
//      (quotient_cut);
//   2. the scores not below it, typically a few times t, become the keys that step 3 sorts.
// A rotation with more of them than fit (many equal scores) has its t-th score found in two
// further histograms (k_wide_compact, k_wide_value), and of the entries that equal it the first
// ones are taken (k_wide_ties), all workgroups sharing those rotations.
#include <hip/hip_runtime.h>

#include "mdk_internal.h"
#include "../../include/mdk_hip.h"

namespace {

constexpr int kChunk = 4096;     // map entries per histogram workgroup (16 per thread)
constexpr int kTSortLds = 8192;  // keys sorted in LDS
// Wide select.  kWideT: a list of kTSortLds keys leaves 16 times t for the threshold's bucket and
// its ties; above, the bucket alone may not fit.
constexpr int kWideT = kTSortLds / 16, kWideShift = 19, kWideBuckets = 1 << (32 - kWideShift);
constexpr unsigned kWideChunk = 32768;  // map entries per workgroup: 32 KB of buckets are cleared and added for 128 KB
// Rotations whose list does not fit: histograms of 2^10 quotients a bucket, at the start of the
// rotation's keys, and of single ones, behind the kTieKeys keys that are kept.  A wide bucket is 2^19
// neighbouring scores of one binade, and a division leaves at most twice as many units of the last place
// between them, so its quotients fall into buckets 0 .. 1024; the last bucket takes what lies above.
constexpr int kCoarseShift = 10, kCoarse = 2048, kFine = 1 << kCoarseShift;
constexpr int kTieThreads = 512, kTieBlocks = 512;
constexpr unsigned kTieKeys = kTSortLds - kFine * sizeof(unsigned) / sizeof(unsigned long long);
static_assert(kCoarse * sizeof(unsigned) <= kTieKeys * sizeof(unsigned long long) && kTieKeys >= 2 * kWideT,
              "the histograms lie where the keys go; the second clear of the keys written");
static_assert(kWideBuckets * sizeof(unsigned) <= kTSortLds * sizeof(unsigned long long),
              "the histogram lies where the keys go");

__device__ __forceinline__ unsigned sortable(float f) {
    const unsigned u = __float_as_uint(f);
    return u ^ ((u & 0x80000000u) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ unsigned long long topt_key(float v, float nf3f, unsigned i) {
    const float f = v / nf3f + 0.0f;  // the reference's key; -0 -> +0
    return ((unsigned long long)sortable(f) << 32) | (0xffffffffu - i);
}

__device__ __forceinline__ unsigned sortable_score(float v) { return sortable(v + 0.0f); }  // -0 as +0
__device__ __forceinline__ unsigned sortable_quotient(float v, float nf3f) { return sortable(v / nf3f + 0.0f); }  // as topt_key

__device__ __forceinline__ float key_float(unsigned long long k) {
    const unsigned u = (unsigned)(k >> 32);
    return __uint_as_float((u & 0x80000000u) ? (u ^ 0x80000000u) : ~u);
}

__global__ void k_tsel_init(TopTState *st, unsigned rank) {
    TopTState &s = st[blockIdx.x];
    s.hist[threadIdx.x] = 0u;
    if (threadIdx.x == 0) {
        s.prefix = 0ull;
        s.mask = 0ull;
        s.rank = rank;
        s.count = 0u;
        s.done = 0u;
    }
}

// grid (chunks, B): histogram of digit `shift` over the entries matching the prefix
__global__ void __launch_bounds__(256) k_tsel_hist(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                   TopTState *st, int shift) {
    __shared__ unsigned h[256];
    TopTState &s = st[blockIdx.y];
    if (s.done) return;  // uniform
    h[threadIdx.x] = 0u;
    __syncthreads();
    const unsigned long long prefix = s.prefix, mask = s.mask;
    const float *m = smap + (size_t)blockIdx.y * n3;
    const unsigned i0 = blockIdx.x * (unsigned)kChunk;
    const unsigned i1 = min(n3, i0 + (unsigned)kChunk);
    for (unsigned i = i0 + threadIdx.x; i < i1; i += 256u) {
        const unsigned long long k = topt_key(m[i], nf3f, i);
        if ((k & mask) == prefix) atomicAdd(&h[(unsigned)(k >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&s.hist[threadIdx.x], h[threadIdx.x]);
}

// one block per rotation: the digit of the wanted key at this level
__global__ void k_tsel_pick(TopTState *st, int shift) {
    TopTState &s = st[blockIdx.x];
    if (threadIdx.x == 0 && !s.done) {
        unsigned c = 0u;
        for (int d = 255; d >= 0; d--) {
            const unsigned h = s.hist[d];
            if (c + h >= s.rank) {
                s.prefix |= (unsigned long long)d << shift;
                s.mask |= 255ull << shift;
                s.rank -= c;
                if (s.rank == h) s.done = 1u;  // the whole bucket is wanted
                break;
            }
            c += h;
        }
    }
    __syncthreads();
    for (int d = threadIdx.x; d < 256; d += blockDim.x) s.hist[d] = 0u;
}

// grid (chunks, B): the entries at or above the threshold, in any order
__global__ void __launch_bounds__(256) k_tsel_compact(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                      TopTState *st, unsigned long long *keys, unsigned P) {
    TopTState &s = st[blockIdx.y];
    const unsigned long long thr = s.prefix;
    const float *m = smap + (size_t)blockIdx.y * n3;
    unsigned long long *out = keys + (size_t)blockIdx.y * P;
    const unsigned i0 = blockIdx.x * (unsigned)kChunk;
    const unsigned i1 = min(n3, i0 + (unsigned)kChunk);
    for (unsigned i = i0 + threadIdx.x; i < i1; i += 256u) {
        const unsigned long long k = topt_key(m[i], nf3f, i);
        if (k >= thr) out[atomicAdd(&s.count, 1u)] = k;
    }
}

// ---- wide select; a rotation's histogram lies at the start of its keys and is zero between batches
// (k_tsel_sort_out clears it: a launch of its own for that cost 2000 rotations of 64^3, t = 20, 0.1 of 5.1 ms)
// grid (chunks, B); n3 is a multiple of 8 (nf is even)
__global__ void __launch_bounds__(1024) k_wide_hist(const float *__restrict__ smap, unsigned n3, TopTState *st,
                                                    unsigned long long *keys) {
    __shared__ unsigned h[kWideBuckets];
    for (int q = threadIdx.x; q < kWideBuckets; q += 1024) h[q] = 0u;
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) st[0].nover = 0u;
    __syncthreads();
    const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)blockIdx.y * n3);
    const unsigned i0 = blockIdx.x * (kWideChunk / 4), i1 = min(n3 / 4, i0 + kWideChunk / 4);
    for (unsigned i = i0 + threadIdx.x; i < i1; i += 1024u) {
        const float4 v = m[i];
        atomicAdd(&h[sortable_score(v.x) >> kWideShift], 1u);
        atomicAdd(&h[sortable_score(v.y) >> kWideShift], 1u);
        atomicAdd(&h[sortable_score(v.z) >> kWideShift], 1u);
        atomicAdd(&h[sortable_score(v.w) >> kWideShift], 1u);
    }
    __syncthreads();
    unsigned *g = reinterpret_cast<unsigned *>(keys + (size_t)blockIdx.y * kTSortLds);
    for (int q = threadIdx.x; q < kWideBuckets; q += 1024)
        if (h[q]) atomicAdd(&g[q], h[q]);
}

// one workgroup per rotation: the score below which nothing reaches the top `rank` (in st.prefix, as
// sortable bits), and whether the entries of the buckets down to that score's fit the list; if not,
// st.base is the least quotient of the bucket, as sortable bits, and the rotation's histograms are cleared
__global__ void __launch_bounds__(1024) k_wide_pick(TopTState *st, unsigned long long *keys, unsigned rank, float nf3f) {
    constexpr int PER = kWideBuckets / 1024;
    __shared__ unsigned cum[1024], cut_bits;
    __shared__ bool over;
    unsigned *h = reinterpret_cast<unsigned *>(keys + (size_t)blockIdx.x * kTSortLds);
    const int top = kWideBuckets - 1 - (int)threadIdx.x * PER;  // this thread's buckets: top, top - 1, ...
    unsigned n[PER], s = 0u;
#pragma unroll
    for (int q = 0; q < PER; q++) s += n[q] = h[top - q];
    cum[threadIdx.x] = s;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned add = (int)threadIdx.x >= d ? cum[threadIdx.x - d] : 0u;
        __syncthreads();
        cum[threadIdx.x] += add;
        __syncthreads();
    }
    const unsigned above = cum[threadIdx.x] - s;  // entries above this thread's buckets
    if (above < rank && cum[threadIdx.x] >= rank) {
        int b = top;
        unsigned c = above;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            c += n[q];
            if (c < rank) b--;
        }
        const unsigned long long edge = (unsigned long long)((unsigned)b << kWideShift) << 32;
        const float cut = quotient_cut(key_float(edge), nf3f);
        over = cut != cut;  // a bucket of what is not a number
        cut_bits = sortable_score(cut);
        st[blockIdx.x].base = sortable_quotient(key_float(edge), nf3f);
    }
    __syncthreads();
    const int last = (int)(cut_bits >> kWideShift);
    if (top >= last && top - PER < last) {
        unsigned c = above;
#pragma unroll
        for (int q = 0; q < PER; q++)
            if (top - q >= last) c += n[q];
        TopTState &S = st[blockIdx.x];
        over = over || c > (unsigned)kTSortLds;
        S.prefix = cut_bits;
        S.count = 0u;
        S.over = over;
        if (over) st[atomicAdd(&st[0].nover, 1u)].nth_over = blockIdx.x;
    }
    __syncthreads();
    if (over)
        for (int q = threadIdx.x; q < kCoarse; q += 1024) {
            h[q] = 0u;
            if (q < kFine) h[2 * kTieKeys + q] = 0u;
        }
}

// Adds one to h[bucket] for the lanes that are `in`.  Equal buckets are the rule here: one lane adds
// for all that have the first one's.
__device__ __forceinline__ void add_bucket(unsigned *h, bool in, int bucket) {
    const unsigned long long some = __ballot(in);
    if (some == 0ull) return;
    const int first = __ffsll((long long)some) - 1, b0 = __builtin_amdgcn_readlane(bucket, first);
    const unsigned long long same = __ballot(in && bucket == b0);
    if ((int)(threadIdx.x & 63) == first)
        atomicAdd(&h[b0], (unsigned)__popcll(same));
    else if (in && bucket != b0)
        atomicAdd(&h[bucket], 1u);
}

// grid (chunks, B): the keys of the scores not below the cut, of rotations where they fit; of the others,
// the quotients from st.base on by kCoarseShift bits
__global__ void __launch_bounds__(1024) k_wide_compact(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                       TopTState *st, unsigned long long *keys) {
    __shared__ unsigned h[kCoarse];
    TopTState &s = st[blockIdx.y];
    const unsigned cut = (unsigned)s.prefix;
    const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)blockIdx.y * n3);
    unsigned long long *out = keys + (size_t)blockIdx.y * kTSortLds;
    auto put = [&](float v, unsigned i) {
        if (sortable_score(v) >= cut) out[atomicAdd(&s.count, 1u)] = topt_key(v, nf3f, i);
    };
    const unsigned i0 = blockIdx.x * (kWideChunk / 4), i1 = min(n3 / 4, i0 + kWideChunk / 4);
    if (s.over) {  // uniform
        const unsigned base = s.base;
        for (int q = threadIdx.x; q < kCoarse; q += 1024) h[q] = 0u;
        __syncthreads();
        for (unsigned i = i0 + threadIdx.x; i < i1; i += 1024u) {
            const float4 v = m[i];
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned q = sortable_quotient(e[k], nf3f);
                add_bucket(h, q >= base, (int)min((q - base) >> kCoarseShift, (unsigned)kCoarse - 1u));
            }
        }
        __syncthreads();
        unsigned *g = reinterpret_cast<unsigned *>(out);
        for (int q = threadIdx.x; q < kCoarse; q += 1024)
            if (h[q]) atomicAdd(&g[q], h[q]);
        return;
    }
    for (unsigned i = i0 + threadIdx.x; i < i1; i += 1024u) {
        const float4 v = m[i];
        if (sortable_score(v.x) >= cut || sortable_score(v.y) >= cut || sortable_score(v.z) >= cut || sortable_score(v.w) >= cut) {
            put(v.x, 4 * i);
            put(v.y, 4 * i + 1);
            put(v.z, 4 * i + 2);
            put(v.w, 4 * i + 3);
        }
    }
}

// The bucket of the want-th entry from the top of a histogram of PER * kTieThreads buckets, and how many of
// its entries are wanted; by every workgroup for itself.
struct Picked {
    int bucket;
    unsigned want;
};
template <int PER> __device__ __forceinline__ Picked pick_from_top(const unsigned *hist, unsigned want) {
    __shared__ unsigned wave_sum[kTieThreads / 64];
    __shared__ Picked picked;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, top = PER * kTieThreads - 1 - PER * tid;
    unsigned in[PER], s = 0u;
#pragma unroll
    for (int k = 0; k < PER; k++) s += in[k] = hist[top - k];
    unsigned c = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned o = __shfl_up(c, d, 64);
        if (lane >= d) c += o;
    }
    if (lane == 63) wave_sum[wave] = c;
    if (tid == 0) picked = Picked{0, want};
    __syncthreads();
    for (int w = 0; w < wave; w++) c += wave_sum[w];
    if (c - s < want && c >= want) {
        int b = top;
        unsigned a = c - s;
#pragma unroll
        for (int k = 0; k + 1 < PER; k++)
            if (b == top - k && a + in[k] < want) {
                a += in[k];
                b--;
            }
        picked = Picked{b, want - a};
    }
    __syncthreads();
    const Picked p = picked;
    __syncthreads();  // the next rotation's
    return p;
}

// Rotations whose keys do not fit: k_wide_compact has their quotients by 2^10 from the wide bucket's least on,
// k_wide_value counts the single quotients of the bucket that holds the t-th one, and k_wide_ties takes
// the entries above that quotient and, of those that equal it, the first ones of each share of the map, as many as are
// wanted of all: the final sort drops what is too many.  A launch's workgroups share out the rotations (with
// one, all of them read its map).  Without such rotations the two launches end at their first load, but each
// still waits until the other stream's kernels leave room for it: a search of 112^3, 1024 rotations, t = 64,
// takes 12.20 ms with 512 threads a workgroup, 12.33 with 1024 (12.19 with one launch of one workgroup a
// rotation; five levels of 12 bits in six launches of 1024 threads took 1.6 to 3.4% more than that).  Docking
// with every score equal takes 0.39 ms a rotation of 112^3 with t = 64, 0.60 and 0.90 of 256^3 with t = 64
// and 512, 2.58 ms 128 rotations of 112^3 (8.98, 106, 100 and 14.1 ms with one workgroup a rotation).
struct TieShare {  // this workgroup's part of the rotations q0, q0 + step, ...
    unsigned n, parts, part, q0;
};
__device__ __forceinline__ TieShare tie_share(const TopTState *st) {
    const unsigned n = st[0].nover;
    if (n == 0u) return TieShare{0u, 1u, 0u, 0u};
    if (n >= gridDim.x) return TieShare{n, 1u, 0u, blockIdx.x};
    const unsigned part = blockIdx.x / n, parts = gridDim.x / n;
    return TieShare{part < parts ? n : 0u, parts, part, blockIdx.x % n};
}

__global__ void __launch_bounds__(kTieThreads) k_wide_value(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                     TopTState *st, unsigned long long *keys, unsigned rank) {
    __shared__ unsigned h[kFine];
    const TieShare T = tie_share(st);
    const int tid = threadIdx.x;
    for (unsigned q = T.q0; q < T.n; q += gridDim.x) {  // uniform
        const unsigned b = st[q].nth_over;
        TopTState &S = st[b];
        unsigned *hist = reinterpret_cast<unsigned *>(keys + (size_t)b * kTSortLds);
        const Picked p = pick_from_top<kCoarse / kTieThreads>(hist, rank);
        const unsigned base = S.base + ((unsigned)p.bucket << kCoarseShift);
        if (T.part == 0 && tid == 0) {
            S.fine_base = base;
            S.fine_want = p.want;
            S.above = 0u;
        }
        for (int k = tid; k < kFine; k += kTieThreads) h[k] = 0u;
        __syncthreads();
        const unsigned share = (n3 / 4 + T.parts - 1) / T.parts, i0 = T.part * share, i1 = min(n3 / 4, i0 + share);
        const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)b * n3);
        for (unsigned i = i0 + tid; i < i1; i += (unsigned)kTieThreads) {
            const float4 f = m[i];
            const float e[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned d = sortable_quotient(e[k], nf3f) - base;
                add_bucket(h, d < (unsigned)kFine, (int)d);
            }
        }
        __syncthreads();
        for (int k = tid; k < kFine; k += kTieThreads)
            if (h[k]) atomicAdd(&hist[2 * kTieKeys + k], h[k]);
        __syncthreads();  // the next rotation clears h
    }
}

__global__ void __launch_bounds__(kTieThreads) k_wide_ties(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                    TopTState *st, unsigned long long *keys, unsigned rank) {
    __shared__ unsigned wave_sum[kTieThreads / 64];
    const TieShare T = tie_share(st);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (unsigned q = T.q0; q < T.n; q += gridDim.x) {  // uniform
        const unsigned b = st[q].nth_over;
        TopTState &S = st[b];
        unsigned long long *out = keys + (size_t)b * kTSortLds;
        const Picked p = pick_from_top<kFine / kTieThreads>(reinterpret_cast<const unsigned *>(out) + 2 * kTieKeys, S.fine_want);
        const unsigned value = S.fine_base + (unsigned)p.bucket, want = p.want, above = rank - want;
        // above + parts * want <= kTieKeys
        const unsigned parts = min(T.parts, (kTieKeys - (unsigned)kWideT) / want);
        if (T.part >= parts) continue;
        if (T.part == 0 && tid == 0) S.count = above + parts * want;
        unsigned long long *mine = out + above + T.part * want;
        const unsigned share = (n3 / 4 + parts - 1) / parts, i0 = T.part * share, i1 = min(n3 / 4, i0 + share);
        const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)b * n3);
        unsigned found = 0u;  // entries of this share that equal the value, in index order
        for (unsigned r = i0; r < i1; r += (unsigned)kTieThreads) {
            const unsigned i = r + tid;
            const bool on = i < i1;
            const float4 f = on ? m[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            const float e[4] = {f.x, f.y, f.z, f.w};
            unsigned equal = 0u;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned s = sortable_quotient(e[k], nf3f);
                if (on && s > value) {
                    const unsigned at = atomicAdd(&S.above, 1u);
                    if (at < above) out[at] = topt_key(e[k], nf3f, 4 * i + k);
                }
                equal |= (unsigned)(on && s == value) << k;
            }
            if (found >= want || !__syncthreads_or((int)equal)) continue;  // uniform
            unsigned c = __popc(equal);
            const unsigned n = c;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const unsigned o = __shfl_up(c, d, 64);
                if (lane >= d) c += o;
            }
            if (lane == 63) wave_sum[wave] = c;
            __syncthreads();
            unsigned at = found + c - n, all = 0u;
            for (int w = 0; w < kTieThreads / 64; w++) {
                if (w < wave) at += wave_sum[w];
                all += wave_sum[w];
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (equal >> k & 1u) {
                    if (at < want) mine[at] = topt_key(e[k], nf3f, 4 * i + k);
                    at++;
                }
            found += all;
            __syncthreads();  // the next round writes wave_sum
        }
        for (unsigned k = found + tid; k < want; k += (unsigned)kTieThreads) mine[k] = 0ull;  // sorts last
    }
}

// one workgroup per rotation: descending bitonic sort of its P keys (padded with 0, which
// sorts last; P = 0, wide select: of its count rounded up to a power of two, at most kTSortLds), then the
// rotation's t results; a rotation's keys lie `stride` apart
__global__ void __launch_bounds__(1024) k_tsel_sort_out(unsigned long long *keys, unsigned stride, unsigned P,
                                                        const TopTState *st, int t, int nf, mdk_sortscore *__restrict__ out,
                                                        const int *__restrict__ rot_id, const int *__restrict__ boff) {
    __shared__ unsigned long long sl[kTSortLds];
    const int b = blockIdx.x;
    const unsigned n = st[b].count;
    unsigned long long *g = keys + (size_t)b * stride;
    const bool wide = P == 0u;
    if (wide)
        for (P = 1u; P < n;) P <<= 1;
    const bool lds = P <= (unsigned)kTSortLds;
    unsigned long long *s = lds ? sl : g;
    for (unsigned i = threadIdx.x; i < P; i += 1024u) s[i] = i < n ? g[i] : 0ull;
    __syncthreads();
    if (wide)  // the next batch's histogram
        for (unsigned i = threadIdx.x; i < kWideBuckets / 2; i += 1024u) g[i] = 0ull;
    for (unsigned k = 2; k <= P; k <<= 1)
        for (unsigned j = k >> 1; j > 0; j >>= 1) {
            for (unsigned i = threadIdx.x; i < P; i += 1024u) {
                const unsigned l = i ^ j;
                if (l > i) {
                    const unsigned long long a = s[i], c = s[l];
                    const bool desc = (i & k) == 0;
                    if (desc ? (a < c) : (a > c)) {
                        s[i] = c;
                        s[l] = a;
                    }
                }
            }
            __syncthreads();
        }
    const int b0 = boff ? *boff : 0;
    const int rid = rot_id[b0 + b];
    mdk_sortscore *o = out + ((size_t)b0 + b) * t;
    const int nf2 = nf * nf;
    for (int q = threadIdx.x; q < t; q += 1024) {
        mdk_sortscore r;
        const unsigned long long k = (unsigned)q < n ? s[q] : 0ull;
        const float key = key_float(k);
        // sorted, so the kept entries are a prefix; the reference's slots start at -99999
        const bool keep = (unsigned)q < n && key > -99999.0f;
        const int idx = keep ? (int)(0xffffffffu - (unsigned)(k & 0xffffffffull)) : 0;
        r.score = keep ? key : -99999.0f;
        r.index[0] = rid;
        r.index[1] = idx / nf2;
        r.index[2] = (idx / nf) % nf;
        r.index[3] = idx % nf;
        o[q] = r;
    }
}

}  // namespace

unsigned topt_sort_size(int t, int nf) {
    const unsigned long long n3 = (unsigned long long)nf * nf * nf;
    const unsigned rank = (unsigned long long)t < n3 ? (unsigned)t : (unsigned)n3;
    if (rank <= (unsigned)kWideT) return kTSortLds;
    unsigned P = 1;
    while (P < rank) P <<= 1;
    return P;
}

hipError_t launch_topt(const float *smap, int B, int nf, int t, TopTState *st, unsigned long long *keys,
                       mdk_sortscore *out, const int *rot_id, const int *boff, hipStream_t s) {
    if (B < 1) return hipSuccess;
    const unsigned n3 = (unsigned)nf * nf * nf;
    const float nf3f = (float)n3;
    const unsigned rank = (unsigned)t < n3 ? (unsigned)t : n3;
    const unsigned P = topt_sort_size(t, nf);
    if (rank <= (unsigned)kWideT) {
        const dim3 wide((n3 + kWideChunk - 1) / kWideChunk, B);
        k_wide_hist<<<wide, 1024, 0, s>>>(smap, n3, st, keys);
        k_wide_pick<<<B, 1024, 0, s>>>(st, keys, rank, nf3f);
        k_wide_compact<<<wide, 1024, 0, s>>>(smap, n3, nf3f, st, keys);
        k_wide_value<<<kTieBlocks, kTieThreads, 0, s>>>(smap, n3, nf3f, st, keys, rank);
        k_wide_ties<<<kTieBlocks, kTieThreads, 0, s>>>(smap, n3, nf3f, st, keys, rank);
        k_tsel_sort_out<<<B, 1024, 0, s>>>(keys, P, 0u, st, t, nf, out, rot_id, boff);
        return hipGetLastError();
    }
    const dim3 grid((n3 + kChunk - 1) / kChunk, B);
    k_tsel_init<<<B, 256, 0, s>>>(st, rank);
    for (int shift = 56; shift >= 0; shift -= 8) {
        k_tsel_hist<<<grid, 256, 0, s>>>(smap, n3, nf3f, st, shift);
        k_tsel_pick<<<B, 256, 0, s>>>(st, shift);
    }
    k_tsel_compact<<<grid, 256, 0, s>>>(smap, n3, nf3f, st, keys, P);
    k_tsel_sort_out<<<B, 1024, 0, s>>>(keys, P, P, st, t, nf, out, rot_id, boff);
    return hipGetLastError();
}
