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
// A rotation with more of them than fit (many equal scores) is selected by levels of 12 bits
// (k_wide_level), all workgroups sharing those rotations.
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
constexpr int kLevels = 5, kLevelBuckets = 4096, kLevelBlocks = 512;  // two workgroups a CU
static_assert(3 * kLevelBuckets * sizeof(unsigned) <= kTSortLds * sizeof(unsigned long long) &&
                  kWideT * sizeof(unsigned long long) <= kLevelBuckets * sizeof(unsigned),
              "the levels' histograms lie where the keys go, the last one picked clear of the keys written");
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

// ---- wide select; a rotation's histogram lies at the start of its keys
__global__ void __launch_bounds__(1024) k_wide_init(TopTState *st, unsigned long long *keys) {
    unsigned *h = reinterpret_cast<unsigned *>(keys + (size_t)blockIdx.x * kTSortLds);
    for (int q = threadIdx.x; q < kWideBuckets; q += 1024) h[q] = 0u;
    if (threadIdx.x == 0) st[blockIdx.x].count = st[blockIdx.x].nover = 0u;
}

// grid (chunks, B); n3 is a multiple of 8 (nf is even)
__global__ void __launch_bounds__(1024) k_wide_hist(const float *__restrict__ smap, unsigned n3, unsigned long long *keys) {
    __shared__ unsigned h[kWideBuckets];
    for (int q = threadIdx.x; q < kWideBuckets; q += 1024) h[q] = 0u;
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
// the rotation's first level histogram is cleared
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
        S.over = over;
        if (over) st[atomicAdd(&st[0].nover, 1u)].nth_over = blockIdx.x;
    }
    __syncthreads();
    if (over)
        for (int q = threadIdx.x; q < kLevelBuckets; q += 1024) h[q] = 0u;
}

// grid (chunks, B): the keys of the scores not below the cut, of rotations where they fit
__global__ void __launch_bounds__(1024) k_wide_compact(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                       TopTState *st, unsigned long long *keys) {
    TopTState &s = st[blockIdx.y];
    if (s.over) return;  // uniform
    const unsigned cut = (unsigned)s.prefix;
    const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)blockIdx.y * n3);
    unsigned long long *out = keys + (size_t)blockIdx.y * kTSortLds;
    auto put = [&](float v, unsigned i) {
        if (sortable_score(v) >= cut) out[atomicAdd(&s.count, 1u)] = topt_key(v, nf3f, i);
    };
    const unsigned i0 = blockIdx.x * (kWideChunk / 4), i1 = min(n3 / 4, i0 + kWideChunk / 4);
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

// Rotations whose keys do not fit: radix select of the keys
//   sortable(score / nf^3) << 28 | (2^28 - 1 - index)          (60 bits; nf <= 640)
// by five levels of 12 bits, a launch each, whose workgroups share out those rotations (with one
// rotation all of them read its map).  A launch first picks the last level's digit of its
// rotation, each workgroup for itself, from the histogram that the launch before left; the
// sixth (level 5) writes the keys from the threshold on, rank of them.  The histograms take turns in three
// places of the rotation's keys: level l - 1 is read, l added to, l + 1 cleared.  Without such
// rotations a launch ends at its first load: six of them take 10-14 us of a call of one rotation, under 1%
// of a search (112^3, 1024 rotations on two streams: 11.77 ms without, 11.86 with).  Docking one rotation
// with every score equal, t = 64, took 9.1 ms at 112^3 and 106 at 256^3 with one workgroup that read the
// map nine times, 0.30 and 0.77 with levels of 8 bits in 17 launches over every rotation, and takes 0.19
// and 0.41; 128 such rotations of 112^3 14.3, 5.8 and 3.1 (with 256 threads a workgroup 4.2, in twice as many 3.4).
__device__ __forceinline__ unsigned long long level_key(float v, float nf3f, unsigned i) {
    return ((unsigned long long)sortable(v / nf3f + 0.0f) << 28) | (0xfffffffu - i);
}

__global__ void __launch_bounds__(1024) k_wide_level(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                     TopTState *st, unsigned long long *keys, unsigned rank, int level) {
    __shared__ unsigned h[kLevelBuckets], wave_sum[16], picked[3];
    const unsigned n = st[0].nover, parts = max(1u, gridDim.x / max(n, 1u));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned part = n < gridDim.x ? blockIdx.x / max(n, 1u) : 0u;
    if (part >= parts) return;  // uniform, as all that follows but the entries
    for (unsigned q = n < gridDim.x ? blockIdx.x % max(n, 1u) : blockIdx.x; q < n; q += gridDim.x) {
        const unsigned b = st[q].nth_over;
        TopTState &S = st[b];
        unsigned long long *out = keys + (size_t)b * kTSortLds;
        unsigned *hist = reinterpret_cast<unsigned *>(out);
        unsigned long long prefix = 0ull;
        unsigned want = rank;
        if (level > 0) {
            prefix = S.level_prefix[level - 1];
            want = S.level_wanted[level - 1];
        }
        if (level > 0 && want > 0) {
            // this thread's buckets: 4095 - 4 tid downwards
            const unsigned *last = hist + (level - 1) % 3 * kLevelBuckets;
            const uint4 v = reinterpret_cast<const uint4 *>(last)[1023 - tid];
            const unsigned s = v.x + v.y + v.z + v.w;
            unsigned c = s;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const unsigned o = __shfl_up(c, d, 64);
                if (lane >= d) c += o;
            }
            if (lane == 63) wave_sum[wave] = c;
            __syncthreads();
            for (int w = 0; w < wave; w++) c += wave_sum[w];
            const unsigned above = c - s;
            if (above < want && c >= want) {
                const unsigned in[4] = {v.w, v.z, v.y, v.x};
                unsigned digit = kLevelBuckets - 1 - 4 * tid, a = above, here = in[0];
#pragma unroll
                for (int k = 1; k < 4; k++)
                    if (a + here < want) {
                        a += here;
                        here = in[k];
                        digit--;
                    }
                picked[0] = digit;
                picked[1] = want - a;
                picked[2] = want - a == here;  // the whole bucket is wanted
            }
            __syncthreads();
            prefix |= (unsigned long long)picked[0] << (60 - 12 * level);
            want = picked[2] ? 0u : picked[1];
            __syncthreads();  // the next rotation writes them
        }
        // this workgroup's share of the map, in fours
        const unsigned share = (n3 / 4 + parts - 1) / parts, i0 = part * share, i1 = min(n3 / 4, i0 + share);
        const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)b * n3);
        if (level == kLevels) {
            for (unsigned i = i0 + tid; i < i1; i += 1024u) {
                const float4 f = m[i];
                const float e[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                for (int k = 0; k < 4; k++)
                    if (level_key(e[k], nf3f, 4 * i + k) >= prefix)
                        out[atomicAdd(&S.count, 1u)] = topt_key(e[k], nf3f, 4 * i + k);
            }
            continue;
        }
        if (part == 0) {
            if (tid == 0) {
                S.level_prefix[level] = prefix;
                S.level_wanted[level] = want;
            }
            for (int k = tid; k < kLevelBuckets; k += 1024) hist[(level + 1) % 3 * kLevelBuckets + k] = 0u;
        }
        if (want == 0u) continue;
        for (int k = tid; k < kLevelBuckets; k += 1024) h[k] = 0u;
        __syncthreads();
        const int shift = 48 - 12 * level;
        for (unsigned i = i0 + tid; i < i1; i += 1024u) {
            const float4 f = m[i];
            const float e[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned long long key = level_key(e[k], nf3f, 4 * i + k);
                const bool in = level == 0 || key >> (shift + 12) == prefix >> (shift + 12);
                const int digit = (int)(key >> shift) & (kLevelBuckets - 1);
                // equal digits are the rule here: one lane adds for all that have the first one's
                const unsigned long long some = __ballot(in);
                if (some == 0ull) continue;
                const int first = __ffsll((long long)some) - 1, d0 = __builtin_amdgcn_readlane(digit, first);
                const unsigned long long same = __ballot(in && digit == d0);
                if (lane == first) atomicAdd(&h[d0], (unsigned)__popcll(same));
                else if (in && digit != d0) atomicAdd(&h[digit], 1u);
            }
        }
        __syncthreads();
        for (int k = tid; k < kLevelBuckets; k += 1024)
            if (h[k]) atomicAdd(&hist[level % 3 * kLevelBuckets + k], h[k]);
        __syncthreads();  // the next rotation clears h
    }
}

// one workgroup per rotation: descending bitonic sort of its P keys (padded with 0, which
// sorts last; P = 0: of its count rounded up to a power of two, at most kTSortLds), then the
// rotation's t results; a rotation's keys lie `stride` apart
__global__ void __launch_bounds__(1024) k_tsel_sort_out(unsigned long long *keys, unsigned stride, unsigned P,
                                                        const TopTState *st, int t, int nf, mdk_sortscore *__restrict__ out,
                                                        const int *__restrict__ rot_id, const int *__restrict__ boff) {
    __shared__ unsigned long long sl[kTSortLds];
    const int b = blockIdx.x;
    const unsigned n = st[b].count;
    unsigned long long *g = keys + (size_t)b * stride;
    if (P == 0u)
        for (P = 1u; P < n;) P <<= 1;
    const bool lds = P <= (unsigned)kTSortLds;
    unsigned long long *s = lds ? sl : g;
    for (unsigned i = threadIdx.x; i < P; i += 1024u) s[i] = i < n ? g[i] : 0ull;
    __syncthreads();
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
        k_wide_init<<<B, 1024, 0, s>>>(st, keys);
        k_wide_hist<<<wide, 1024, 0, s>>>(smap, n3, keys);
        k_wide_pick<<<B, 1024, 0, s>>>(st, keys, rank, nf3f);
        k_wide_compact<<<wide, 1024, 0, s>>>(smap, n3, nf3f, st, keys);
        for (int level = 0; level <= kLevels; level++)
            k_wide_level<<<kLevelBlocks, 1024, 0, s>>>(smap, n3, nf3f, st, keys, rank, level);
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
