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
// A rotation with more of them than fit (many equal scores) is selected by one workgroup with
// the levels above.
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
    if (threadIdx.x == 0) st[blockIdx.x].count = 0u;
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
        atomicAdd(&h[sortable(v.x + 0.0f) >> kWideShift], 1u);
        atomicAdd(&h[sortable(v.y + 0.0f) >> kWideShift], 1u);
        atomicAdd(&h[sortable(v.z + 0.0f) >> kWideShift], 1u);
        atomicAdd(&h[sortable(v.w + 0.0f) >> kWideShift], 1u);
    }
    __syncthreads();
    unsigned *g = reinterpret_cast<unsigned *>(keys + (size_t)blockIdx.y * kTSortLds);
    for (int q = threadIdx.x; q < kWideBuckets; q += 1024)
        if (h[q]) atomicAdd(&g[q], h[q]);
}

// one workgroup per rotation: the score below which nothing reaches the top `rank` (its bits in
// st.prefix)
__global__ void __launch_bounds__(1024) k_wide_pick(TopTState *st, const unsigned long long *keys, unsigned rank,
                                                    float nf3f) {
    constexpr int PER = kWideBuckets / 1024;
    __shared__ unsigned cum[1024];
    const unsigned *h = reinterpret_cast<const unsigned *>(keys + (size_t)blockIdx.x * kTSortLds);
    const int top = kWideBuckets - 1 - (int)threadIdx.x * PER;  // this thread's buckets: top, top - 1, ...
    unsigned n[PER], s = 0u;
    for (int q = 0; q < PER; q++) s += n[q] = h[top - q];
    cum[threadIdx.x] = s;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {
        const unsigned add = (int)threadIdx.x >= d ? cum[threadIdx.x - d] : 0u;
        __syncthreads();
        cum[threadIdx.x] += add;
        __syncthreads();
    }
    unsigned c = cum[threadIdx.x] - s;  // entries above this thread's buckets
    if (c < rank && cum[threadIdx.x] >= rank) {
        int q = 0;
        while (c + n[q] < rank) c += n[q++];
        const unsigned long long edge = (unsigned long long)((unsigned)(top - q) << kWideShift) << 32;
        st[blockIdx.x].prefix = __float_as_uint(quotient_cut(key_float(edge), nf3f));
    }
}

// grid (chunks, B): the keys of the scores not below the cut (a score that is not a number is
// not), as many as fit
__global__ void __launch_bounds__(1024) k_wide_compact(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                       TopTState *st, unsigned long long *keys) {
    TopTState &s = st[blockIdx.y];
    const float cut = __uint_as_float((unsigned)s.prefix);
    const float4 *m = reinterpret_cast<const float4 *>(smap + (size_t)blockIdx.y * n3);
    unsigned long long *out = keys + (size_t)blockIdx.y * kTSortLds;
    auto put = [&](float v, unsigned i) {
        if (!(v < cut)) {
            const unsigned k = atomicAdd(&s.count, 1u);
            if (k < (unsigned)kTSortLds) out[k] = topt_key(v, nf3f, i);
        }
    };
    const unsigned i0 = blockIdx.x * (kWideChunk / 4), i1 = min(n3 / 4, i0 + kWideChunk / 4);
    for (unsigned i = i0 + threadIdx.x; i < i1; i += 1024u) {
        const float4 v = m[i];
        if (!(v.x < cut && v.y < cut && v.z < cut && v.w < cut)) {
            put(v.x, 4 * i);
            put(v.y, 4 * i + 1);
            put(v.z, 4 * i + 2);
            put(v.w, 4 * i + 3);
        }
    }
}

// A rotation whose keys did not fit: the radix select of the levels by one workgroup, whose keys
// (exactly rank of them) replace the list.
__global__ void __launch_bounds__(1024) k_wide_slow(const float *__restrict__ smap, unsigned n3, float nf3f,
                                                    TopTState *st, unsigned long long *keys, unsigned rank) {
    __shared__ unsigned h[256], n;
    __shared__ unsigned long long prefix, mask;
    __shared__ unsigned want;
    __shared__ bool done;
    const int b = blockIdx.x;
    if (st[b].count <= (unsigned)kTSortLds) return;  // uniform
    const float *m = smap + (size_t)b * n3;
    if (threadIdx.x == 0) {
        prefix = mask = 0ull;
        want = rank;
        n = 0u;
        done = false;
    }
    for (int shift = 56; shift >= 0; shift -= 8) {
        if (threadIdx.x < 256) h[threadIdx.x] = 0u;
        __syncthreads();
        const unsigned long long p = prefix, k0 = mask;
        for (unsigned i = threadIdx.x; i < n3; i += 1024u) {
            const unsigned long long k = topt_key(m[i], nf3f, i);
            if ((k & k0) == p) atomicAdd(&h[(unsigned)(k >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned c = 0u;
            int d = 255;
            while (d > 0 && c + h[d] < want) c += h[d--];
            prefix |= (unsigned long long)d << shift;
            mask |= 255ull << shift;
            want -= c;
            done = want == h[d];  // the whole bucket is wanted
        }
        __syncthreads();
        if (done) break;  // uniform
    }
    const unsigned long long thr = prefix;
    unsigned long long *out = keys + (size_t)b * kTSortLds;
    for (unsigned i = threadIdx.x; i < n3; i += 1024u) {
        const unsigned long long k = topt_key(m[i], nf3f, i);
        if (k >= thr) out[atomicAdd(&n, 1u)] = k;
    }
    __syncthreads();
    if (threadIdx.x == 0) st[b].count = n;
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
        k_wide_slow<<<B, 1024, 0, s>>>(smap, n3, nf3f, st, keys, rank);
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
