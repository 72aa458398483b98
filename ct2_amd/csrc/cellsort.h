// cellsort.h -- the particles of an index range in the order of a cell key, as
// records (x, y, z, position in the range), stable: inside a cell the positions
// ascend, so the order does not depend on scheduling.
//
// Least-significant-digit counting sort of the records themselves, digits of up
// to 11 bits: the keys of the grids in use (18 to 22 bits) take two passes.  A
// pass is a count of each tile's digits, their prefix over the tiles, and the
// placement: a tile's records stay in registers, a wave ranks 64 of them at a
// time by matching digits with ballots, and its counters lie in LDS.  Bound by
// the 16-byte records' way to memory and back, in runs of (tile / digits) of
// them; the keys are formed again from the positions in every kernel, and no
// gather by index follows.  2^21 records on 64^3 cells (18-bit keys): 69 us, and 8
// for the starts; keys and indices through a library radix sort of three passes
// with fills between them, then a gather and a search per cell, took 150 and 9.
#pragma once

#include "internal.h"
#include "wave.h"

namespace ct2 {
namespace cellsort {

constexpr int THREADS = 1024, WAVES = THREADS / 64;
constexpr int DIGIT_BITS = 11;
constexpr int FEW_TILES = 32;  // so few that the placement sums their counts itself

struct Soa {  // the container's positions
    const uint32_t *x, *y, *z;
    __device__ __forceinline__ uint4 operator()(long e) const { return make_uint4(x[e], y[e], z[e], (uint32_t)e); }
};
struct Records {
    const uint4* r;
    __device__ __forceinline__ uint4 operator()(long e) const { return r[e]; }
};

// cnt[tile][digit]
template <int ITEMS, typename SRC, typename KEY>
__global__ __launch_bounds__(THREADS) void count(SRC src, KEY key, int n, int shift, int dbits, int* __restrict__ cnt) {
    __shared__ int h[1 << DIGIT_BITS];
    const int D = 1 << dbits;
    const long e0 = (long)blockIdx.x * (ITEMS * THREADS) + threadIdx.x;
    uint32_t k[ITEMS];
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
        const long e = e0 + u * THREADS;
        k[u] = e < n ? key(src(e)) >> shift & (D - 1) : ~0u;
    }
    for (int d = threadIdx.x; d < D; d += THREADS) h[d] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ITEMS; ++u)
        if (k[u] != ~0u) atomicAdd(&h[k[u]], 1);
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += THREADS) cnt[(size_t)blockIdx.x * D + d] = h[d];
}

// cnt[tile][digit] -> the digit's records in the tiles before; total[digit].  16
// digits a workgroup, 64 threads to each.
constexpr int PREFIX_DIGITS = 16, PREFIX_GROUPS = THREADS / PREFIX_DIGITS;
static __global__ __launch_bounds__(THREADS) void prefix(int* __restrict__ cnt, int tiles, int D, int* __restrict__ total) {
    __shared__ int red[PREFIX_GROUPS][PREFIX_DIGITS];
    const int k = threadIdx.x % PREFIX_DIGITS, g = threadIdx.x / PREFIX_DIGITS;
    const int d = blockIdx.x * PREFIX_DIGITS + k;
    const int per = (tiles + PREFIX_GROUPS - 1) / PREFIX_GROUPS;
    const int b = min(tiles, g * per), e = d < D ? min(tiles, b + per) : b;
    int s = 0;
#pragma unroll 8
    for (int t = b; t < e; ++t) s += cnt[(size_t)t * D + d];
    red[g][k] = s;
    __syncthreads();
    int run = 0, all = 0;
    for (int q = 0; q < PREFIX_GROUPS; ++q) {
        if (q < g) run += red[q][k];
        all += red[q][k];
    }
    if (g == 0 && d < D) total[d] = all;
    constexpr int AHEAD = 8;  // counts read together: the stores would otherwise hold back the next loads
    for (int t0 = b; t0 < e; t0 += AHEAD) {
        int v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = t0 + u < e ? cnt[(size_t)(t0 + u) * D + d] : 0;
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (t0 + u < e) cnt[(size_t)(t0 + u) * D + d] = run;
            run += v[u];
        }
    }
}

// Places a tile's records.  cnt, total: after `prefix`; total null: the counts
// of at most FEW_TILES tiles as they are; cnt null: the only tile.
template <int ITEMS, typename SRC, typename KEY>
__global__ __launch_bounds__(THREADS) void place(SRC src, KEY key, int n, int shift, int dbits, int tiles,
                                                 const int* __restrict__ cnt, const int* __restrict__ total,
                                                 uint4* __restrict__ out) {
    typedef uint32_t __attribute__((may_alias)) word;           // two neighbouring counters
    __shared__ __align__(4) uint16_t h[WAVES << DIGIT_BITS];  // [wave][digit]
    __shared__ int first[1 << DIGIT_BITS];               // where the tile's records of a digit start
    __shared__ int part[WAVES];
    word* const h32 = (word*)h;
    const int D = 1 << dbits, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int tile = (int)blockIdx.x;
    const long e0 = (long)tile * (ITEMS * THREADS) + w * (ITEMS * 64) + lane;
    uint4 r[ITEMS];
#pragma unroll
    for (int u = 0; u < ITEMS; ++u)
        r[u] = e0 + u * 64 < n ? src(e0 + u * 64) : make_uint4(0u, 0u, 0u, 0u);
    for (int i = tid; i < WAVES * D / 2; i += THREADS) h32[i] = 0u;
    __syncthreads();
    uint16_t* const hw = h + w * D;
    uint32_t at[ITEMS];  // digit << 16 | rank among the wave's records of it
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
        const bool have = e0 + u * 64 < n;
        const uint32_t d = have ? key(r[u]) >> shift & (D - 1) : 0u;
        uint64_t same = __ballot(have);  // lanes with this digit
        for (int b = 0; b < dbits; ++b) {
            const bool bit = d >> b & 1;
            const uint64_t v = __ballot(bit);
            same &= bit ? v : ~v;
        }
        const uint32_t rank =
            __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
        const uint32_t before = hw[d];
        wave_sync();
        if (have && rank == 0) hw[d] = (uint16_t)(before + (uint32_t)__popcll(same));
        wave_sync();
        at[u] = d << 16 | (before + rank);
    }
    __syncthreads();
    // thread t takes digits 2t and 2t + 1: their counts over the waves (both
    // halves of a word at once), and the records before them
    int v0 = 0, v1 = 0, b0 = 0, b1 = 0;
    const int d0 = 2 * tid;
    if (d0 < D) {
        uint32_t run = 0;
        for (int q = 0; q < WAVES; ++q) {
            const uint32_t v = h32[(q * D + d0) / 2];
            h32[(q * D + d0) / 2] = run;
            run += v;
        }
        if (!cnt) {
            v0 = (int)(run & 0xffffu);
            v1 = (int)(run >> 16);
        } else if (total) {
            const int2 c = *(const int2*)(cnt + (size_t)tile * D + d0), a = *(const int2*)(total + d0);
            b0 = c.x;
            b1 = c.y;
            v0 = a.x;
            v1 = a.y;
        } else {
#pragma unroll 8
            for (int t = 0; t < tiles; ++t) {
                const int2 c = *(const int2*)(cnt + (size_t)t * D + d0);
                b0 += t < tile ? c.x : 0;
                b1 += t < tile ? c.y : 0;
                v0 += c.x;
                v1 += c.y;
            }
        }
    }
    int s = v0 + v1;  // inclusive over the wave, then over the waves
    for (int off = 1; off < 64; off <<= 1) {
        const int q = __shfl_up(s, off);
        if (lane >= off) s += q;
    }
    if (lane == 63) part[w] = s;
    __syncthreads();
    if (d0 < D) {
        int run = s - v0 - v1;
        for (int q = 0; q < w; ++q) run += part[q];
        first[d0] = run + b0;
        first[d0 + 1] = run + v0 + b1;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < ITEMS; ++u) {
        const uint32_t d = at[u] >> 16;
        if (e0 + u * 64 < n) out[first[d] + (int)hw[d] + (int)(at[u] & 0xffffu)] = r[u];
    }
}

template <int ITEMS, typename SRC, typename KEY>
int pass(SRC src, KEY key, int n, int shift, int dbits, int* cnt, uint4* out, hipStream_t st) {
    const int tiles = (int)(((long)n + ITEMS * THREADS - 1) / (ITEMS * THREADS)), D = 1 << dbits;
    int* total = nullptr;
    if (tiles == 1) {
        cnt = nullptr;
    } else {
        count<ITEMS><<<tiles, THREADS, 0, st>>>(src, key, n, shift, dbits, cnt);
        CT2_LAUNCH_CHECK();
        if (tiles > FEW_TILES) {
            total = cnt + (size_t)tiles * D;
            prefix<<<(D + PREFIX_DIGITS - 1) / PREFIX_DIGITS, THREADS, 0, st>>>(cnt, tiles, D, total);
            CT2_LAUNCH_CHECK();
        }
    }
    place<ITEMS><<<tiles, THREADS, 0, st>>>(src, key, n, shift, dbits, tiles, cnt, total, out);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

template <int ITEMS, typename KEY>
int run(Soa src, KEY key, int n, int bits, uint4* out, uint4* other, void** scratch, size_t* have, hipStream_t st) {
    const int passes = (bits + DIGIT_BITS - 1) / DIGIT_BITS, dbits = (bits + passes - 1) / passes;
    const size_t tiles = ((size_t)n + ITEMS * THREADS - 1) / (ITEMS * THREADS);
    CT2_TRY(ensure_scratch(scratch, have, ((tiles + 1) << dbits) * sizeof(int), "cell sort counts"));
    for (int p = 0; p < passes; ++p) {
        uint4* const to = (passes - p) % 2 ? out : other;
        if (p == 0)
            CT2_TRY(pass<ITEMS>(src, key, n, 0, dbits, (int*)*scratch, to, st));
        else
            CT2_TRY(pass<ITEMS>(Records{to == out ? other : out}, key, n, p * dbits, dbits, (int*)*scratch, to, st));
    }
    return CT2_OK;
}

}  // namespace cellsort

// out[0 .. n): the records of positions (x, y, z)[0 .. n) in ascending order of
// key(record), a key of `bits` bits (at least 1), equal keys in the order they
// came.  other: n more records of room; scratch: grown as ensure_scratch does.
template <typename KEY>
int cell_sort(const uint32_t* x, const uint32_t* y, const uint32_t* z, int n, KEY key, int bits, uint4* out,
              uint4* other, void** scratch, size_t* have, hipStream_t st) {
    // tiles of 8,192 records, in longer runs to memory, where they make a workgroup
    // for every CU; below, of 2,048, for more of them
    const cellsort::Soa src{x, y, z};
    return n >= 1 << 21 ? cellsort::run<8>(src, key, n, bits, out, other, scratch, have, st)
                        : cellsort::run<2>(src, key, n, bits, out, other, scratch, have, st);
}

// put(q, s) for q = 0 .. nkeys: the first place s of the sorted records whose key
// is at least q (n for q = nkeys).  cell_starts_fill: a thread per record writes
// those of the keys since the one before it, a wave together where they are many,
// and of SEGMENT keys and more (sets that leave most of the box empty) the waves of
// the first `segments` blocks, each its own SEGMENT keys of them: such a gap holds
// the first or the last key of every segment that it meets.  2^21 records and
// keys: 13 us uniform, 11 with all records under one key (12 and 420 with every gap
// one wave's).  cell_starts_search: a binary search per key (35 and 20 us of those),
// for grids that are mostly empty.
constexpr int SEGMENT = 1024;

// The first place of a key of at least q, by the 32 lanes of a half wave that share q.
template <typename KEY>
__device__ __forceinline__ int first_by_half(const uint4* __restrict__ P, const KEY& key, int n, long q) {
    const int lane = threadIdx.x & 63;
    int lo = 0, len = n;  // it lies in lo .. lo + len
    while (__any(len > 0)) {
        const int step = len / 32 + (len % 32 != 0), i = (lane & 31) * step;
        const uint64_t below = __ballot(i < len && (long)key(P[lo + i]) < q);
        const int c = __popc((uint32_t)(lane < 32 ? below : below >> 32));  // lane 0's to lane c - 1's
        const int skip = c > 0 ? (c - 1) * step + 1 : 0;
        len = c == 0 ? 0 : (c < 32 ? min(c * step, len) : len) - skip;
        lo += skip;
    }
    return lo;
}

template <typename KEY, typename PUT>
__global__ __launch_bounds__(256) void cell_starts_fill(const uint4* __restrict__ P, KEY key, int n, long nkeys, PUT put,
                                                        unsigned segments) {
    const int lane = threadIdx.x & 63;
    // keys a .. b start at the records at e
    auto gap = [&](long e, long& a, long& b) {
        a = e > 0 ? (long)key(P[e - 1]) + 1 : 0;
        b = e < n ? (long)key(P[e]) : nkeys;
    };
    if (blockIdx.x < segments) {
        const long q0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * SEGMENT;
        if (q0 > nkeys) return;
        const long q1 = min(q0 + SEGMENT - 1, nkeys);
        const long e = first_by_half(P, key, n, lane < 32 ? q0 : q1);
        long a, b;
        gap(e, a, b);
        const long e1 = __shfl(e, 32);
        for (int l = 0; l < 64; l += 32) {
            const long ea = __shfl(a, l), eb = __shfl(b, l), ee = __shfl(e, l);
            if (eb - ea >= SEGMENT - 1)
                for (long q = max(ea, q0) + lane; q <= min(eb, q1); q += 64) put(q, ee);
            if (ee == e1) break;  // one gap holds both ends
        }
        return;
    }
    const long e = (long)(blockIdx.x - segments) * 256 + threadIdx.x;
    long a = 0, b = -1;
    if (e <= n) gap(e, a, b);
    constexpr int ALONE = 16;
    const bool many = b - a >= ALONE;
    if (!many)
        for (long q = a; q <= b; ++q) put(q, e);
    for (uint64_t m = __ballot(many && b - a < SEGMENT - 1); m; m &= m - 1) {
        const int l = __ffsll((unsigned long long)m) - 1;
        const long ea = __shfl(a, l), eb = __shfl(b, l), ee = __shfl(e, l);
        for (long q = ea + lane; q <= eb; q += 64) put(q, ee);
    }
}

template <typename KEY, typename PUT>
__global__ __launch_bounds__(256) void cell_starts_search(const uint4* __restrict__ P, KEY key, int n, long nkeys, PUT put) {
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q > nkeys) return;
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = lo + (hi - lo) / 2;
        if ((long)key(P[mid]) < q)
            lo = mid + 1;
        else
            hi = mid;
    }
    put(q, (long)lo);
}

template <typename KEY, typename PUT>
int cell_starts(const uint4* P, KEY key, int n, long nkeys, PUT put, hipStream_t st) {
    if (nkeys > 4L * n) {
        cell_starts_search<<<(unsigned)((nkeys + 256) / 256), 256, 0, st>>>(P, key, n, nkeys, put);
    } else {
        const unsigned records = (unsigned)(((long)n + 256) / 256), segments = (unsigned)(nkeys / (4 * SEGMENT) + 1);
        cell_starts_fill<<<segments + records, 256, 0, st>>>(P, key, n, nkeys, put, segments);
    }
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

}  // namespace ct2
