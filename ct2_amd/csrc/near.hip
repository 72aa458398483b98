// near.hip -- the near field of the PM force on gfx950: a direct pair sum over
// cell neighbourhoods beside the mesh far field, the structure of ct2's kick()
// (kick.cpp:105-125: neighbour list at :117, direct pairs through kick_cell
// :36-67, far field from the mesh expansion at :118 and :29).
//
// The Gaussian-filtered PM force (pm.hip) already carries, for every pair, the
// filtered Newtonian kernel phi_long = erf(u)/r, u = r/(2 rs).  For each
// minimum-image pair closer than rcut the near field adds the softened kernel
// minus that:
//     F += GM dx (k_soft(r) - [erf(u) - (2u/sqrt(pi)) e^{-u^2}] / r^3)
//     pot += GM (p_soft(r) - erf(u)/r)
// and the potential drops the background integral GM N 4 pi rs^2, so that
// PM + near field tends to the periodic direct sum.
//
// Pipeline (all on the library stream, deterministic):
//   cell_sort     the particles as (x, y, z, index) records, sorted stably by
//                 slice key ((x, y) column, then z slice, NEAR_SUB per cell):
//                 the order is (column, slice, particle index) for any
//                 scheduling and any clustering, so the summation order never
//                 depends on atomics (cellsort.h)
//   cell_starts   start of every slice and cell
//   near_scan     exclusive scan over the rows -> work-item prefix (runs of
//                 NEAR_SINKS sinks per row)
//   near_items    the (row, run) of every work item
//   near_force    one wave per work item: 16 sinks, each in four lanes that
//                 take every fourth source; the 9 (or 25) neighbouring rows'
//                 slice ranges read 64 sources at a time; sources farther than
//                 rcut from the sinks' bounding box are dropped and the rest
//                 gathered in an LDS ring, 64 per tile; the filtered kernel
//                 from cubic pieces in LDS, FP32 pair terms with TwoSum per 64
//                 terms; adds into the stored force of each particle.
// Cells have side >= rcut, so every partner of a sink lies in the 3x3x3 cells
// around it; a work item's sinks span a run of slices along z in one row, and
// the union of their neighbourhoods is 9 contiguous (or wrapped) slice ranges
// of the sorted array, each widened by the slices rcut spans.
#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

#include "cellsort.h"
#include "internal.h"
#include "wave.h"

namespace ct2 {
namespace {

constexpr int NEAR_SINKS = 16;  // sinks per work item (see near_force)
constexpr int NEAR_TILE = 64;   // sources tested at a time (one per lane), and summed at a time
constexpr int NEAR_WAVES = 4;   // waves (work items) per workgroup
constexpr int NEAR_MAX_NC = 64;  // cells per side at most (along z; x and y: NEAR_MAX_NC * F)
// Cells of more than NEAR_SPLIT_DENSITY particles on average are split F = 2
// ways in x and y, so a work item's sinks span a squarer box (a quarter of the
// cross-section, four times the z extent); partners then lie in the 5 x 5
// neighbouring columns.  Below that density a column's range holds too few
// sources to fill the tiles it is tested in.  Near field with F = 1 / 2, ms:
// 8 per cell (2^21 particles, 256^3 grid, rs 1, to 4 rs) 0.55 / 1.05; 22 (2^21
// clustered, 512^3) 8.11 / 7.90; 70 (2^21, 256^3, rs 1.5, to 5.5 rs) 1.35 / 1.25;
// 172 (2^24, 512^3, rs 2) 20.2 / 16.7.
constexpr int NEAR_SPLIT_DENSITY = 16;
constexpr int NEAR_MAX_ROWS = 25;  // (2F + 1)^2
// Each cell is cut into NEAR_SUB slices along z; a cell's segment is ordered
// by (slice, particle index), so a row's particles are in slice order and a
// work item's neighbour ranges start and end at slice boundaries.
#ifndef NEAR_SUB_N
#define NEAR_SUB_N 16
#endif
constexpr int NEAR_SUB = NEAR_SUB_N;
// The filtered Newtonian kernel is evaluated from NEAR_NT + 1 cubic pieces of
// its potential in r^2 over [0, rcut^2] (built on the host in FP64 by
// near_potential_table).  Force error of the pieces, relative to the force's value,
// before and after their coefficients are rounded to FP32: 8e-10 and 6e-8 to 4 rs,
// 6e-9 and 6e-8 to 5.5 rs, 5e-8 and 1e-7 to 8 rs; beyond, where the pieces are long
// against rs, 6e-7 to 12 rs, 1.3e-5 to 20 rs and 1e-2 to 64 rs, the largest cutoff;
// the potential's is smaller.  Fewer, quartic pieces
// (64, 20 bytes to gather) or 64 pieces each of force and potential (32 bytes)
// cost more LDS and VALU per pair.
constexpr int NEAR_NT = 512;
constexpr int SCAN_THREADS = 1024;

struct NearState {
    double rcut_rs = 0.0;  // 0 = off
    int nc = 0;
    size_t cap = 0;                // particles the buffers hold
    uint4* P0 = nullptr;           // [cap] the sort's second buffer
    uint4* P = nullptr;            // [cap] sorted (x, y, z, index)
    void* sort_tmp = nullptr;      // its counts
    size_t sort_tmp_bytes = 0;
    size_t ncell_cap = 0, nrow_cap = 0;  // cells and (x, y) columns the index buffers hold
    int* start = nullptr;          // [nc^3 + 1]
    int* row_chunk = nullptr;      // [nc^2 + 1]
    int* subst = nullptr;          // [nc^3 NEAR_SUB + 1] sorted index of each slice's first particle
    int2* item = nullptr;          // [cap / NEAR_SINKS + rows] (row, run) per work item
    size_t item_cap = 0;
    float4* table = nullptr;       // [NEAR_NT + 1] p_l pieces (c0..c3)
    double table_rsu = 0.0, table_rcu = 0.0;  // what the table was built for
} g_near;

struct NearConst {
    float rc2u;      // rcut^2 in 2^-64 units
    float rcu;       // rcut in 2^-32 units
    float eps2u;     // Plummer eps^2
    float h2u, hinvu, hinv3u;  // ct2 kernel
    float tscale;    // NEAR_NT / rcut^2: r^2 -> table coordinate
    float kscale;    // 2 tscale: k_l = -kscale dp_l/df, f the table coordinate within a piece
};

__device__ __forceinline__ uint32_t cell_of(uint32_t x, uint32_t nc) {
    return (uint32_t)(((uint64_t)x * nc) >> 32);
}

// z slice of a particle along its row: u = floor(z nzs / 2^32), nzs = nc NEAR_SUB
// slices per row; u / NEAR_SUB is the cell along z.
__device__ __forceinline__ uint32_t slice_of(uint32_t z, uint32_t nzs) {
    return (uint32_t)(((uint64_t)z * nzs) >> 32);
}

// Sort key of a particle: its (x, y) column row = cx nxy + cy and its z
// slice u along the row, key = row nzs + u -- the index of its slice in
// subst (cells: (row nc + u / NEAR_SUB) = key / NEAR_SUB).
struct SliceKey {
    uint32_t nxy, nzs;
    __device__ __forceinline__ uint32_t operator()(const uint4& p) const {
        return (cell_of(p.x, nxy) * nxy + cell_of(p.y, nxy)) * nzs + slice_of(p.z, nzs);
    }
};

// subst[q] = first sorted position with key >= q (q = 0 .. nkeys, subst[nkeys]
// = n), and the cell starts start[c] = subst[c NEAR_SUB].
struct PutSlice {
    int *subst, *start;
    __device__ __forceinline__ void operator()(long q, long e) const {
        subst[q] = (int)e;
        if (q % NEAR_SUB == 0) start[q / NEAR_SUB] = (int)e;
    }
};

// Exclusive scan (one workgroup) of the work items per row: out[0..len],
// out[len] = total; row i holds ceil(m / NEAR_SINKS) items, m = in[(i+1)*nc] -
// in[i*nc] (in = cell starts).
__global__ __launch_bounds__(SCAN_THREADS) void near_scan(const int* __restrict__ in, int len, int nc,
                                                          int* __restrict__ out) {
    __shared__ int part[SCAN_THREADS / 64];
    const int t = threadIdx.x, lane = t & 63;
    int carry = 0;
    for (int b = 0; b < len; b += SCAN_THREADS) {
        const int i = b + t;
        const int v = i < len ? (in[(i + 1) * nc] - in[i * nc] + NEAR_SINKS - 1) / NEAR_SINKS : 0;
        int s = v;  // inclusive scan over the wave, then over the waves
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(s, off);
            if (lane >= off) s += u;
        }
        if (lane == 63) part[t >> 6] = s;
        __syncthreads();
        int before = carry, total = carry;
        for (int k = 0; k < SCAN_THREADS / 64; ++k) {
            if (k < t >> 6) before += part[k];
            total += part[k];
        }
        if (i < len) out[i] = before + s - v;
        carry = total;
        __syncthreads();
    }
    if (t == 0) out[len] = carry;
}

// Softened kernel minus the filtered Newtonian kernel for one pair, in
// 2^-32 units: returns the force factor k (F += dx k) and potential p.  The
// filtered potential p_l comes from cubic pieces in LDS and the filtered force
// from their derivative, k_l = -2 dp_l/d(r^2), so a pair gathers one 16-byte
// entry and no branch depends on the separation beyond the kernel's own.
template <int KERNEL>
__device__ __forceinline__ void near_pair(float r2, const NearConst& q, const float4* tab, float& k, float& p) {
    float ks, ps;
    if constexpr (KERNEL == CT2_KERNEL_PLUMMER) {
        const float w = __builtin_amdgcn_rsqf(r2 + q.eps2u);
        ks = (w * w) * w;
        ps = w;
    } else {
        if (r2 < q.h2u) {
            ks = q.hinv3u;
            ps = fmaf(-0.5f * q.hinv3u, r2, 1.5f * q.hinvu);
        } else {
            const float w = __builtin_amdgcn_rsqf(r2);
            ks = (w * w) * w;
            ps = w;
        }
    }
    // t in [0, NEAR_NT] inside the cutoff; piece i = t rounded to nearest (from
    // the low bits of t + 1.5 2^23), f = t - i in [-1/2, 1/2]
    const float t = r2 * q.tscale, tm = t + 0x1.8p23f;
    const float f = t - (tm - 0x1.8p23f);
    const float4 c = tab[__builtin_bit_cast(int, tm) - 0x4B400000];
    float v = fmaf(c.w, f, c.z), d = fmaf(c.w, f, v);
    v = fmaf(v, f, c.y);
    d = fmaf(d, f, v);
    v = fmaf(v, f, c.x);
    k = fmaf(d, q.kscale, ks);
    p = ps - v;
}

// Work items, one per NEAR_SINKS sinks of a row: item[row_chunk[r] + k] = (r, k); one
// wave per row.
__global__ __launch_bounds__(256) void near_items(const int* __restrict__ row_chunk, int nrow, int2* __restrict__ item) {
    const int r = (blockIdx.x * 256 + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (r >= nrow) return;
    const int k0 = row_chunk[r], k1 = row_chunk[r + 1];
    for (int k = k0 + lane; k < k1; k += 64) item[k] = make_int2(r, k - k0);
}

// One wave per work item of S sinks, NEAR_WAVES waves per workgroup (they share
// the table only).  Lane l holds sink l % S and takes sources l / S, l / S + G,
// ... of every tile of 64 (G = 64 / S streams), so the wave's sinks span a box
// of S particles, not 64, and each sink meets fewer sources out of range; the
// streams' sums are added at the end.  Bound by VALU issue: 10 instructions to
// place a pair, 20 more when it is in range, ~30 to test a tile of candidates
// for a box.  Smaller boxes leave fewer pairs and more tests per sink; 8, 16,
// 32 and 64 sinks took 1.33, 1.25, 1.6 and 1.8 ms near field at 2^21 particles
// (256^3 grid, rs 1.5, to 5.5 rs), 18.4, 16.7, 18.6 and 21.8 at 2^24 (512^3, rs
// 2).  With 64 sinks per wave and 64-bit box tests, and 32 bytes gathered per
// pair for the filtered kernel (LDS busy 72 % of the time), this kernel took
// 1.57 ms of the first, now 1.15 (median of 60 traced passes 1.10).  Sources as exact pairs of floats, to subtract
// instead of converting each separation from integers: 1.52.
template <int KERNEL>
__global__ __launch_bounds__(64 * NEAR_WAVES) void near_force(
    const uint4* __restrict__ P, const int* __restrict__ start, const int* __restrict__ subst,
    const int* __restrict__ row_chunk, const int2* __restrict__ item, int nxy, int nc, int F, int R, NearConst q,
    const float4* __restrict__ table, double fscale, double pscale, double pconst, float* __restrict__ fx,
    float* __restrict__ fy, float* __restrict__ fz, float* __restrict__ pot) {
    constexpr int S = NEAR_SINKS, G = 64 / S;
    __shared__ float4 tab[NEAR_NT + 1];  // the filtered potential's cubic pieces
    __shared__ int rngs[NEAR_WAVES][2 * NEAR_MAX_ROWS][2];
    __shared__ uint4 rings[NEAR_WAVES][2 * NEAR_TILE];  // survivors, consumed a tile at a time from rb
    for (int e = threadIdx.x; e <= NEAR_NT; e += 64 * NEAR_WAVES) {
        tab[e] = table[e];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int b = (int)(blockIdx.y * gridDim.x + blockIdx.x) * NEAR_WAVES + w;
    if (b >= row_chunk[nxy * nxy]) return;  // uniform across the wave; no workgroup barrier follows
    int(*rng)[2] = rngs[w];
    uint4* ring = rings[w];
    const int2 it = item[b];
    const int row = it.x;
    const int s0 = start[row * nc] + it.y * S;
    const int s1 = min(start[(row + 1) * nc], s0 + S);
    const int cx = row / nxy, cy = row % nxy;
    const int side = 2 * F + 1, nr = side * side;  // neighbouring rows: (cx, cy) +- F
    if (lane < nr) {  // one neighbouring row per lane: at most two index ranges (z wraps)
        // the sinks' slices (a row is in slice order) widened by R slices, the
        // most a partner within rcut can differ
        const int Z = nc * NEAR_SUB;
        const int lo = (int)slice_of(P[s0].z, (uint32_t)Z) - R, hi = (int)slice_of(P[s1 - 1].z, (uint32_t)Z) + R;
        const int di = lane / side - F, dj = lane % side - F;
        const int* sr = subst + (((cx + di + nxy) % nxy) * nxy + (cy + dj + nxy) % nxy) * Z;  // slice starts of the row
        int a0, e0, a1 = 0, e1 = 0;
        if (hi - lo + 1 >= Z) {  // the whole row
            a0 = sr[0];
            e0 = sr[Z];
        } else if (lo < 0) {
            a0 = sr[lo + Z];
            e0 = sr[Z];
            a1 = sr[0];
            e1 = sr[hi + 1];
        } else if (hi >= Z) {
            a0 = sr[lo];
            e0 = sr[Z];
            a1 = sr[0];
            e1 = sr[hi - Z + 1];
        } else {
            a0 = sr[lo];
            e0 = sr[hi + 1];
        }
        rng[2 * lane][0] = a0;
        rng[2 * lane][1] = e0;
        rng[2 * lane + 1][0] = a1;
        rng[2 * lane + 1][1] = e1;
    }
    const int i = s0 + lane % S, stream = lane / S;
    const uint4 me = P[i < s1 ? i : s1 - 1];
    float sx = 0.f, sy = 0.f, sz = 0.f, sp = 0.f, cx_ = 0.f, cy_ = 0.f, cz_ = 0.f, cp_ = 0.f;
    // The sinks' bounding box: per axis the offsets [L, H] about a centre cc.
    // A source whose distance to the box is >= rcut has no partner among the
    // sinks and is dropped as its tile is loaded.  The gaps are FP32 and
    // shortened by more than their rounding (2^9 units of 2^-32), so a source
    // with a partner always passes; the pair's own test decides.  An axis whose
    // half-extent plus rcut nears half the box is not tested (there the
    // source's offset from cc could wrap).
    const uint4 ref = P[s0];
    int lo[3] = {(int32_t)(me.x - ref.x), (int32_t)(me.y - ref.y), (int32_t)(me.z - ref.z)};
    int hi[3] = {lo[0], lo[1], lo[2]};
#pragma unroll
    for (int m = S / 2; m >= 1; m >>= 1)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = min(lo[a], __shfl_xor(lo[a], m));
            hi[a] = max(hi[a], __shfl_xor(hi[a], m));
        }
    uint32_t cc[3];
    float L[3], H[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const long long mid = (long long)lo[a] + (((long long)hi[a] - (long long)lo[a]) >> 1);
        cc[a] = (a == 0 ? ref.x : a == 1 ? ref.y : ref.z) + (uint32_t)mid;
        const double l = (double)((long long)lo[a] - mid), h = (double)((long long)hi[a] - mid);
        const bool on = fmax(h, -l) + (double)q.rcu < 0x1p31 - 0x1p24;
        L[a] = on ? (float)l - 512.f : -0x1p33f;
        H[a] = on ? (float)h + 512.f : 0x1p33f;
    }
    const float rc2t = q.rc2u * (1.0f + 0x1p-20f);
    int fill = 0, rb = 0, terms = 0;
    float tx = 0.f, ty = 0.f, tz = 0.f, tp = 0.f;
    auto pair = [&](const uint4 s) {
        const float dx = (float)(int32_t)(s.x - me.x);
        const float dy = (float)(int32_t)(s.y - me.y);
        const float dz = (float)(int32_t)(s.z - me.z);
        const float r2 = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
        if (r2 < q.rc2u) {
            float k, p;
            near_pair<KERNEL>(r2, q, tab, k, p);
            tx = fmaf(dx, k, tx);
            ty = fmaf(dy, k, ty);
            tz = fmaf(dz, k, tz);
            tp += p;
        }
    };
    auto fold = [&]() {
        two_sum(sx, cx_, tx);
        two_sum(sy, cy_, ty);
        two_sum(sz, cz_, tz);
        two_sum(sp, cp_, tp);
        tx = ty = tz = tp = 0.f;
        terms = 0;
    };
    wave_sync();
    // the tiles of the ranges in turn, the next one's sources fetched while
    // this one's are tested and summed
    int r = -1, j0 = 0, e = 0;
    auto next = [&]() {
        j0 += NEAR_TILE;
        while (j0 >= e && ++r < 2 * nr) {
            j0 = __builtin_amdgcn_readfirstlane(rng[r][0]);
            e = __builtin_amdgcn_readfirstlane(rng[r][1]);
        }
    };
    next();
    uint4 pre = make_uint4(0u, 0u, 0u, 0u);
    if (r < 2 * nr && j0 + lane < e) pre = P[j0 + lane];
    while (r < 2 * nr) {
        const uint4 s = pre;
        const bool have = j0 + lane < e;
        next();
        if (r < 2 * nr && j0 + lane < e) pre = P[j0 + lane];
        const float dx = (float)(int32_t)(s.x - cc[0]), dy = (float)(int32_t)(s.y - cc[1]),
                    dz = (float)(int32_t)(s.z - cc[2]);
        const float gx = fmaxf(fmaxf(L[0] - dx, dx - H[0]), 0.f), gy = fmaxf(fmaxf(L[1] - dy, dy - H[1]), 0.f),
                    gz = fmaxf(fmaxf(L[2] - dz, dz - H[2]), 0.f);
        const bool keep = have && fmaf(gz, gz, fmaf(gy, gy, gx * gx)) < rc2t;
        const uint64_t m = __ballot(keep);
        const int below = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (keep) ring[(rb + fill + below) & (2 * NEAR_TILE - 1)] = s;
        fill += (int)__popcll(m);
        if (fill >= NEAR_TILE) {
            wave_sync();
            const uint4* T = ring + rb + stream;
#pragma unroll 2
            for (int j = 0; j < NEAR_TILE; j += 4 * G) {
                // four sources read together: the in-range branch inside
                // pair() would otherwise keep each read next to its use
                const uint4 u0 = T[j], u1 = T[j + G], u2 = T[j + 2 * G], u3 = T[j + 3 * G];
                pair(u0);
                pair(u1);
                pair(u2);
                pair(u3);
            }
            terms += NEAR_TILE / G;
            if (terms == 64) fold();
            rb ^= NEAR_TILE;
            fill -= NEAR_TILE;
            wave_sync();
        }
    }
    wave_sync();
    for (int j = stream; j < fill; j += G) pair(ring[rb + j]);
    fold();
    double a[4] = {(double)sx + (double)cx_, (double)sy + (double)cy_, (double)sz + (double)cz_,
                   (double)sp + (double)cp_};
#pragma unroll
    for (int m = S; m < 64; m <<= 1)
#pragma unroll
        for (int c = 0; c < 4; ++c) a[c] += __shfl_xor(a[c], m);
    if (lane < S && i < s1) {
        const uint32_t p = me.w;
        fx[p] += (float)(a[0] * fscale);
        fy[p] += (float)(a[1] * fscale);
        fz[p] += (float)(a[2] * fscale);
        pot[p] += (float)(a[3] * pscale - pconst);
    }
}

void free_near_buffers() {
    dev_free(g_near.P0);
    dev_free(g_near.P);
    dev_free(g_near.sort_tmp);
    g_near.sort_tmp = nullptr;
    g_near.sort_tmp_bytes = 0;
    dev_free(g_near.start);
    dev_free(g_near.row_chunk);
    dev_free(g_near.subst);
    g_near.subst = nullptr;
    dev_free(g_near.item);
    dev_free(g_near.table);
    g_near.table = nullptr;
    g_near.table_rsu = g_near.table_rcu = 0.0;
    g_near.P0 = g_near.P = nullptr;
    g_near.start = g_near.row_chunk = nullptr;
    g_near.item = nullptr;
    g_near.item_cap = 0;
    g_near.cap = 0;
    g_near.ncell_cap = g_near.nrow_cap = 0;
}

int ensure_buffers(size_t n, size_t ncell, size_t nrow) {
    if (n > g_near.cap) {
        dev_free(g_near.P0);
        dev_free(g_near.P);
        g_near.P0 = g_near.P = nullptr;
        g_near.cap = 0;
        CT2_TRY(dev_alloc((void**)&g_near.P0, n * sizeof(uint4), "near-field sort"));
        CT2_TRY(dev_alloc((void**)&g_near.P, n * sizeof(uint4), "near-field sorted particles"));
        g_near.cap = n;
    }
    if (ncell > g_near.ncell_cap || nrow > g_near.nrow_cap) {
        dev_free(g_near.start);
        dev_free(g_near.row_chunk);
        dev_free(g_near.subst);
        g_near.start = g_near.row_chunk = g_near.subst = nullptr;
        g_near.ncell_cap = g_near.nrow_cap = 0;
        CT2_TRY(dev_alloc((void**)&g_near.start, (ncell + 1) * sizeof(int), "near-field cell starts"));
        CT2_TRY(dev_alloc((void**)&g_near.row_chunk, (nrow + 1) * sizeof(int), "near-field work items"));
        CT2_TRY(dev_alloc((void**)&g_near.subst, (ncell * NEAR_SUB + 1) * sizeof(int), "near-field slice starts"));
        g_near.ncell_cap = ncell;
        g_near.nrow_cap = nrow;
    }
    const size_t items = n / NEAR_SINKS + 1 + nrow;
    if (items > g_near.item_cap) {
        dev_free(g_near.item);
        g_near.item = nullptr;
        g_near.item_cap = 0;
        CT2_TRY(dev_alloc((void**)&g_near.item, items * sizeof(int2), "near-field work items"));
        g_near.item_cap = items;
    }
    return CT2_OK;
}

}  // namespace

// Long-range (filtered) part of the pair kernel at t = u^2, u = r / (2 rs),
// without the 1/(2 rs)^3 and 1/(2 rs) factors:
//   K(t) = [erf(u) - (2u/sqrt(pi)) e^{-u^2}] / u^3,   P(t) = erf(u) / u,
// by their Taylor series in t below u = 0.05, where the closed forms cancel.
static double lr_K(double t) {
    const double c = 2.0 / std::sqrt(M_PI);
    if (t < 0.0025) return c * (2.0 / 3.0 + t * (-2.0 / 5.0 + t * (1.0 / 7.0 + t * (-1.0 / 27.0))));
    const double u = std::sqrt(t);
    return (std::erf(u) - c * u * std::exp(-t)) / (t * u);
}
static double lr_P(double t) {
    const double c = 2.0 / std::sqrt(M_PI);
    if (t < 0.0025) return c * (1.0 + t * (-1.0 / 3.0 + t * (1.0 / 10.0 + t * (-1.0 / 42.0))));
    const double u = std::sqrt(t);
    return std::erf(u) / u;
}

// nt cubic pieces of k_l = K(t)/(2 rs)^3 and p_l = P(t)/(2 rs) over r^2 in
// [0, rcut^2) (2^-32 position units); piece i is a polynomial in
// f = r^2 nt / rcut^2 - i in [0, 1), coefficients (c0, c1, c2, c3), computed in
// FP64 by interpolation at the four Chebyshev nodes of the piece.
void near_kernel_table(double rsu, double rcu, int nt, float* k4, float* p4) {
    constexpr int D = 4;
    double node[D], inv[D][D];
    for (int j = 0; j < D; ++j) node[j] = 0.5 - 0.5 * std::cos(M_PI * (j + 0.5) / D);
    // inverse of the Vandermonde matrix V[j][m] = node[j]^m (Gauss-Jordan)
    double a[D][2 * D];
    for (int j = 0; j < D; ++j)
        for (int m = 0; m < 2 * D; ++m) a[j][m] = m < D ? std::pow(node[j], m) : (m - D == j ? 1.0 : 0.0);
    for (int col = 0; col < D; ++col) {
        int piv = col;
        for (int r = col + 1; r < D; ++r)
            if (std::fabs(a[r][col]) > std::fabs(a[piv][col])) piv = r;
        for (int m = 0; m < 2 * D; ++m) std::swap(a[col][m], a[piv][m]);
        const double d = a[col][col];
        for (int m = 0; m < 2 * D; ++m) a[col][m] /= d;
        for (int r = 0; r < D; ++r)
            if (r != col) {
                const double f = a[r][col];
                for (int m = 0; m < 2 * D; ++m) a[r][m] -= f * a[col][m];
            }
    }
    for (int m = 0; m < D; ++m)
        for (int j = 0; j < D; ++j) inv[m][j] = a[m][D + j];
    const double s = 0.5 / rsu;  // 1 / (2 rs)
    const double tmax = rcu * rcu * s * s;  // u^2 at the cutoff
    for (int i = 0; i < nt; ++i) {
        double vk[D], vp[D];
        for (int j = 0; j < D; ++j) {
            const double t = (i + node[j]) * tmax / nt;
            vk[j] = lr_K(t) * s * s * s;
            vp[j] = lr_P(t) * s;
        }
        for (int m = 0; m < D; ++m) {
            double ck = 0.0, cp = 0.0;
            for (int j = 0; j < D; ++j) {
                ck += inv[m][j] * vk[j];
                cp += inv[m][j] * vp[j];
            }
            k4[4 * i + m] = (float)ck;
            p4[4 * i + m] = (float)cp;
        }
    }
}

// The table near_force reads: p_l = P(t)/(2 rs) over r^2 in [0, rcut^2]
// (2^-32 position units) in NEAR_NT + 1 cubic pieces, piece i in f = r^2
// NEAR_NT / rcut^2 - i over [-1/2, 1/2] (piece 0: [0, 1/2]).  Their derivative
// carries k_l = K(t)/(2 rs)^3, so it is k_l that is interpolated, by a quadratic
// at three Chebyshev nodes of the piece, and integrated:
// dp_l/df = -k_l rcut^2 / (2 NEAR_NT); the constant matches p_l at f = 0.
static void near_potential_table(double rsu, double rcu, float* out) {
    const double s = 0.5 / rsu, step = rcu * rcu / NEAR_NT;  // 1 / (2 rs); r^2 per piece
    for (int i = 0; i <= NEAR_NT; ++i) {
        const double f0 = i ? -0.5 : 0.0;
        double f[3], dd[3];  // nodes; divided differences of k_l
        for (int j = 0; j < 3; ++j) {
            f[j] = f0 + (0.5 - f0) * (0.5 - 0.5 * std::cos(M_PI * (j + 0.5) / 3));
            dd[j] = lr_K((i + f[j]) * step * s * s) * s * s * s;
        }
        for (int l = 1; l < 3; ++l)
            for (int j = 2; j >= l; --j) dd[j] = (dd[j] - dd[j - 1]) / (f[j] - f[j - l]);
        // Newton form to powers of f
        const double c[3] = {dd[0] - f[0] * (dd[1] - f[1] * dd[2]), dd[1] - (f[0] + f[1]) * dd[2], dd[2]};
        out[4 * i] = (float)(lr_P(i * step * s * s) * s);
        for (int m = 0; m < 3; ++m) out[4 * i + m + 1] = (float)(-0.5 * step * c[m] / (m + 1));
    }
}

bool near_enabled() { return g_near.rcut_rs > 0.0; }
double near_rcut_rs() { return g_near.rcut_rs; }

// Adds the near field to the stored PM force (rs in box units).
int near_forces(double rs) {
    Context& c = ctx();
    const double rcut = g_near.rcut_rs * rs;
    int nc = (int)std::floor(1.0 / (rcut * (1.0 + 1e-6)));
    nc = std::min(nc, NEAR_MAX_NC);
    if (nc < 3) return set_error(CT2_ERR_INVALID, "near-field cutoff %g exceeds a third of the box", rcut);
    const int n = (int)c.n;
    const int F = (double)n / ((double)nc * nc * nc) > NEAR_SPLIT_DENSITY ? 2 : 1;
    const int nxy = F * nc;
    const int c3 = nxy * nxy * nc, nrow = nxy * nxy;
    CT2_TRY(ensure_buffers(c.n, (size_t)c3, (size_t)nrow));
    g_near.nc = nc;
    hipStream_t st = c.stream;
    // sorted stably by slice: the order is (row, z slice, particle index)
    // whatever the scheduling
    const uint32_t nzs = (uint32_t)(nc * NEAR_SUB);
    const int nkeys = c3 * NEAR_SUB;  // = nrow nzs < 2^25
    int bits = 1;
    while ((1 << bits) < nkeys) ++bits;
    const SliceKey key{(uint32_t)nxy, nzs};
    CT2_TRY(cell_sort(c.x, c.y, c.z, n, key, bits, g_near.P, g_near.P0, &g_near.sort_tmp, &g_near.sort_tmp_bytes, st));
    CT2_TRY(cell_starts(g_near.P, key, n, nkeys, PutSlice{g_near.subst, g_near.start}, st));
    near_scan<<<1, SCAN_THREADS, 0, st>>>(g_near.start, nrow, nc, g_near.row_chunk);
    CT2_LAUNCH_CHECK();

    const double u = 0x1p32;
    const double rsu = rs * u, rcu = rcut * u, h = c.opts.hsoft, hu = h * u;
    NearConst q;
    q.rc2u = (float)(rcu * rcu);
    q.rcu = (float)rcu;
    q.eps2u = (float)(hu * hu);
    q.h2u = (float)(hu * hu);
    q.hinvu = (float)(1.0 / hu);
    q.hinv3u = (float)(1.0 / (hu * hu * hu));
    q.tscale = (float)(NEAR_NT / (rcu * rcu));
    q.kscale = 2.0f * q.tscale;
    constexpr size_t table_floats = 4 * (NEAR_NT + 1);
    if (!g_near.table) CT2_TRY(dev_alloc((void**)&g_near.table, table_floats * sizeof(float), "near-field table"));
    if (g_near.table_rsu != rsu || g_near.table_rcu != rcu) {
        float t[table_floats];
        near_potential_table(rsu, rcu, t);
        CT2_HIP(hipMemcpyAsync(g_near.table, t, sizeof t, hipMemcpyHostToDevice, st));
        CT2_HIP(hipStreamSynchronize(st));  // t is released on return
        g_near.table_rsu = rsu;
        g_near.table_rcu = rcu;
    }
    const double gm = c.opts.GM;
    const double fscale = gm * 0x1p64, pscale = gm * 0x1p32;
    const double pconst = gm * (double)n * 4.0 * M_PI * rs * rs;
    near_items<<<(nrow + 3) / 4, 256, 0, st>>>(g_near.row_chunk, nrow, g_near.item);
    CT2_LAUNCH_CHECK();
    // slices a partner within rcut can be away along z (rcut <= 1 / nc: R <= NEAR_SUB)
    const int R = std::min(NEAR_SUB, (int)std::ceil(rcut * nc * NEAR_SUB));
    // work items: at most one partial one per row beyond n / NEAR_SINKS full ones
    const unsigned items = (unsigned)(((long)n + NEAR_SINKS - 1) / NEAR_SINKS + nrow);
    // at most 2^31 threads along x: a launch takes less than 2^32, and 2^30 particles need more
    const unsigned blocks = (items + NEAR_WAVES - 1) / NEAR_WAVES, across = std::min(blocks, (1u << 31) / (64 * NEAR_WAVES));
    const dim3 grid(across, (blocks + across - 1) / across);
#define CT2_NEAR(KER)                                                                                          \
    near_force<KER><<<grid, 64 * NEAR_WAVES, 0, st>>>(                                                         \
        g_near.P, g_near.start, g_near.subst, g_near.row_chunk, g_near.item, nxy, nc, F, R, q, g_near.table,   \
        fscale, pscale, pconst, c.fx, c.fy, c.fz, c.pot)
    if (c.opts.kernel == CT2_KERNEL_PLUMMER)
        CT2_NEAR(CT2_KERNEL_PLUMMER);
    else
        CT2_NEAR(CT2_KERNEL_CT2);
#undef CT2_NEAR
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

int near_set(double rcut_rs) {
    if (!(rcut_rs >= 0.0) || rcut_rs > 64.0) return set_error(CT2_ERR_INVALID, "bad near-field cutoff %g", rcut_rs);
    g_near.rcut_rs = rcut_rs;
    return CT2_OK;
}

int near_cells() { return g_near.nc; }

void release_near() {
    free_near_buffers();
    g_near.rcut_rs = 0.0;
    g_near.nc = 0;
}

}  // namespace ct2

static_assert(CT2_NEAR_PIECES == ct2::NEAR_NT + 1, "the pieces of near_force");

extern "C" int ct2_near_potential_table(double rs_u, double rcut_u, float* p4) {
    if (!(rs_u > 0.0) || !(rcut_u > 0.0) || !p4)
        return ct2::set_error(CT2_ERR_INVALID, "ct2_near_potential_table: bad argument");
    ct2::near_potential_table(rs_u, rcut_u, p4);
    return CT2_OK;
}

extern "C" int ct2_near_kernel_table(double rs_u, double rcut_u, int nt, float* k4, float* p4) {
    if (!(rs_u > 0.0) || !(rcut_u > 0.0) || nt < 1 || !k4 || !p4)
        return ct2::set_error(CT2_ERR_INVALID, "ct2_near_kernel_table: bad argument");
    ct2::near_kernel_table(rs_u, rcut_u, nt, k4, p4);
    return CT2_OK;
}
