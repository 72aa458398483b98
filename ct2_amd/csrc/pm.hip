// pm.hip -- the particle-mesh force on gfx950.
//
// Replaces the reference's multipole-mesh far field (particle_compute_multipoles
// and particle_compute_expansions, particle.cpp:180-271, evaluated by L2P at
// kick.cpp:29) with cloud-in-cell mass assignment, keeping its pipeline:
//   deposit       fixed-point CIC (default) or TSC weights, uint64 atomics:
//                 deterministic, bit-identical to the CPU oracle.  Where
//                 tiles_pay says so: particles binned by 16^3-node tile
//                 (bin_*), each tile summed in LDS and stored (dep_tile);
//                 elsewhere one global atomic per particle and stencil
//                 node (mesh_deposit)
//   rfft_zy_density  z and y passes of the density's FP32 transform to its
//                 half spectrum (fft.hip; the first reads the uint64 grid
//                 directly)
//   pm_xpass      the x pass, rho_hat * G (FP64 Green's table, octant-
//                 symmetric), the spectral gradient, and the inverse x passes;
//                 two real fields share one complex grid: A = Fx + i Fy,
//                 B = Fz + i pot
//   fft_inverse_yz  the inverse y and z passes of A and B
//   interp        force and potential at the particles (same weights): in
//                 deposit-tile order from LDS-staged tiles (interp_tile)
//                 when tiles hold enough particles, else per particle
//                 (mesh_interp)
// Grid layout: (i*ng + j)*ng + k with i along x; node c at position c/ng.
#include <algorithm>
#include <cmath>
#include <vector>

#include "epilogue.h"
#include "fft_stages.h"
#include "internal.h"
#include "wave.h"

namespace ct2 {
namespace {

constexpr int CIC_BITS = 21;  // weight resolution per axis
constexpr int PM_BLOCK = 256;

struct PmState {
    int ng = 0, g = 0;
    double rs_cells = 0.0;
    int order_table = 0;              // assignment order the table was built for
    float gm_table = 0.0f;  // GM the table was built for
    unsigned long long* W = nullptr;  // density, 2^-32 particle units
    float2* half = nullptr;           // the density's half spectrum
    float2* A = nullptr;              // Fx + i Fy, and right after it
    float2* B = nullptr;              // Fz + i pot
    double* G = nullptr;              // Green's table on the octant, (ng/2+1)^3
    // tiled deposit: particles binned by tile of 16^3 nodes
    int ntile = 0;
    int* tcount = nullptr;  // [ntile]
    int* tstart = nullptr;  // [ntile + 1]
    int* bins = nullptr;    // [BIN_WGS][ntile] counts per binning workgroup
    size_t cap = 0;         // particles order has room for (of one slab)
    int* order = nullptr;   // [cap MAX_COPIES] particle indices grouped by tile, ~index where at home in another
} g_pm;
int g_assign = 1;  // mass assignment: 1 CIC, 2 TSC (kept across ct2_pm_init)

// Per-axis weights, 21-bit fixed point summing to 2^21, and the first node:
//   ORDER 1 (CIC): nodes lo, lo+1 with lo = x >> s, a1 = fraction >> (s-21);
//   ORDER 2 (TSC): nearest node c = (x + 2^(s-1)) >> s, signed offset D in
//     [-2^20, 2^20) (2^-21 cells); nodes c-1, c, c+1 get round((2^20-D)^2/2^22),
//     the rest, round((2^20+D)^2/2^22): the quadratic spline (1/2)(1/2 -+ d)^2.
// Everything but the squares fits in 32 bits.
template <int ORDER>
__device__ __forceinline__ void assign_axis(uint32_t x, int s, uint32_t& lo, uint32_t (&w)[ORDER + 1]) {
    if constexpr (ORDER == 1) {
        lo = x >> s;
        const uint32_t t = x & ((1u << s) - 1u);
        w[1] = t >> (s - CIC_BITS);
        w[0] = (1u << CIC_BITS) - w[1];
    } else {
        const uint32_t half = 1u << (s - 1);
        const uint32_t xs = x + half;
        const int32_t d = (int32_t)(xs & ((1u << s) - 1u)) - (int32_t)half;
        const int32_t D = d >> (s - CIC_BITS);
        const uint32_t a = (uint32_t)((1 << 20) - D), b = (uint32_t)((1 << 20) + D);
        w[0] = (uint32_t)(((uint64_t)a * a + (1ull << 21)) >> 22);
        w[2] = (uint32_t)(((uint64_t)b * b + (1ull << 21)) >> 22);
        w[1] = (1u << CIC_BITS) - w[0] - w[2];
        lo = (xs >> s) - 1u;
    }
}

__global__ __launch_bounds__(PM_BLOCK) void fill_u64(unsigned long long* __restrict__ p, long n) {
    const long i = (long)blockIdx.x * PM_BLOCK + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

template <int ORDER>
__global__ __launch_bounds__(PM_BLOCK) void mesh_deposit(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                        const uint32_t* __restrict__ Z, int n, int g,
                                                        unsigned long long* __restrict__ W) {
    const int p = blockIdx.x * PM_BLOCK + threadIdx.x;
    if (p >= n) return;
    const int s = 32 - g;
    const uint32_t ng = 1u << g, mask = ng - 1;
    uint32_t i0, j0, k0;
    uint32_t ax[ORDER + 1], ay[ORDER + 1], az[ORDER + 1];
    assign_axis<ORDER>(X[p], s, i0, ax);
    assign_axis<ORDER>(Y[p], s, j0, ay);
    assign_axis<ORDER>(Z[p], s, k0, az);
#pragma unroll
    for (int dx = 0; dx <= ORDER; ++dx)
#pragma unroll
        for (int dy = 0; dy <= ORDER; ++dy) {
            const uint64_t axy = (uint64_t)ax[dx] * ay[dy];
            const size_t row = ((size_t)((i0 + dx) & mask) * ng + ((j0 + dy) & mask)) * ng;
#pragma unroll
            for (int dz = 0; dz <= ORDER; ++dz)
                atomicAdd(W + row + ((k0 + dz) & mask), (unsigned long long)((axy * az[dz]) >> 31));
        }
}

// Tiled deposit for grids of 32 nodes and more a side.  The grid is cut into
// tiles of 16^3 nodes; a particle's home is the tile of its anchor node (CIC:
// its first node; TSC: its nearest node), and where its stencil reaches over a
// face of that tile it is listed in the neighbours there too (1.4 entries per
// particle with TSC, 1.2 with CIC).  One workgroup per tile (dep_tile) adds the
// weights that fall on the tile's own nodes in LDS (uint64 LDS atomics) and
// stores them, each node once.  No global atomics: on this chip they leave the
// XCD's L2.  Adding the LDS copies of grown tiles into a cleared grid with them
// took 186 us for 2^21 particles on 256^3 (TSC), and a binning that counted with
// them 54; tiles and binning take 43 and 48 this way.  Setting the nodes around
// each tile aside for a second pass over the faces, instead of listing particles
// twice: 127 and 46 (the z faces touch every line of the grid again).  The
// weights are those of mesh_deposit and integer sums do not depend on order, so
// the grid is bit-identical to mesh_deposit's.
constexpr int TILE_B = 4;  // log2 of the tile's side
constexpr int TS = 1 << TILE_B;
constexpr int TROW = TS + 1;                 // padded LDS row
constexpr int TL = TS + 2;                   // side of the grown tile
constexpr int TL_NODES = TL * TL * TL;
// Threads to a tile: 1,024 on grids of at most two tiles per CU, 512 (four workgroups
// per CU) on larger ones.  us of deposit and interpolation of 2^21 particles on 256^3
// (TSC) 169 with 512, 176 with 1,024; a force on 128^3 188 / 196 with 1,024 / 512, and
// where the set lies in a corner, a few tiles' work, 9.8 / 16.7 ms (in 1/1000 of the box).
constexpr int tile_threads(int tiles) { return tiles <= 2 * 256 ? 1024 : 512; }
constexpr int TILE_MIN_G = TILE_B + 1;  // grids of at least 2^5 nodes a side
constexpr int BIN_THREADS = 1024;
constexpr int BIN_WGS = 128;            // binning workgroups at most
constexpr int BIN_TILES = 32768;        // tiles whose counters fit in LDS (512^3 grids)
constexpr int MAX_COPIES = 8;           // tiles a stencil can touch
// Entries are counted in int, and none can be refused: a list holds MAX_COPIES for
// each of its particles.  Containers of more particles than this go slab by slab,
// each adding its density to the last one's; the lists then take 8.6 GB.
constexpr long SLAB_MAX = (1L << 31) / MAX_COPIES - 1;

template <int ORDER>
__device__ __forceinline__ uint32_t anchor_node(uint32_t x, int s) {
    return ORDER == 1 ? x >> s : (uint32_t)(x + (1u << (s - 1))) >> s;
}

// f(tile, home) for every tile the particle's stencil touches, its home first.
template <int ORDER, typename F>
__device__ __forceinline__ void for_tiles(uint32_t x, uint32_t y, uint32_t z, int g, const F& f) {
    const int s = 32 - g, gt = g - TILE_B, m = (1 << gt) - 1;
    int t[3][2];
    bool two[3];
    const uint32_t v[3] = {x, y, z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int n = (int)anchor_node<ORDER>(v[a], s), o = n & (TS - 1);
        const bool up = o == TS - 1, down = ORDER == 2 && o == 0;
        t[a][0] = n >> TILE_B;
        t[a][1] = (t[a][0] + (up ? 1 : m)) & m;
        two[a] = up || down;
    }
    f((((t[0][0] << gt) + t[1][0]) << gt) + t[2][0], true);
    if (!(two[0] || two[1] || two[2])) return;
#pragma unroll
    for (int d = 1; d < 8; ++d) {
        const bool ux = d & 1, uy = d & 2, uz = d & 4;
        if ((ux && !two[0]) || (uy && !two[1]) || (uz && !two[2])) continue;
        f((((t[0][ux] << gt) + t[1][uy]) << gt) + t[2][uz], false);
    }
}

// The first node of a tile along each axis.
__device__ __forceinline__ void tile_origin(int tile, int g, uint32_t& ox, uint32_t& oy, uint32_t& oz) {
    const int gt = g - TILE_B, m = (1 << gt) - 1;
    ox = (uint32_t)(tile >> (2 * gt)) << TILE_B;
    oy = (uint32_t)((tile >> gt) & m) << TILE_B;
    oz = (uint32_t)(tile & m) << TILE_B;
}

// Binning, first half: the entries of workgroup w's particles [w per,
// (w + 1) per) counted by tile in LDS, cnt[w][tile].
template <int ORDER, int TILES>
__global__ __launch_bounds__(BIN_THREADS) void bin_count(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                        const uint32_t* __restrict__ Z, int n, int per, int g, int nt,
                                                        int* __restrict__ cnt) {
    __shared__ int h[TILES];
    for (int t = threadIdx.x; t < nt; t += BIN_THREADS) h[t] = 0;
    __syncthreads();
    const int p1 = (int)min((long)n, (long)(blockIdx.x + 1) * per);
    for (int p = blockIdx.x * per + threadIdx.x; p < p1; p += BIN_THREADS)
        for_tiles<ORDER>(X[p], Y[p], Z[p], g, [&](int t, bool) { atomicAdd(&h[t], 1); });
    __syncthreads();
    for (int t = threadIdx.x; t < nt; t += BIN_THREADS) cnt[(size_t)blockIdx.x * nt + t] = h[t];
}

// cnt[w][tile] -> the tile's entries from the workgroups before w, and the
// tile's total.
__global__ __launch_bounds__(PM_BLOCK) void bin_prefix(int* __restrict__ cnt, int nw, int nt, int* __restrict__ total) {
    const int t = blockIdx.x * PM_BLOCK + threadIdx.x;
    if (t >= nt) return;
    int run = 0;
    constexpr int AHEAD = 16;  // counts read together: the stores would otherwise hold back the next loads
    for (int w0 = 0; w0 < nw; w0 += AHEAD) {
        int v[AHEAD];
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = w0 + u < nw ? cnt[(size_t)(w0 + u) * nt + t] : 0;
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            if (w0 + u < nw) cnt[(size_t)(w0 + u) * nt + t] = run;
            run += v[u];
        }
    }
    total[t] = run;
}

// Exclusive scan of nt values by one workgroup of BIN_THREADS: out(t, prefix)
// for every t, in thread-contiguous pieces; returns the total.
template <typename IN, typename OUT>
__device__ __forceinline__ int block_scan(int nt, const IN& in, const OUT& out) {
    __shared__ int part[BIN_THREADS / 64];
    const int t = threadIdx.x, lane = t & 63;
    const int per = (nt + BIN_THREADS - 1) / BIN_THREADS;
    const int b = min(nt, t * per), e = min(nt, b + per);
    int sum = 0;
    for (int i = b; i < e; ++i) sum += in(i);
    int s = sum;  // inclusive over the wave
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(s, off);
        if (lane >= off) s += u;
    }
    if (lane == 63) part[t >> 6] = s;
    __syncthreads();
    int run = s - sum, total = 0;
    for (int k = 0; k < BIN_THREADS / 64; ++k) {
        if (k < t >> 6) run += part[k];
        total += part[k];
    }
    for (int i = b; i < e; ++i) {
        const int v = in(i);
        out(i, run);
        run += v;
    }
    return total;
}

// Binning, second half: every workgroup scans the tile totals (workgroup 0
// writes them out as tstart) and places its particles' entries, grouped by
// tile, in order.  total null: no bin_prefix has run, and every workgroup sums
// the counts as they are (bin_in_lds).  Which of a tile's slots an entry gets depends on scheduling;
// the set does not.
template <int ORDER, int TILES>
__global__ __launch_bounds__(BIN_THREADS) void bin_scatter(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                          const uint32_t* __restrict__ Z, int n, int per, int g, int nt,
                                                          const int* __restrict__ cnt, const int* __restrict__ total,
                                                          int* __restrict__ tstart, int* __restrict__ order) {
    __shared__ int h[TILES];
    const bool first = blockIdx.x == 0;
    int sum;
    if (total) {
        const int* mine = cnt + (size_t)blockIdx.x * nt;
        sum = block_scan(nt, [&](int t) { return total[t]; },
                         [&](int t, int s) {
                             h[t] = s + mine[t];
                             if (first) tstart[t] = s;
                         });
    } else {  // at most one tile a thread
        int before = 0, all = 0;
        const int t = threadIdx.x, nw = gridDim.x;
        if (t < nt)
#pragma unroll 8
            for (int w = 0; w < nw; ++w) {
                const int v = cnt[(size_t)w * nt + t];
                before += w < (int)blockIdx.x ? v : 0;
                all += v;
            }
        sum = block_scan(nt, [&](int) { return all; },
                         [&](int k, int s) {
                             h[k] = s + before;
                             if (first) tstart[k] = s;
                         });
    }
    if (first && threadIdx.x == 0) tstart[nt] = sum;
    __syncthreads();
    const int p1 = (int)min((long)n, (long)(blockIdx.x + 1) * per);
    for (int p = blockIdx.x * per + threadIdx.x; p < p1; p += BIN_THREADS)
        for_tiles<ORDER>(X[p], Y[p], Z[p], g, [&](int t, bool home) { order[atomicAdd(&h[t], 1)] = home ? p : ~p; });
}

// The same for grids of more tiles than LDS holds counters for, with global
// atomics: one per run of particles of one home tile, one per further entry.
__global__ __launch_bounds__(PM_BLOCK) void fill_i32(int* __restrict__ p, int n) {
    const int i = blockIdx.x * PM_BLOCK + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <int ORDER, bool PLACE>
__global__ __launch_bounds__(PM_BLOCK) void bin_global(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                       const uint32_t* __restrict__ Z, int n, int g,
                                                       int* __restrict__ counter, int* __restrict__ order) {
    const int p = blockIdx.x * PM_BLOCK + threadIdx.x;
    int home = -1;
    if (p < n)
        for_tiles<ORDER>(X[p], Y[p], Z[p], g, [&](int t, bool h) {
            if (h) {
                home = t;
            } else {
                const int k = atomicAdd(counter + t, 1);
                if (PLACE) order[k] = ~p;
            }
        });
    const int k = run_increment(counter, home);  // every lane of the wave takes part
    if (PLACE && p < n) order[k] = p;
}

// Exclusive scan into out[0 .. len] and, as cursors for the placement, over in.
__global__ __launch_bounds__(BIN_THREADS) void tile_scan(int* __restrict__ in, int len, int* __restrict__ out) {
    const int sum = block_scan(len, [&](int t) { return in[t]; }, [&](int t, int s) { out[t] = in[t] = s; });
    if (threadIdx.x == 0) out[len] = sum;
}

template <int ORDER, int THREADS>
__global__ __launch_bounds__(THREADS) void dep_tile(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                        const uint32_t* __restrict__ Z, const int* __restrict__ order,
                                                        const int* __restrict__ tstart, int g, bool add,
                                                        unsigned long long* __restrict__ W) {
    __shared__ unsigned long long acc[TS * TS * TROW];
    const int tile = (int)xcd_contiguous(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int b = tstart[tile], e = tstart[tile + 1];
    const int s = 32 - g;
    const uint32_t mask = (1u << g) - 1u;
    uint32_t ox, oy, oz;
    tile_origin(tile, g, ox, oy, oz);
    for (int i = tid; i < TS * TS * TROW; i += THREADS) acc[i] = 0ull;
    __syncthreads();
    for (int k = b + tid; k < e; k += THREADS) {
        const int o = order[k], p = o < 0 ? ~o : o;
        const uint32_t x = X[p], y = Y[p], z = Z[p];
        uint32_t lo;
        uint32_t ax[ORDER + 1], ay[ORDER + 1], az[ORDER + 1];
        assign_axis<ORDER>(x, s, lo, ax);
        assign_axis<ORDER>(y, s, lo, ay);
        assign_axis<ORDER>(z, s, lo, az);
        // the stencil's first node from the tile's first, -2 .. TS
        constexpr int SHIFT = ORDER == 1 ? 1 : 2;
        const int lx = (int)((anchor_node<ORDER>(x, s) - ox + 1u) & mask) - SHIFT;
        const int ly = (int)((anchor_node<ORDER>(y, s) - oy + 1u) & mask) - SHIFT;
        const int lz = (int)((anchor_node<ORDER>(z, s) - oz + 1u) & mask) - SHIFT;
#pragma unroll
        for (int dx = 0; dx <= ORDER; ++dx)
#pragma unroll
            for (int dy = 0; dy <= ORDER; ++dy) {
                if ((unsigned)(lx + dx) >= TS || (unsigned)(ly + dy) >= TS) continue;
                const uint64_t axy = (uint64_t)ax[dx] * ay[dy];
                unsigned long long* row = acc + ((lx + dx) * TS + (ly + dy)) * TROW + lz;
#pragma unroll
                for (int dz = 0; dz <= ORDER; ++dz)
                    if ((unsigned)(lz + dz) < TS) atomicAdd(row + dz, (unsigned long long)((axy * az[dz]) >> 31));
            }
    }
    __syncthreads();
    for (int i = tid; i < TS * TS * TS; i += THREADS) {
        const int lz = i % TS, ly = i / TS % TS, lx = i / (TS * TS);
        unsigned long long* const w = W + (((((size_t)(ox + lx) << g) + (oy + ly)) << g) + (oz + lz));
        const unsigned long long v = acc[(lx * TS + ly) * TROW + lz];
        *w = add ? *w + v : v;
    }
}

// The x pass of the force transforms, forward and inverse in one kernel.  A
// workgroup takes COLS columns (ky, kz <= N/2) of the half spectrum (after its
// z and y passes), transforms them along x, keeps phi_hat = G rho_hat (FP64) in
// registers (a lane's outputs of a transform are its inputs of the next), and
// from it transforms back the columns of
//   A = F_hat_x + i F_hat_y,  B = F_hat_z + i pot_hat,
// F_hat = -i k phi_hat with the Nyquist components of k zeroed, pot_hat =
// -phi_hat, at (ky, kz) and, for 0 < kz < N/2, at (-ky, -kz), where rho_hat is
// the conjugate; there element i holds -kx, so the forward sign inverts it.
// Bound by HBM: 4 B of half spectrum and 4 of table in, 16 out per cell: 109 us
// on a 256^3 grid, 3.7 TB/s.  The forward x pass of the whole spectrum, the
// product and the two inverse x passes as kernels of their own moved 72 B per
// cell in 205 us; with the half-spectrum z and y passes before it the
// transforms of one force on 256^3 went from 453 to 327 us, on 64^3 from 36 to
// 22 us (ten launches to four).
// 16 columns to a workgroup, a 128-byte line's, where there are so many: fewer do not
// pay for more workgroups nor more columns for fuller ones (us with 32 / 16 / 8 / 4
// columns: 64^3 7.7 / 7.0 / 7.4 / 7.5; 32^3 - / 5.1 / 5.7 / 5.8; 16^3, 8 at most, 3.7 /
// 3.9; 128^3 - / 15.3 / 14.7 / 16.3; runs of one differ by 4 %).
template <int N>
constexpr int xpass_cols() {
    return Cfg<float, N, N / 2>::COLS < 16 ? Cfg<float, N, N / 2>::COLS : 16;
}

template <int N>
__global__ __launch_bounds__((Cfg<float, N, N / 2>::P * xpass_cols<N>())) void pm_xpass(
    const float2* __restrict__ half, float2* __restrict__ A, const double* __restrict__ G,
    const float2* __restrict__ twg) {
    constexpr int H = N / 2;
    using CF = Cfg<float, N, H>;
    constexpr int COLS = xpass_cols<N>();
    constexpr unsigned MAIN = (unsigned)N * (H / COLS);
    constexpr double twopi = 6.283185307179586476925;
    __shared__ float2 sm[N * COLS];
    __shared__ float2 tw[N];
    load_twiddles<N>(tw, twg, CF::P * COLS);
    const int c = threadIdx.x % COLS, p = threadIdx.x / COLS;
    int ky, kz;
    const float2* d;
    long stride;
    if (blockIdx.x < MAIN) {
        const unsigned b = xcd_contiguous(blockIdx.x, MAIN);
        ky = b / (H / COLS);
        kz = b % (H / COLS) * COLS + c;
        d = half + (long)ky * H + kz;
        stride = (long)N * H;
    } else {  // kz = N/2: nyq[ky][x]
        ky = (blockIdx.x - MAIN) * COLS + c;
        kz = H;
        d = half + (long)N * N * H + (long)ky * N;
        stride = 1;
    }
    const int my = ky < H ? ky : ky - N;
    auto ix = [&](int i) { return i * COLS + c; };
    auto wave_x = [](int i) { return i == H ? 0.0 : twopi * (i < H ? i : i - N); };
    const double wy = ky == H ? 0.0 : twopi * my, wz = kz == H ? 0.0 : twopi * kz;
    double2 phi[CF::RM];
    const double* Gc = G + (long)abs(my) * (H + 1) + kz;
    double g[CF::RM];  // read ahead of the transform they wait for
#pragma unroll
    for (int m = 0; m < CF::RM; ++m) {
        const int i = p + m * CF::P;
        g[m] = Gc[(long)(i < H ? i : N - i) * (H + 1) * (H + 1)];
    }
    run_stages<float, N, 1, false, false>(
        [&](int i, int) { return d[(long)i * stride]; },
        [&](int i, int m, float2 v) {
            phi[m] = double2{g[m] * (double)v.x, g[m] * (double)v.y};
        },
        ix, sm, tw, p);
    constexpr long N2 = (long)N * N, N3 = N2 * N;
    float2* out = A + (long)ky * N + kz;
    __syncthreads();
    run_stages<float, N, -1, false, false>(
        [&](int i, int m) {
            const double kx = wave_x(i);
            return float2{(float)(kx * phi[m].y + wy * phi[m].x), (float)(-kx * phi[m].x + wy * phi[m].y)};
        },
        [&](int i, int, float2 v) { out[i * N2] = v; }, ix, sm, tw, p);
    __syncthreads();
    run_stages<float, N, -1, false, false>(
        [&](int, int m) { return float2{(float)((wz + 1.0) * phi[m].y), (float)(-(wz + 1.0) * phi[m].x)}; },
        [&](int i, int, float2 v) { out[N3 + i * N2] = v; }, ix, sm, tw, p);
    if (blockIdx.x >= MAIN) return;  // uniform: the kz = N/2 plane is its own mirror
    const bool mirror = kz > 0;      // and so is kz = 0
    out = A + (long)((N - ky) % N) * N + (N - kz);
    __syncthreads();
    run_stages<float, N, 1, false, false>(
        [&](int i, int m) {
            const double kx = wave_x(i);
            return float2{(float)(kx * phi[m].y - wy * phi[m].x), (float)(kx * phi[m].x + wy * phi[m].y)};
        },
        [&](int i, int, float2 v) {
            if (mirror) out[i * N2] = v;
        },
        ix, sm, tw, p);
    __syncthreads();
    run_stages<float, N, 1, false, false>(
        [&](int, int m) { return float2{(float)((wz - 1.0) * phi[m].y), (float)((wz - 1.0) * phi[m].x)}; },
        [&](int i, int, float2 v) {
            if (mirror) out[N3 + i * N2] = v;
        },
        ix, sm, tw, p);
}

template <int N>
int xpass_launch(const float2* half, float2* A, const double* G, hipStream_t st) {
    using CF = Cfg<float, N, N / 2>;
    const float2* tw = nullptr;
    CT2_TRY(fft_table_f32(N, &tw));
    constexpr int COLS = xpass_cols<N>();
    pm_xpass<N><<<N * (N / 2) / COLS + N / COLS, CF::P * COLS, 0, st>>>(half, A, G, tw);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

int xpass(int n, const float2* half, float2* A, const double* G, hipStream_t st) {
    switch (n) {
        case 8: return xpass_launch<8>(half, A, G, st);
        case 16: return xpass_launch<16>(half, A, G, st);
        case 32: return xpass_launch<32>(half, A, G, st);
        case 64: return xpass_launch<64>(half, A, G, st);
        case 128: return xpass_launch<128>(half, A, G, st);
        case 256: return xpass_launch<256>(half, A, G, st);
        case 512: return xpass_launch<512>(half, A, G, st);
        case 1024: return xpass_launch<1024>(half, A, G, st);
        default: return set_error(CT2_ERR_INVALID, "unsupported PM grid %d", n);
    }
}

// EPI: a kick of nothing but this force goes on to its epilogue, a launch and 13
// bytes read again per particle fewer.
template <int ORDER, bool EPI>
__global__ __launch_bounds__(PM_BLOCK) void mesh_interp(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                       const uint32_t* __restrict__ Z, int n, int g,
                                                       const float2* __restrict__ A, const float2* __restrict__ B,
                                                       float* __restrict__ fx, float* __restrict__ fy,
                                                       float* __restrict__ fz, float* __restrict__ pot, Sinks epi) {
    const int t = blockIdx.x * PM_BLOCK + threadIdx.x;
    const int p = min(t, n - 1);
    const int s = 32 - g;
    const uint32_t ng = 1u << g, mask = ng - 1;
    uint32_t i0, j0, k0;
    uint32_t ax[ORDER + 1], ay[ORDER + 1], az[ORDER + 1];
    assign_axis<ORDER>(X[p], s, i0, ax);
    assign_axis<ORDER>(Y[p], s, j0, ay);
    assign_axis<ORDER>(Z[p], s, k0, az);
    const float q = 0x1p-21f;
    float acc0 = 0.f, acc1 = 0.f, acc2 = 0.f, acc3 = 0.f;
#pragma unroll
    for (int dx = 0; dx <= ORDER; ++dx)
#pragma unroll
        for (int dy = 0; dy <= ORDER; ++dy) {
            const float wxy = ((float)ax[dx] * q) * ((float)ay[dy] * q);
            const size_t row = ((size_t)((i0 + dx) & mask) * ng + ((j0 + dy) & mask)) * ng;
#pragma unroll
            for (int dz = 0; dz <= ORDER; ++dz) {
                const size_t cc = row + ((k0 + dz) & mask);
                const float w = wxy * ((float)az[dz] * q);
                const float2 a = A[cc], b = B[cc];
                acc0 = fmaf(w, a.x, acc0);
                acc1 = fmaf(w, a.y, acc1);
                acc2 = fmaf(w, b.x, acc2);
                acc3 = fmaf(w, b.y, acc3);
            }
        }
    if (t < n) {
        fx[p] = acc0;
        fy[p] = acc1;
        fz[p] = acc2;
        pot[p] = acc3;
    }
    if constexpr (EPI) {
        int rmax = 0;
        if (t < n && t >= epi.first) epi.apply(t, acc0, acc1, acc2, rmax);
        epi.store_max(rmax);
    }
}

// Interpolation in tile order, for grids with enough particles per tile: a
// workgroup per deposit tile and grid (blockIdx.y: A = (Fx, Fy), B = (Fz, pot))
// stages the grown tile's 18^3 nodes in LDS (47 KB) and
// interpolates the particles at home in it.  The same weights and summation
// order as mesh_interp, so the results are identical.  Bound by the reads of the
// grown tiles (rows of 144 bytes, 2.1 lines each): 130 us for 2^21 particles on
// 256^3 with neighbouring tiles on one XCD, 165 with the tiles dealt to the XCDs
// in turn.
template <int ORDER, int THREADS>
__global__ __launch_bounds__(THREADS) void interp_tile(const uint32_t* __restrict__ X, const uint32_t* __restrict__ Y,
                                                           const uint32_t* __restrict__ Z, const int* __restrict__ order,
                                                           const int* __restrict__ tstart, int g,
                                                           const float2* __restrict__ A, float* __restrict__ fx,
                                                           float* __restrict__ fy, float* __restrict__ fz,
                                                           float* __restrict__ pot) {
    __shared__ float2 nd[TL_NODES];
    const int tile = (int)xcd_contiguous(blockIdx.x, gridDim.x);
    const int b = tstart[tile], e = tstart[tile + 1];
    if (b == e) return;  // uniform across the workgroup
    const int tid = threadIdx.x;
    const int s = 32 - g;
    const uint32_t mask = (1u << g) - 1u;
    uint32_t ox, oy, oz;
    tile_origin(tile, g, ox, oy, oz);
    A += (size_t)blockIdx.y << (3 * g);
    float* out0 = blockIdx.y ? fz : fx;
    float* out1 = blockIdx.y ? pot : fy;
    constexpr int LOADS = (TL_NODES + THREADS - 1) / THREADS;
    float2 v[LOADS];  // all in flight before the first is stored
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
        const int i = min(tid + u * THREADS, TL_NODES - 1);
        const int lx = i / (TL * TL), ly = i / TL % TL, lz = i % TL;
        const size_t gx = (ox + lx - 1u) & mask, gy = (oy + ly - 1u) & mask, gz = (oz + lz - 1u) & mask;
        v[u] = A[(((gx << g) + gy) << g) + gz];
    }
#pragma unroll
    for (int u = 0; u < LOADS; ++u)
        if (tid + u * THREADS < TL_NODES) nd[tid + u * THREADS] = v[u];
    __syncthreads();
    constexpr uint32_t SHIFT = ORDER == 1 ? 1u : 0u;
    const float q = 0x1p-21f;
    for (int k = b + tid; k < e; k += THREADS) {
        const int p = order[k];
        if (p < 0) continue;  // at home in a neighbour
        const uint32_t x = X[p], y = Y[p], z = Z[p];
        uint32_t lo;
        uint32_t ax[ORDER + 1], ay[ORDER + 1], az[ORDER + 1];
        assign_axis<ORDER>(x, s, lo, ax);
        assign_axis<ORDER>(y, s, lo, ay);
        assign_axis<ORDER>(z, s, lo, az);
        const uint32_t hx = anchor_node<ORDER>(x, s) - ox, hy = anchor_node<ORDER>(y, s) - oy,
                       hz = anchor_node<ORDER>(z, s) - oz;
        const int lx = (int)(hx + SHIFT), ly = (int)(hy + SHIFT), lz = (int)(hz + SHIFT);
        float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
        for (int dx = 0; dx <= ORDER; ++dx)
#pragma unroll
            for (int dy = 0; dy <= ORDER; ++dy) {
                const float wxy = ((float)ax[dx] * q) * ((float)ay[dy] * q);
                const float2* row = nd + ((lx + dx) * TL + (ly + dy)) * TL + lz;
#pragma unroll
                for (int dz = 0; dz <= ORDER; ++dz) {
                    const float w = wxy * ((float)az[dz] * q);
                    const float2 v = row[dz];
                    acc0 = fmaf(w, v.x, acc0);
                    acc1 = fmaf(w, v.y, acc1);
                }
            }
        out0[p] = acc0;
        out1[p] = acc1;
    }
}

void free_pm() {
    dev_free(g_pm.W);
    dev_free(g_pm.half);
    dev_free(g_pm.A);
    dev_free(g_pm.G);
    dev_free(g_pm.tcount);
    dev_free(g_pm.tstart);
    dev_free(g_pm.bins);
    dev_free(g_pm.order);
    g_pm = PmState{};
}

// The tile lists' entries, grown to what n particles can need.
int ensure_deposit(size_t n) {
    if (n <= g_pm.cap) return CT2_OK;
    dev_free(g_pm.order);
    g_pm.order = nullptr;
    g_pm.cap = 0;
    CT2_TRY(dev_alloc((void**)&g_pm.order, n * MAX_COPIES * sizeof(int), "PM deposit order"));
    g_pm.cap = n;
    return CT2_OK;
}

// Slab k of count: the container's particles [k per, (k + 1) per), per = ceil(n / count).
struct Slab {
    const uint32_t *x, *y, *z;
    long first;
    int n;
};
int slab_count(const Context& c) { return (int)(((long)c.n + SLAB_MAX - 1) / SLAB_MAX); }
Slab slab(const Context& c, int k) {
    const long count = slab_count(c), per = ((long)c.n + count - 1) / count, p0 = k * per;
    return {c.x + p0, c.y + p0, c.z + p0, p0, (int)std::min(per, (long)c.n - p0)};
}

// A slab's particles grouped by tile: g_pm.tstart, g_pm.order (indices in the slab).
template <int ORDER, int TILES>
int bin_in_lds(const Slab& p, hipStream_t st) {
    const int n = p.n, g = g_pm.g, nt = g_pm.ntile;
    // at least 4 particles per thread, at most BIN_WGS workgroups: the counts of
    // each are a row that bin_prefix walks
    const int nw = std::max(1, std::min(BIN_WGS, n / (4 * BIN_THREADS)));
    const int per = (n + nw - 1) / nw;
    bin_count<ORDER, TILES><<<nw, BIN_THREADS, 0, st>>>(p.x, p.y, p.z, n, per, g, nt, g_pm.bins);
    CT2_LAUNCH_CHECK();
    // few counts: cheaper summed by every workgroup than by one more launch
    const bool few = nw <= 16 && nt <= BIN_THREADS;
    if (!few) {
        bin_prefix<<<(nt + PM_BLOCK - 1) / PM_BLOCK, PM_BLOCK, 0, st>>>(g_pm.bins, nw, nt, g_pm.tcount);
        CT2_LAUNCH_CHECK();
    }
    bin_scatter<ORDER, TILES><<<nw, BIN_THREADS, 0, st>>>(p.x, p.y, p.z, n, per, g, nt, g_pm.bins,
                                                          few ? nullptr : g_pm.tcount, g_pm.tstart, g_pm.order);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

template <int ORDER>
int bin_particles(const Slab& p, hipStream_t st) {
    CT2_TRY(ensure_deposit((size_t)p.n));
    const int n = p.n, g = g_pm.g, nt = g_pm.ntile;
    if (nt <= BIN_TILES / 8) return bin_in_lds<ORDER, BIN_TILES / 8>(p, st);
    if (nt <= BIN_TILES) return bin_in_lds<ORDER, BIN_TILES>(p, st);
    const unsigned pb = (unsigned)((n + PM_BLOCK - 1) / PM_BLOCK);
    fill_i32<<<(nt + PM_BLOCK - 1) / PM_BLOCK, PM_BLOCK, 0, st>>>(g_pm.tcount, nt);
    CT2_LAUNCH_CHECK();
    bin_global<ORDER, false><<<pb, PM_BLOCK, 0, st>>>(p.x, p.y, p.z, n, g, g_pm.tcount, nullptr);
    CT2_LAUNCH_CHECK();
    tile_scan<<<1, BIN_THREADS, 0, st>>>(g_pm.tcount, nt, g_pm.tstart);
    CT2_LAUNCH_CHECK();
    bin_global<ORDER, true><<<pb, PM_BLOCK, 0, st>>>(p.x, p.y, p.z, n, g, g_pm.tcount, g_pm.order);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

// Whether the deposit goes by tiles: below 2^17 stencil nodes in all, clearing
// the grid and one global atomic per particle and node are fewer launches and
// faster (us per PM force, per particle / tiled: CIC 4,096 particles on 32^3
// 23.1 / 32.6, 8,000 on 64^3 32.3 / 42.7, 32,768 on 64^3 36.3 / 40.0 from a
// lattice and 52.5 / 45.5 clustered; TSC 4,096 on 32^3 27.0 / 37.1, 32,768 on 64^3
// 52.1 / 44.2).
template <int ORDER>
bool tiles_pay(long n, int g) {
    return g >= TILE_MIN_G && n * (ORDER == 1 ? 8 : 27) > 1L << 17;
}

// Density of the container's particles into g_pm.W.
template <int ORDER>
int deposit(const Context& c) {
    const int n = (int)c.n, g = g_pm.g;
    if (!tiles_pay<ORDER>(n, g)) {
        const long n3 = 1L << (3 * g);
        fill_u64<<<(unsigned)((n3 + PM_BLOCK - 1) / PM_BLOCK), PM_BLOCK, 0, c.stream>>>(g_pm.W, n3);
        CT2_LAUNCH_CHECK();
        mesh_deposit<ORDER><<<(n + PM_BLOCK - 1) / PM_BLOCK, PM_BLOCK, 0, c.stream>>>(c.x, c.y, c.z, n, g, g_pm.W);
        CT2_LAUNCH_CHECK();
        return CT2_OK;
    }
    const int nt = g_pm.ntile, count = slab_count(c);
    for (int k = 0; k < count; ++k) {
        const Slab p = slab(c, k);
        CT2_TRY(bin_particles<ORDER>(p, c.stream));
        auto dep = [&](auto kernel) {
            kernel<<<nt, tile_threads(nt), 0, c.stream>>>(p.x, p.y, p.z, g_pm.order, g_pm.tstart, g, k > 0, g_pm.W);
        };
        tile_threads(nt) == 1024 ? dep(dep_tile<ORDER, 1024>) : dep(dep_tile<ORDER, 512>);
        CT2_LAUNCH_CHECK();
    }
    return CT2_OK;
}

// Force and potential by tiles; the lists of the last slab are in place.
template <int ORDER>
int interp_by_tiles(const Context& c) {
    const int count = slab_count(c), nt = g_pm.ntile;
    for (int k = count - 1; k >= 0; --k) {
        const Slab p = slab(c, k);
        if (k < count - 1) CT2_TRY(bin_particles<ORDER>(p, c.stream));
        auto interp = [&](auto kernel) {
            kernel<<<dim3(nt, 2), tile_threads(nt), 0, c.stream>>>(p.x, p.y, p.z, g_pm.order, g_pm.tstart, g_pm.g, g_pm.A,
                                                                   c.fx + p.first, c.fy + p.first, c.fz + p.first,
                                                                   c.pot + p.first);
        };
        tile_threads(nt) == 1024 ? interp(interp_tile<ORDER, 1024>) : interp(interp_tile<ORDER, 512>);
        CT2_LAUNCH_CHECK();
    }
    return CT2_OK;
}

// FP64 Green's table on the octant |m_d| <= ng/2 (host, libm):
//   G(m) = -4 pi GM exp(-k^2 rs^2) / (k^2 W(m)^2), W = prod_d sinc^(order+1)(pi m_d/ng),
//   G(0) = 0.
std::vector<double> green_table(int ng, double gm, double rs_cells, int order) {
    const int h = ng / 2 + 1;
    const double rs = rs_cells / ng;
    std::vector<double> t((size_t)h * h * h);
    std::vector<double> sinc2(h), k2(h);
    for (int m = 0; m < h; ++m) {
        const double u = M_PI * m / ng;
        const double sc = m ? std::sin(u) / u : 1.0;
        sinc2[m] = order == 1 ? sc * sc : sc * sc * sc;
        k2[m] = (2.0 * M_PI * m) * (2.0 * M_PI * m);
    }
    for (int a = 0; a < h; ++a)
        for (int b = 0; b < h; ++b)
            for (int c = 0; c < h; ++c) {
                double v = 0.0;
                if (a || b || c) {
                    const double w = sinc2[a] * sinc2[b] * sinc2[c];
                    const double kk = k2[a] + k2[b] + k2[c];
                    v = -4.0 * M_PI * gm * std::exp(-kk * rs * rs) / (kk * w * w);
                }
                t[((size_t)a * h + b) * h + c] = v;
            }
    return t;
}

int ensure_table() {
    Context& c = ctx();
    if (g_pm.gm_table == c.opts.GM && g_pm.order_table == g_assign) return CT2_OK;
    const std::vector<double> t = green_table(g_pm.ng, (double)c.opts.GM, g_pm.rs_cells, g_assign);
    CT2_HIP(hipMemcpyAsync(g_pm.G, t.data(), t.size() * sizeof(double), hipMemcpyHostToDevice, c.stream));
    CT2_HIP(hipStreamSynchronize(c.stream));
    g_pm.gm_table = c.opts.GM;
    g_pm.order_table = g_assign;
    return CT2_OK;
}

}  // namespace

int pm_require() {
    CT2_TRY(require_particles());
    if (!g_pm.ng) return set_error(CT2_ERR_STATE, "ct2_pm_init has not been called");
    return CT2_OK;
}

// The PM force and potential of the container into the context force arrays.
// epi: the sinks to kick where the interpolation can do it (then *applied).
static int pm_forces(const Sinks* epi, bool* applied) {
    CT2_TRY(pm_require());
    CT2_TRY(ensure_table());
    Context& c = ctx();
    const int n = (int)c.n, g = g_pm.g;
    const unsigned pb = (unsigned)((n + PM_BLOCK - 1) / PM_BLOCK);
    CT2_TRY(g_assign == 1 ? deposit<1>(c) : deposit<2>(c));
    CT2_TRY(rfft_zy_density(g_pm.W, g_pm.half, g_pm.ng));
    CT2_TRY(xpass(g_pm.ng, g_pm.half, g_pm.A, g_pm.G, c.stream));
    CT2_TRY(fft_inverse_yz(g_pm.A, g_pm.ng, 2));
    // tiles hold n / ntile particles on average: stage a tile's nodes once when
    // that beats one L2 read per particle and stencil node.  Measured, PM force
    // per particle / tiled (TSC): 2^24 particles on 512^3, lattice 6.06 / 5.12 ms,
    // half in Plummer spheres 12.7 / 10.7, random field 4.98 / 5.06.
    // CIC's eight nodes are fewer reads than the lists' on 512^3: 2^26 particles, per
    // particle / tiled: lattice 6.27 / 6.35 ms, cell order 7.53 / 6.44, random order
    // 23.4 / 30.4, half in 64 spheres 21.8 / 34.9.
    const bool tiled = (g_assign == 1 ? tiles_pay<1>(n, g) && g <= 8 : tiles_pay<2>(n, g) && g <= 9) &&
                       (long)n * (g_assign == 1 ? 8 : 27) > 2L * TL_NODES * g_pm.ntile;
    if (tiled) {
        CT2_TRY(g_assign == 1 ? interp_by_tiles<1>(c) : interp_by_tiles<2>(c));
    } else {
        const bool fuse = epi && !near_enabled();
        auto interp = [&](auto kernel) {
            kernel<<<pb, PM_BLOCK, 0, c.stream>>>(c.x, c.y, c.z, n, g, g_pm.A, g_pm.B, c.fx, c.fy, c.fz, c.pot,
                                                  fuse ? *epi : Sinks{});
        };
        if (g_assign == 1)
            fuse ? interp(mesh_interp<1, true>) : interp(mesh_interp<1, false>);
        else
            fuse ? interp(mesh_interp<2, true>) : interp(mesh_interp<2, false>);
        CT2_LAUNCH_CHECK();
        if (applied) *applied = fuse;
    }
    if (near_enabled()) CT2_TRY(near_forces(g_pm.rs_cells / g_pm.ng));
    c.forces_valid = true;
    return CT2_OK;
}

int pm_forces() { return pm_forces(nullptr, nullptr); }

// Device grids for the learned correction's feature gather.
void pm_config(int* ng, double* rs_cells, int* order, double* rcut_rs) {
    *ng = g_pm.ng;
    *rs_cells = g_pm.rs_cells;
    *order = g_assign;
    *rcut_rs = near_rcut_rs();
}

void pm_grids(int* g, const unsigned long long** W, const float2** A, const float2** B) {
    *g = g_pm.g;
    *W = g_pm.W;
    *A = g_pm.A;
    *B = g_pm.B;
}

void release_pm() { free_pm(); }

}  // namespace ct2

using namespace ct2;

extern "C" int ct2_pm_init(int ng, double rs_cells) {
    CT2_TRY(require_init());
    if (!is_pow2(ng) || ng < 8 || ng > 1024)
        return set_error(CT2_ERR_INVALID, "PM grid %d is not a power of two in [8, 1024]", ng);
    if (!(rs_cells >= 0.0) || rs_cells > 64.0) return set_error(CT2_ERR_INVALID, "bad split radius %g", rs_cells);
    if (g_pm.ng == ng && g_pm.rs_cells == rs_cells) return CT2_OK;
    free_pm();
    const size_t n3 = (size_t)ng * ng * ng, h = ng / 2 + 1;
    int rc;
    if ((rc = dev_alloc((void**)&g_pm.W, n3 * sizeof(unsigned long long), "PM density")) ||
        (rc = dev_alloc((void**)&g_pm.half, fft_half_elems(ng) * sizeof(float2), "PM half spectrum")) ||
        (rc = dev_alloc((void**)&g_pm.A, 2 * n3 * sizeof(float2), "PM grids")) ||
        (rc = dev_alloc((void**)&g_pm.G, h * h * h * sizeof(double), "PM Green's table"))) {
        free_pm();
        return rc;
    }
    g_pm.B = g_pm.A + n3;
    g_pm.ng = ng;
    g_pm.g = ilog2(ng);
    if (g_pm.g >= TILE_MIN_G) {
        g_pm.ntile = 1 << (3 * (g_pm.g - TILE_B));
        const size_t nt = (size_t)g_pm.ntile;
        if ((rc = dev_alloc((void**)&g_pm.tcount, nt * sizeof(int), "PM tile counts")) ||
            (nt <= BIN_TILES && (rc = dev_alloc((void**)&g_pm.bins, nt * BIN_WGS * sizeof(int), "PM bins"))) ||
            (rc = dev_alloc((void**)&g_pm.tstart, (size_t)(g_pm.ntile + 1) * sizeof(int), "PM tile starts"))) {
            free_pm();
            return rc;
        }
    }
    g_pm.rs_cells = rs_cells;
    g_pm.gm_table = 0.0f;
    return CT2_OK;
}

extern "C" int ct2_pm_near(double rcut_rs) {
    CT2_TRY(require_init());
    if (!g_pm.ng) return set_error(CT2_ERR_STATE, "ct2_pm_init has not been called");
    if (rcut_rs > 0.0 && !(g_pm.rs_cells > 0.0))
        return set_error(CT2_ERR_INVALID, "the near field needs a PM split radius rs > 0");
    if (rcut_rs > 0.0 && rcut_rs * g_pm.rs_cells / g_pm.ng > 1.0 / 3.0)
        return set_error(CT2_ERR_INVALID, "near-field cutoff %g rs exceeds a third of the box", rcut_rs);
    return near_set(rcut_rs);
}

extern "C" int ct2_pm_near_cells(void) { return near_cells(); }

extern "C" int ct2_pm_assignment(int order) {
    CT2_TRY(require_init());
    if (order != 1 && order != 2) return set_error(CT2_ERR_INVALID, "assignment order %d is not 1 (CIC) or 2 (TSC)", order);
    g_assign = order;
    return CT2_OK;
}

extern "C" int ct2_pm_forces(void) { return pm_forces(); }

extern "C" int ct2_kick_pm(const ct2_kick_params* p, unsigned flags, int* max_rung) {
    CT2_TRY(pm_require());
    CT2_TRY(check_kick_params(p));
    if (flags & ~(unsigned)CT2_KICK_STORE) return set_error(CT2_ERR_INVALID, "unknown flags 0x%x", flags);
    Sinks sinks;
    bool applied = false;
    CT2_TRY(begin_epilogue(p, &sinks));
    CT2_TRY(pm_forces(epilogue_active(p) ? &sinks : nullptr, &applied));
    ctx().last_path = near_enabled() ? CT2_PATH_PM_NEAR : CT2_PATH_PM;
    return finish_epilogue(p, sinks, applied, max_rung);
}

extern "C" int ct2_pm_density_download(uint64_t* host) {
    CT2_TRY(require_init());
    if (!g_pm.ng) return set_error(CT2_ERR_STATE, "ct2_pm_init has not been called");
    if (!host) return set_error(CT2_ERR_INVALID, "null output");
    Context& c = ctx();
    const size_t n3 = (size_t)g_pm.ng * g_pm.ng * g_pm.ng;
    CT2_HIP(hipMemcpyAsync(host, g_pm.W, n3 * 8, hipMemcpyDeviceToHost, c.stream));
    CT2_HIP(hipStreamSynchronize(c.stream));
    return CT2_OK;
}

extern "C" int ct2_pm_grid_download(int which, float* host) {
    CT2_TRY(require_init());
    if (!g_pm.ng) return set_error(CT2_ERR_STATE, "ct2_pm_init has not been called");
    if (!host || (which != 0 && which != 1)) return set_error(CT2_ERR_INVALID, "bad grid request");
    Context& c = ctx();
    const size_t n3 = (size_t)g_pm.ng * g_pm.ng * g_pm.ng;
    CT2_HIP(hipMemcpyAsync(host, which ? g_pm.B : g_pm.A, n3 * 8, hipMemcpyDeviceToHost, c.stream));
    CT2_HIP(hipStreamSynchronize(c.stream));
    return CT2_OK;
}
