// mm.hip -- ct2's multipole-mesh force (particle.cpp:116-271, kick.cpp:11-29,
// 105-125) on gfx950.
//
// ct2's kick() sums, for the particles of each cell, direct pairs with the
// cells of its neighbour list and a local expansion of everything else about
// the cell centre; the expansions are a convolution over the cell grid done
// with one FFT per multipole component.  The reference's P2M, MG2L and L2P
// come from sfmm (spherical harmonics, PORDER = 8), which is not in the tree;
// this module uses Cartesian Taylor expansions of total order P <= 8.
//
//   cells      nc^3, nc a power of two in [8, 256]; lengths below in cells;
//   P2M        M_l(c) = sum_{j in c} (-b_j)^l / l!   (b = x - centre, unit mass);
//   table      D_n(rho) = d^n G_far(rho) at the cell offsets rho, G_far the
//              periodic Green's function minus the nearest image 1/|rho| on the
//              near set |rho|^2 <= 10 (particle.cpp:136), transformed once:
//              Dt[n][q] = D^_n(q) / nc^3 (real for even |n|, i x real for odd);
//   MG2L       L^_k(q) = sum_{|k|+|l|<=P} M^_l(q) D^_{k+l}(q), per wave vector;
//   L2P        pot = sum_k a^k/k! L_k,  F_q = sum_k a^{k-e_q}/(k-e_q)! L_k;
//   near       softened direct pairs with the particles of the near set's cells.
//
// Box units: force GM (near + nc^2 far), potential GM (near + nc far).
//
// The table: G = G_short + G_long (Ewald split beta = 0.5 per cell).
// G_short = sum_m erfc(beta |rho + nc m|)/|rho + nc m| is expanded on the host in
// FP64: for a radial f(s), s = |rho + h|^2, the Taylor coefficients in h are
// sum_j f^(j)(s0)/j! [h^n] (2 rho.h + h.h)^j with f^(j) = (-1/2)^j B_j and
// B_0 = erfc(beta r)/r, B_j = ((2j-1) B_{j-1} + (2 beta^2)^j e^{-beta^2 r^2}/(beta sqrt pi))/r^2
// (Smith 1998); a near offset's own image is -erf(beta r)/r, a power series in s.
// Its samples are transformed with the FP64 3-D FFT.  G_long's sampled
// transform is analytic: sum over aliases kappa = q/nc + m of
// (2 pi i kappa)^n e^{-pi^2 kappa^2/beta^2} / (pi kappa^2), and -pi/beta^2 at 0.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <thread>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "cellsort.h"
#include "epilogue.h"
#include "fft_stages.h"
#include "internal.h"
#include "wave.h"

namespace ct2 {
namespace {

constexpr int MM_PMAX = 8;
constexpr int MM_KMAX = 165;       // components at P = 8
constexpr int MM_NEAR2 = 10;       // |cell offset|^2 of the direct set (particle.cpp:136)
constexpr double MM_BETA = 0.5;    // Ewald split per cell
constexpr int MM_QB = 64;          // wave vectors per MG2L workgroup, one per lane
constexpr int MM_COLS_MAX = 48;    // (dx, dy) columns of the near set (37 at |d|^2 <= 10)
constexpr int MM_WAVES = 4;        // waves per near-field workgroup

// An MG2L work list (one per wave), three times 64 words.  First the outputs:
// P - |k| (0: two components of degree P) | output grid << 4 | degree |k| << 11;
// then, output by output, the rows of the first multipole (8 bits) and of the
// first table value of each run, two runs to a word; last what the wave stages,
// and in its last word the number of outputs.  Rows are the components in column
// order (by (a, b), then the z exponent).
constexpr uint32_t MG2L_NONE = 255u;
constexpr int MG2L_STEPS = 64, MG2L_LIST = 3 * MG2L_STEPS;  // words per list
constexpr uint32_t mg2l_rows(int m, int d) { return (uint32_t)m | (uint32_t)d << 8; }

__constant__ int c_e[MM_KMAX][3];         // exponents of component c
__constant__ float c_ifact[MM_KMAX];      // 1 / (a! b! c!)
__constant__ int c_cols[MM_COLS_MAX][3];  // near set by column: dx, dy, half-height w in z

struct MMIndex {
    int P = 0, K = 0;
    int e[MM_KMAX][3];
    int id[MM_PMAX + 1][MM_PMAX + 1][MM_PMAX + 1];
    double fact[MM_KMAX];
    std::vector<int> pa, pb, pc;  // products within degree P: (i, j) -> i + j
    void init(int p) {
        P = p;
        K = (P + 1) * (P + 2) * (P + 3) / 6;
        std::memset(id, -1, sizeof id);
        int c = 0;
        for (int d = 0; d <= P; ++d)
            for (int a = d; a >= 0; --a)
                for (int b = d - a; b >= 0; --b) {
                    e[c][0] = a;
                    e[c][1] = b;
                    e[c][2] = d - a - b;
                    id[a][b][d - a - b] = c;
                    fact[c] = std::tgamma(a + 1.0) * std::tgamma(b + 1.0) * std::tgamma(d - a - b + 1.0);
                    ++c;
                }
        pa.clear();
        pb.clear();
        pc.clear();
        for (int i = 0; i < K; ++i)
            for (int j = 0; j < K; ++j) {
                const int a = e[i][0] + e[j][0], b = e[i][1] + e[j][1], d = e[i][2] + e[j][2];
                if (a + b + d > P) continue;
                pa.push_back(i);
                pb.push_back(j);
                pc.push_back(id[a][b][d]);
            }
    }
    int deg(int c) const { return e[c][0] + e[c][1] + e[c][2]; }
};

struct MMState {
    int nc = 0, P = 0, K = 0, nz = 0;  // nz = complex grids (K/2 rounded up)
    int ncols = 0;
    double* Dt = nullptr;  // [K][nc^3]
    size_t Dt_bytes = 0;
    float* Dt32 = nullptr;  // the same rounded to FP32, the rows MG2L reads
    size_t Dt32_bytes = 0;
    float2* Zm = nullptr;  // multipole grids [nz][nc^3], then their transforms
    float2* Zl = nullptr;  // local-expansion grids
    size_t Z_bytes = 0;
    uint4* other = nullptr;    // the sort's second buffer (n)
    size_t other_bytes = 0;
    void* sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    uint4* Ps = nullptr;  // sorted (x, y, z, index)
    size_t Ps_bytes = 0;
    int* start = nullptr;  // cell starts (nc^3 + 1)
    size_t start_bytes = 0;
    int2* items = nullptr;  // near-field work items, then their count
    size_t items_bytes = 0;
    int* cnt = nullptr;  // items per cell, the cells' first item (exclusive sum), 16 bits per cell for the runs
    size_t cnt_bytes = 0;
    void* scan_tmp = nullptr;
    size_t scan_tmp_bytes = 0;
    double2* tabz = nullptr;  // one FP64 complex grid while the table is built
    size_t tabz_bytes = 0;
    uint32_t* sched = nullptr;  // the MG2L lists [waves][MG2L_LIST]
    size_t sched_bytes = 0;
    float4* far = nullptr;  // far field per sorted particle, where Zm is too small for it
    size_t far_bytes = 0;
};
MMState g_mm;

// ------------------------------------------------------------ the table (host, FP64)

// s-derivatives of erfc(beta sqrt s)/sqrt s at s = r^2
void erfc_sderiv(int P, double r, double* fs) {
    const double b = MM_BETA, r2 = r * r, ex = std::exp(-b * b * r2) / (b * std::sqrt(M_PI));
    double B = std::erfc(b * r) / r, tb = 1.0, sgn = 1.0;
    fs[0] = B;
    for (int j = 1; j <= P; ++j) {
        tb *= 2.0 * b * b;
        B = ((2 * j - 1) * B + tb * ex) / r2;
        sgn *= -0.5;
        fs[j] = sgn * B;
    }
}

// s-derivatives of -erf(beta sqrt s)/sqrt s = -(2 beta/sqrt pi) sum_i (-beta^2 s)^i/(i! (2i+1))
void erf_sderiv(int P, double s, double* fs) {
    const double b2 = MM_BETA * MM_BETA, c0 = -2.0 * MM_BETA / std::sqrt(M_PI);
    for (int j = 0; j <= P; ++j) {
        double sum = 0.0, term = std::pow(-b2, j);
        for (int i = j; i < j + 400; ++i) {
            const double t = term / (2 * i + 1);
            sum += t;
            if (std::fabs(t) < 1e-19 * std::fabs(sum) && i > j + 4) break;
            term *= -b2 * s / (double)(i - j + 1);
        }
        fs[j] = c0 * sum;
    }
}

// T += Taylor coefficients (d^n f / n!) at rho of f(|rho + h|^2), fs = f^(j)(|rho|^2)
void radial_taylor_add(const MMIndex& I, const double* rho, const double* fs, double* T) {
    double delta[MM_KMAX] = {}, pw[MM_KMAX] = {}, nx[MM_KMAX];
    for (int q = 0; q < 3; ++q) {
        int a[3] = {0, 0, 0};
        a[q] = 1;
        delta[I.id[a[0]][a[1]][a[2]]] = 2.0 * rho[q];
        a[q] = 2;
        if (I.P >= 2) delta[I.id[a[0]][a[1]][a[2]]] = 1.0;
    }
    pw[0] = 1.0;
    T[0] += fs[0];
    double jf = 1.0;
    const size_t np = I.pa.size();
    for (int j = 1; j <= I.P; ++j) {
        std::fill(nx, nx + I.K, 0.0);
        for (size_t p = 0; p < np; ++p) nx[I.pc[p]] += pw[I.pa[p]] * delta[I.pb[p]];
        std::copy(nx, nx + I.K, pw);
        jf *= j;
        const double c = fs[j] / jf;
        for (int k = 0; k < I.K; ++k) T[k] += c * pw[k];
    }
}

int wrap_offset(int i, int nc) { return i < nc / 2 ? i : i - nc; }

// D_n of G_short (less the near set's nearest image) at every cell, [K][nc^3];
// cells beyond the cutoff stay zero.  Split over host threads.
void short_samples(const MMIndex& I, int nc, std::vector<double>& S) {
    const size_t n3 = (size_t)nc * nc * nc;
    S.assign(n3 * I.K, 0.0);
    const double rc = 8.0 / MM_BETA;  // erfc(beta r)/r and its derivatives < 1e-16 of their size beyond
    const int mr = (int)std::ceil(rc / nc) + 1;
    auto work = [&](size_t c0, size_t c1) {
        double fs[MM_PMAX + 1], T[MM_KMAX];
        for (size_t cell = c0; cell < c1; ++cell) {
            const int o[3] = {wrap_offset((int)(cell / ((size_t)nc * nc)), nc), wrap_offset((int)(cell / nc % nc), nc),
                              wrap_offset((int)(cell % nc), nc)};
            const bool near = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] <= MM_NEAR2;
            bool any = false;
            std::fill(T, T + I.K, 0.0);
            for (int m0 = -mr; m0 <= mr; ++m0)
                for (int m1 = -mr; m1 <= mr; ++m1)
                    for (int m2 = -mr; m2 <= mr; ++m2) {
                        const double r[3] = {(double)o[0] + nc * m0, (double)o[1] + nc * m1, (double)o[2] + nc * m2};
                        const double s = r[0] * r[0] + r[1] * r[1] + r[2] * r[2];
                        if (near && !m0 && !m1 && !m2) {
                            erf_sderiv(I.P, s, fs);
                        } else {
                            if (s >= rc * rc) continue;
                            erfc_sderiv(I.P, std::sqrt(s), fs);
                        }
                        radial_taylor_add(I, r, fs, T);
                        any = true;
                    }
            if (any)
                for (int k = 0; k < I.K; ++k) S[(size_t)k * n3 + cell] = T[k] * I.fact[k];
        }
    };
    const unsigned nt = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    std::vector<std::thread> th;
    for (unsigned t = 0; t < nt; ++t) th.emplace_back(work, n3 * t / nt, n3 * (t + 1) / nt);
    for (auto& t : th) t.join();
}

// Dt[c][q] = (parity part of the transformed short samples + the analytic
// long-range transform) / nc^3 for one component c of exponents (a, b, d);
// Dt32 the same rounded to FP32.
__global__ __launch_bounds__(256) void mm_table_finish(const double2* __restrict__ Z, int nc, int a, int b, int d,
                                                       double* __restrict__ Dt, float* __restrict__ Dt32) {
    const size_t n3 = (size_t)nc * nc * nc;
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= n3) return;
    const int deg = a + b + d;
    const int q0 = (int)(q / ((size_t)nc * nc)), q1 = (int)(q / nc % nc), q2 = (int)(q % nc);
    const double k0 = (double)(q0 < nc / 2 ? q0 : q0 - nc) / nc, k1 = (double)(q1 < nc / 2 ? q1 : q1 - nc) / nc,
                 k2 = (double)(q2 < nc / 2 ? q2 : q2 - nc) / nc;
    const double b2 = MM_BETA * MM_BETA, tp = 2.0 * M_PI;
    double lr = 0.0;
    for (int m0 = -1; m0 <= 1; ++m0)
        for (int m1 = -1; m1 <= 1; ++m1)
            for (int m2 = -1; m2 <= 1; ++m2) {
                const double x = k0 + m0, y = k1 + m1, z = k2 + m2, kk = x * x + y * y + z * z;
                if (kk == 0.0) continue;
                double mono = exp(-M_PI * M_PI * kk / b2) / (M_PI * kk);
                for (int i = 0; i < a; ++i) mono *= tp * x;
                for (int i = 0; i < b; ++i) mono *= tp * y;
                for (int i = 0; i < d; ++i) mono *= tp * z;
                lr += mono;
            }
    const double s = ((deg >> 1) & 1) ? -1.0 : 1.0;  // i^deg = s or i s
    double v = (deg & 1) ? Z[q].y + s * lr : Z[q].x + s * lr;
    if (deg == 0 && q == 0) v -= M_PI / b2;
    Dt[q] = v / (double)n3;
    Dt32[q] = (float)(v / (double)n3);
}

// ------------------------------------------------------------ binning

struct MMCellKey {
    int lg;
    __device__ __forceinline__ uint32_t operator()(const uint4& p) const {
        const int sh = 32 - lg;
        return (((p.x >> sh) << lg | (p.y >> sh)) << lg) | (p.z >> sh);
    }
};

// start[c] = first sorted slot of cell c, start[n3] = n
struct PutCell {
    int* start;
    __device__ __forceinline__ void operator()(long c, long e) const { start[c] = (int)e; }
};

// Near-field work items.  The sinks of a row of cells (fixed x and y), in cell
// order, form runs of at most MM_RUN that span fewer than zspan cells, and the
// separations of a run are FP32 offsets from the centre of its first cell.  The
// runs are part of the result, not of the split: the rounding of a close pair's
// separation grows with its distance from that centre, so other centres move the
// forces of a set's closest pairs, and so all of them by up to 2.4e-5 (2-norm).  An item is
// at most MM_SINKS sinks of one cell and one run, as even as they go:
// (cell | cells from the run's first to it << 24 | sinks << 27, first sink).
constexpr int MM_SINKS = 10, MM_RUN = 64;
constexpr int mm_zspan(int nc) { return nc >= 32 ? 8 : nc >= 16 ? 4 : 1; }  // the offsets stay minimum images (8^3: exact, no runs)
constexpr int MM_HEAD_BITS = 7;  // of a part: MM_RUN sinks and none

__device__ __forceinline__ int mm_groups(int sinks) { return (sinks + MM_SINKS - 1) / MM_SINKS; }

// A wave per row walks its cells.  part[c]: how many of the cell's sinks at most
// still belong to the run that holds its first one, and that run's first cell (so
// many cells before | << MM_HEAD_BITS); later runs start in the cell, every MM_RUN
// sinks.  cnt[c]: its items.
__global__ __launch_bounds__(256) void mm_item_counts(const int* __restrict__ start, int lg, int zspan,
                                                      int* __restrict__ cnt, uint16_t* __restrict__ part) {
    const int nc = 1 << lg, lane = threadIdx.x & 63;
    const int row = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
    const int* st = start + ((size_t)row << lg);
    int end = 0, ref = 0;  // of the run so far
    for (int z0 = 0; z0 < nc; z0 += 64) {
        const int z = z0 + lane;
        const bool in = z < nc;
        const int a = in ? st[z] : 0, b = in ? st[z + 1] : 0, reach = in ? st[min(z + zspan, nc)] : 0;
        int head = 0, from = 0;
        for (uint64_t m = __ballot(a < b); m; m &= m - 1) {
            const int l = __ffsll((unsigned long long)m) - 1;
            const int ca = __builtin_amdgcn_readlane(a, l), cb = __builtin_amdgcn_readlane(b, l),
                      cr = __builtin_amdgcn_readlane(reach, l);
            if (ca >= end) {
                ref = z0 + l;
                end = ca + min(MM_RUN, cr - ca);
            }
            if (lane == l) {
                head = end - ca;
                from = ref;
            }
            if (end < cb) {  // the last run that starts in this cell
                ref = z0 + l;
                const uint32_t more = ((uint32_t)(cb - end) + MM_RUN - 1) / MM_RUN * MM_RUN;
                end += (int)min(more, (uint32_t)(cr - end));
            }
        }
        if (!in) continue;
        const int c = (row << lg) + z, later = max(b - a - head, 0);
        cnt[c] = mm_groups(min(b - a, head)) + later / MM_RUN * mm_groups(MM_RUN) + mm_groups(later % MM_RUN);
        part[c] = (uint16_t)(min(head, MM_RUN) | (z - from) << MM_HEAD_BITS);
    }
}

// After the counts' exclusive sum: the items and their number.
__global__ __launch_bounds__(256) void mm_items(const int* __restrict__ start, const int* __restrict__ cnt,
                                                const uint16_t* __restrict__ part, const int* __restrict__ first, int n3,
                                                int2* __restrict__ items, int* __restrict__ nitems) {
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= n3) return;
    int f = first[c];
    if (c == n3 - 1) *nitems = f + cnt[c];
    if (cnt[c] == 0) return;
    int a = start[c], back = part[c] >> MM_HEAD_BITS, len = part[c] & ((1 << MM_HEAD_BITS) - 1);
    for (const int b = start[c + 1]; a < b; back = 0, len = MM_RUN) {
        const int n = min(b - a, len), groups = mm_groups(n);
        for (int g = 0; g < groups; ++g) {
            const int s0 = g * n / groups, s1 = (g + 1) * n / groups;
            items[f++] = make_int2(c | back << 24 | (s1 - s0) << 27, a + s0);
        }
        a += n;
    }
}

// ------------------------------------------------------------ P2M

// MM_P2M_CELLS consecutive cells per workgroup, a wave taking every fourth: the
// powers of -b (offset from the cell centre, in cells) of up to MM_P2M_PART
// particles in the wave's LDS slot (one lane per particle and axis), lane c (and
// c + 64, c + 128) sums component c over them in FP64, four particles' reads in
// flight together; the moments of the block's cells collect in LDS and leave as
// rows of MM_P2M_CELLS consecutive cells (128 bytes) per grid.  Component c goes
// to grid c/2, real part for even c, imaginary for odd (an odd K leaves the last
// imaginary part 0).  Bound by the latency of its LDS reads: 19 KB of LDS per
// workgroup, so that eight share a CU (with room for 64 particles per wave and
// 32 cells, three did), took order 8 on 64^3 cells of 8 particles from 299 to
// 125 us.
constexpr int MM_P2M_CELLS = 16, MM_P2M_PART = 16;
__global__ __launch_bounds__(256) void mm_p2m(const uint4* __restrict__ P, const int* __restrict__ start, int lg, int Pord,
                                              int K, size_t n3, float2* __restrict__ Zm) {
    __shared__ float pw[4][MM_P2M_PART][3][MM_PMAX + 1];
    __shared__ float Mo[MM_KMAX + 1][MM_P2M_CELLS + 1];  // + 1: a cell's column spreads over the banks
    static_assert(3 * MM_P2M_PART <= 64 && MM_P2M_PART % 4 == 0, "a lane per particle and axis, four particles at a time");
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const size_t cell0 = (size_t)blockIdx.x * MM_P2M_CELLS;
    const int sh = 32 - lg;
    const uint32_t mask = (1u << sh) - 1u, half = 1u << (sh - 1);
    const float inv = ldexpf(1.0f, -sh);
    const int q = lane / MM_P2M_PART, j = lane % MM_P2M_PART;
    int ex[3][3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        const int c = lane + 64 * r;
        ex[r][0] = c < K ? c_e[c][0] : 0;
        ex[r][1] = c < K ? c_e[c][1] : 0;
        ex[r][2] = c < K ? c_e[c][2] : 0;
    }
    for (int lc = w; lc < MM_P2M_CELLS; lc += 4) {
        const size_t cell = cell0 + lc;
        const int s0 = start[cell], s1 = start[cell + 1];
        double acc[3] = {0.0, 0.0, 0.0};
        for (int base = s0; base < s1; base += MM_P2M_PART) {
            if (q < 3) {
                // past the cell's last particle: all powers 0, so that it adds nothing
                const bool have = base + j < s1;
                const uint32_t v = have ? ((const uint32_t*)(P + base + j))[q] : 0u;
                const float mb = have ? -(float)(int32_t)((v & mask) - half) * inv : 0.0f;  // -b in cells
                float pv = have ? 1.0f : 0.0f;
                for (int e = 0; e <= Pord; ++e) {
                    pw[w][j][q][e] = pv;
                    pv *= mb;
                }
            }
            wave_sync();
            const int cnt = min(MM_P2M_PART, s1 - base);
            for (int j0 = 0; j0 < cnt; j0 += 4) {
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    if (lane + 64 * r >= K) continue;
                    float m[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        m[u] = pw[w][j0 + u][0][ex[r][0]] * pw[w][j0 + u][1][ex[r][1]] * pw[w][j0 + u][2][ex[r][2]];
#pragma unroll
                    for (int u = 0; u < 4; ++u) acc[r] += (double)m[u];
                }
            }
            wave_sync();
        }
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int c = lane + 64 * r;
            if (c < K) Mo[c][lc] = (float)(acc[r] * (double)c_ifact[c]);
            else if (c == K) Mo[c][lc] = 0.0f;  // the imaginary part of an unpaired last component
        }
    }
    __syncthreads();
    // grid j, cells cell0 .. cell0 + MM_P2M_CELLS - 1: (M_2j, M_2j+1)
    const int nz = (K + 1) / 2;
    for (int e = t; e < nz * MM_P2M_CELLS; e += 256) {
        const int jz = e / MM_P2M_CELLS, lc = e % MM_P2M_CELLS;
        Zm[(size_t)jz * n3 + cell0 + lc] = make_float2(Mo[2 * jz][lc], Mo[2 * jz + 1][lc]);
    }
}

// ------------------------------------------------------------ MG2L

// L^_k = sum_l M^_l D^_{k+l} per wave vector.  With M'_l = i^|l| M^_l and the
// table's D^_n = i^|n| D'_n (D' real), L^_k = i^|k| sum_l M'_l D'_{k+l}: one
// complex by real product per term, whatever the parities.  MM_QB wave vectors
// per workgroup, one per lane: the transformed multipoles, unpacked from the
// paired grids (Z(q) and Z(-q)) and turned by i^|l|, and the table rows with
// their sign in LDS, in column order.  An output is the pair k, k + e_z (z
// exponents kz, kz + 1, kz even): for every column (lx, ly) it takes the run of
// R + 1 multipoles and of R + 1 table values from LDS once, for 2 R + 1 products.
// Up to four products sum in FP32 (the multipoles are FP32 already), these sums
// in FP64.  Written as i^|k| (S_k - S_{k+e_z}) = L^_k + i L^_{k+e_z}, ready for
// the inverse transforms; the highest z exponents left over, of one product each,
// in pairs (S_a + i S_b).  The waves of a workgroup walk lists of outputs of about
// equal cost, the same for every workgroup, so that P - |k| is uniform and the
// whole of an output unrolled.  A list of single products, read from LDS for each
// (36 KB per wave vector at order 8, now 22 KB) with five instructions on its
// address and parity, took 507 us on 64^3 cells; this 181.  Bound by LDS reads
// (about 75 us) and by the conversions to FP64, at four waves per SIMD (the LDS).
struct Mg2lSum {
    double ar, ai;
    float tr, ti;
};

// The runs of an output from the N-th of length R + 1 on, r = P - |k|: r - R + 1
// of each length; Q products are done.  `at`: the output's first word of runs.
template <int r, int R, int N, int Q>
__device__ __forceinline__ void mg2l_runs(const float2 (*Mh)[MM_QB], const float (*Dq)[MM_QB], uint32_t rows, int at, int lane,
                                          Mg2lSum& s) {
    if constexpr (N <= r - R) {
        constexpr int n = (r - R) * (r - R + 1) / 2 + N;  // runs done
        const uint32_t w = (uint32_t)__builtin_amdgcn_readlane(rows, at + n / 2) >> 16 * (n & 1);
        const float2* m = &Mh[w & 255u][lane];
        const float* d = &Dq[w >> 8 & 255u][lane];
        float2 mv[R + 1];
        float dv[R + 1];
#pragma unroll
        for (int u = 0; u <= R; ++u) {
            mv[u] = m[u * MM_QB];
            dv[u] = d[u * MM_QB];
        }
#pragma unroll
        for (int p = 0; p < 2 * R + 1; ++p) {  // m_u d_u, then -m_u d_(u+1)
            const float e = p & 1 ? -dv[p / 2 + 1] : dv[p / 2];
            if (((Q + p) & 3) == 0) {
                s.tr = mv[p / 2].x * e;
                s.ti = mv[p / 2].y * e;
            } else {
                s.tr = fmaf(mv[p / 2].x, e, s.tr);
                s.ti = fmaf(mv[p / 2].y, e, s.ti);
            }
            if (((Q + p) & 3) == 3) {
                s.ar += (double)s.tr;
                s.ai += (double)s.ti;
            }
        }
        mg2l_runs<r, R, N + 1, Q + 2 * R + 1>(Mh, Dq, rows, at, lane, s);
    } else if constexpr (R > 0) {
        mg2l_runs<r, R - 1, 0, Q>(Mh, Dq, rows, at, lane, s);
    } else if constexpr (Q & 3) {
        s.ar += (double)s.tr;
        s.ai += (double)s.ti;
    }
}

// v i^d, d uniform
__device__ __forceinline__ float2 turn(float2 v, uint32_t d) {
    const float x = d & 1 ? v.y : v.x, y = d & 1 ? v.x : v.y;
    return make_float2(__uint_as_float(__float_as_uint(x) ^ (d + 1 & 2) << 30), __uint_as_float(__float_as_uint(y) ^ (d & 2) << 30));
}

// PMAX: room for expansions up to that order; WAVES work lists.  At PMAX = 8 one
// workgroup fills a CU's LDS, so the workgroups are persistent and hold the next
// block's reads in registers while they work on this one.
template <int PMAX, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void mm_mg2l(const float2* __restrict__ Zm, const float* __restrict__ Dt32,
                                                      const uint32_t* __restrict__ sched, int nc, int K, int nz,
                                                      float2* __restrict__ Zl) {
    constexpr int KMAX = (PMAX + 1) * (PMAX + 2) * (PMAX + 3) / 6;
    constexpr int NZ = ((KMAX + 1) / 2 + WAVES - 1) / WAVES, ND = (KMAX + WAVES - 1) / WAVES;
    __shared__ float2 Mh[KMAX][MM_QB];
    __shared__ float Dq[KMAX][MM_QB];
    const int n3 = nc * nc * nc, blocks = n3 / MM_QB, m = nc - 1, lg = __ffs(nc) - 1;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t* list = sched + wave * MG2L_LIST;
    uint32_t outs = list[lane], rows = list[MG2L_STEPS + lane], stage = list[2 * MG2L_STEPS + lane];
    // here, so that no wait for them stands between the reads below and their use
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(outs), "+v"(rows), "+v"(stage));
    const int count = (int)__builtin_amdgcn_readlane(stage, 63);
    float2 za[NZ], zb[NZ];
    float dv[ND];
    const auto fetch = [&](int block) {
        const int q = block * MM_QB + lane;
        const int qn = ((-(q >> 2 * lg) & m) << 2 * lg) | ((-(q >> lg) & m) << lg) | (-q & m);
#pragma unroll
        for (int i = 0; i < NZ; ++i) {
            const int j = min(wave + WAVES * i, nz - 1);
            za[i] = Zm[(size_t)j * n3 + q];
            zb[i] = Zm[(size_t)j * n3 + qn];
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) dv[i] = Dt32[(size_t)min(wave + WAVES * i, K - 1) * n3 + q];
    };
    fetch(blockIdx.x);
    for (int block = blockIdx.x; block < blocks; block += gridDim.x) {
        __syncthreads();  // the block before is done with the LDS
#pragma unroll
        for (int i = 0; i < NZ; ++i) {
            const int j = wave + WAVES * i;
            if (j >= nz) break;
            const uint32_t s = __builtin_amdgcn_readlane(stage, i);  // rows and degrees of the components 2j, 2j + 1
            const float2 a = za[i], b = zb[i];
            // (Z(q) + conj Z(-q)) / 2 and / 2i
            Mh[s & 255u][lane] = turn(make_float2(0.5f * (a.x + b.x), 0.5f * (a.y - b.y)), s >> 16);
            if (2 * j + 1 < K)
                Mh[s >> 8 & 255u][lane] = turn(make_float2(0.5f * (a.y + b.y), 0.5f * (b.x - a.x)), s >> 24);
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            if (wave + WAVES * i >= K) break;
            const uint32_t s = __builtin_amdgcn_readlane(stage, 16 + i);  // row and sign of a table component
            Dq[s & 255u][lane] = __uint_as_float(__float_as_uint(dv[i]) ^ (s & 0x80000000u));
        }
        __syncthreads();
        if (block + (int)gridDim.x < blocks) fetch(block + gridDim.x);
        for (int i = 0, at = 0; i < count; ++i) {
            const uint32_t w = __builtin_amdgcn_readlane(outs, i);
            const int r = (int)(w & 15u);
            Mg2lSum s{0.0, 0.0, 0.0f, 0.0f};
            switch (r) {
#define CT2_MM_OUT(R) \
    case R: \
        if constexpr (R <= PMAX) mg2l_runs<R, R, 0, 0>(Mh, Dq, rows, at, lane, s); \
        break;
                CT2_MM_OUT(1) CT2_MM_OUT(2) CT2_MM_OUT(3) CT2_MM_OUT(4) CT2_MM_OUT(5) CT2_MM_OUT(6) CT2_MM_OUT(7) CT2_MM_OUT(8)
#undef CT2_MM_OUT
                default: {  // S_a and S_b of two components of degree P; the second maybe absent
                    const uint32_t c = __builtin_amdgcn_readlane(rows, at);
                    const float2 m0 = Mh[0][lane];
                    const float da = Dq[c & 255u][lane], db = (c >> 8) == MG2L_NONE ? 0.0f : Dq[c >> 8][lane];
                    s.ar = m0.x * da - m0.y * db;
                    s.ai = m0.y * da + m0.x * db;
                }
            }
            at += r ? ((r + 1) * (r + 2) / 2 + 1) / 2 : 1;
            Zl[(size_t)(w >> 4 & 127u) * n3 + block * MM_QB + lane] = turn(make_float2((float)s.ar, (float)s.ai), w >> 11);
        }
    }
}

// ------------------------------------------------------------ L2P

// Where the local expansion's components lie: pairs of z exponents (d, d + 1), d
// even, column by column, then the highest exponents left over two by two.  Two
// components share a complex FP32 transform and its noise, of the size of the larger
// one: the smallest degree's falls on the z force (with components paired by their
// number it fell on x), and the whole force's error does not depend on it.
template <int P>
struct LocalGrids {
    int pair[P + 1][P + 1] = {};    // grid of a column's first pair
    int single[P + 1][P + 1] = {};  // rank of a column's left-over component
    int pairs = 0;
    constexpr LocalGrids() {
        int n = 0;
        for (int e = 0; e <= P; ++e)
            for (int a = e; a >= 0; --a) {
                pair[a][e - a] = pairs;
                pairs += (P - e + 1) / 2;
                if ((P - e) % 2 == 0) single[a][e - a] = n++;
            }
    }
};

// The local expansion of a particle's cell at its offset from the centre, one
// thread per particle in cell order: (d/dx, d/dy, d/dz) and the value, in cells.
// Columns of z exponents by powers over factorials, so that a component costs two
// multiply-adds, with every exponent a constant (order 8: 0.5 k instructions per
// particle; by components with exponents read from a table, behind the near
// pairs, it took 5 k and 220 us of 2^21 particles on 64^3 cells, this 95).
// Bound by reading the grids once.
template <int P>
__global__ __launch_bounds__(256) void mm_l2p(const uint4* __restrict__ Ps, const float2* __restrict__ Zl, int n, int lg,
                                              float4* __restrict__ far) {
    static constexpr LocalGrids<P> G{};
    const int i = (int)xcd_contiguous(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const uint4 me = Ps[i];
    const int sh = 32 - lg;
    const uint32_t half = 1u << (sh - 1), low = (1u << sh) - 1u;
    const size_t n3 = (size_t)1 << 3 * lg;
    const float2* z = Zl + (((size_t)(me.x >> sh) << 2 * lg) | ((size_t)(me.y >> sh) << lg) | (size_t)(me.z >> sh));
    const float inv = ldexpf(1.0f, -sh);
    float px[P + 1], py[P + 1], pz[P + 1];
    px[0] = py[0] = pz[0] = 1.0f;
    const float ax = (float)(int32_t)((me.x & low) - half) * inv, ay = (float)(int32_t)((me.y & low) - half) * inv,
                az = (float)(int32_t)((me.z & low) - half) * inv;
#pragma unroll
    for (int e = 1; e <= P; ++e) {
        px[e] = px[e - 1] * ax * (1.0f / e);
        py[e] = py[e - 1] * ay * (1.0f / e);
        pz[e] = pz[e - 1] * az * (1.0f / e);
    }
    float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int a = 0; a <= P; ++a) {
        float v = 0.f, vy = 0.f, vz = 0.f;
#pragma unroll
        for (int b = 0; b <= P; ++b) {
            if (a + b > P) continue;
            const int top = P - a - b;
            float f = 0.f, fz = 0.f;
#pragma unroll
            for (int d = 0; d <= P; d += 2) {
                if (d > top) continue;
                const int s = G.single[a][b];
                float2 L = z[(size_t)(d < top ? G.pair[a][b] + d / 2 : G.pairs + s / 2) * n3];
                if (d == top && s % 2) L.x = L.y;
                f = fmaf(L.x, pz[d], f);
                if (d) fz = fmaf(L.x, pz[d - 1], fz);
                if (d < top) {
                    f = fmaf(L.y, pz[d + 1], f);
                    fz = fmaf(L.y, pz[d], fz);
                }
            }
            v = fmaf(f, py[b], v);
            vz = fmaf(fz, py[b], vz);
            if (b) vy = fmaf(f, py[b - 1], vy);
        }
        g.w = fmaf(v, px[a], g.w);
        g.y = fmaf(vy, px[a], g.y);
        g.z = fmaf(vz, px[a], g.z);
        if (a) g.x = fmaf(v, px[a - 1], g.x);
    }
    far[i] = g;
}

// ------------------------------------------------------------ near pairs

struct NearK {
    float eps2u, h2u, hinvu, hinv3u;  // as the direct kick, in 2^-32 units
};

// The pair term of the direct set: ddx, ddy, ddz in 2^-32 box units; pad is 0, or
// infinite for a lane past the last source, which makes r^2 infinite and the term 0.
template <int KERNEL>
__device__ __forceinline__ void near_pair(float ddx, float ddy, float ddz, float pad, const NearK& kc, float& tx, float& ty,
                                          float& tz, float& tp) {
    float k, p;
    if constexpr (KERNEL == CT2_KERNEL_PLUMMER) {
        const float r2 = fmaf(ddz, ddz, fmaf(ddy, ddy, fmaf(ddx, ddx, kc.eps2u + pad)));
        const float wv = __builtin_amdgcn_rsqf(r2);
        k = (wv * wv) * wv;
        p = wv;
    } else {
        const float r2 = fmaf(ddz, ddz, fmaf(ddy, ddy, fmaf(ddx, ddx, pad)));
        const bool in = r2 < kc.h2u;
        const float wv = __builtin_amdgcn_rsqf(in ? kc.h2u : r2);
        k = in ? kc.hinv3u : (wv * wv) * wv;
        p = in ? fmaf(-0.5f * kc.hinv3u, r2, 1.5f * kc.hinvu) : wv;
    }
    tx = fmaf(ddx, k, tx);
    ty = fmaf(ddy, k, ty);
    tz = fmaf(ddz, k, tz);
    tp += p;
}

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// One source per lane and step, NS sinks in scalar registers; the partial sums of
// the lanes are left in red[s][16 q + ..], q the component.
constexpr int MM_RED = 68;  // floats per row: 64 and a shift of the banks
template <int KERNEL, bool EXACT, int NS, typename Next>
__device__ __forceinline__ void near_sinks(uint4 own, uint32_t rx, uint32_t ry, uint32_t rz, int steps, const Next& next,
                                           const NearK& kc, int lane, float* __restrict__ red) {
    uint32_t ix[NS], iy[NS], iz[NS];
    float ux[NS], uy[NS], uz[NS], t[4 * NS];
    const float ox = (float)(int32_t)(own.x - rx), oy = (float)(int32_t)(own.y - ry), oz = (float)(int32_t)(own.z - rz);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if constexpr (EXACT) {
            ix[s] = __builtin_amdgcn_readlane(own.x, s);
            iy[s] = __builtin_amdgcn_readlane(own.y, s);
            iz[s] = __builtin_amdgcn_readlane(own.z, s);
        } else {
            ux[s] = lane_value(ox, s);
            uy[s] = lane_value(oy, s);
            uz[s] = lane_value(oz, s);
        }
    }
#pragma unroll
    for (int i = 0; i < 4 * NS; ++i) t[i] = 0.0f;
    float pad1;
    uint4 q1 = next(0, pad1);
    for (int k = 0; k < steps; ++k) {
        const uint4 q = q1;
        const float pad = pad1;
        if (k + 1 < steps) q1 = next(k + 1, pad1);
        if constexpr (EXACT) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
                near_pair<KERNEL>((float)(int32_t)(q.x - ix[s]), (float)(int32_t)(q.y - iy[s]), (float)(int32_t)(q.z - iz[s]),
                                  pad, kc, t[s], t[NS + s], t[2 * NS + s], t[3 * NS + s]);
        } else {
            const float qx = (float)(int32_t)(q.x - rx), qy = (float)(int32_t)(q.y - ry), qz = (float)(int32_t)(q.z - rz);
#pragma unroll
            for (int s = 0; s < NS; ++s)
                near_pair<KERNEL>(qx - ux[s], qy - uy[s], qz - uz[s], pad, kc, t[s], t[NS + s], t[2 * NS + s], t[3 * NS + s]);
        }
    }
    // [aL aH], [bL bH] -> [aL + aH, bL + bH], first by halves of the wave, then by rows of 16
#pragma unroll
    for (int i = 0; i < 2 * NS; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(t[i]), __float_as_uint(t[i + 2 * NS]), false, false);
        t[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(t[s]), __float_as_uint(t[s + NS]), false, false);
        red[s * MM_RED + lane] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
}

// One wave per work item: up to MM_SINKS sinks of a cell, which all have the same
// sources, the particles of the near set's cells.  They are the cells z - w .. z + w
// of the set's (dx, dy) columns, a run of consecutive slots each (one that wraps
// through z = 0 continues a column's length lower); a lane holds a column's run,
// and the runs joined are the item's list, 64 sources to a step, whose lane finds
// its run from the bits of the run heads up to it.  Sources are read and taken as
// FP32 offsets (mm_item_counts says from where) once for all sinks, so that a pair costs
// its 13 instructions, with no lane idle but in the last step; a lane sums every
// 64th source in FP32, then the lanes are summed.  Bound by those instructions at
// the rate that five waves per SIMD issue them: a lane per sink that walked its own
// runs in LDS (idle for a fifth of the time, with 135 instructions per column and
// two per pair on top, but eight waves per SIMD) took 1,109 us for 2^21 particles on
// 64^3 cells, and two small kernels 39 us to cut the rows into its items; this takes
// 1,063 (median of 60 traced passes 1,020) and 18.  12 sinks took 1,081 at five waves and 1,237 at four, 9 the same at
// six; groups of 2 to 6 sinks interleaved by hand 1,177 to 1,320.  EXACT (8^3 cells,
// whose offsets are too coarse): separations from the fixed-point positions.
constexpr int MM_STEPS = 64;  // steps whose run heads are in LDS at a time
template <int KERNEL, bool EXACT>
__global__ __launch_bounds__(64 * MM_WAVES, 5) void mm_near(const uint4* __restrict__ P, const int* __restrict__ start,
                                                         const int2* __restrict__ items, const int* __restrict__ nitems,
                                                         const float* __restrict__ far, int lg, int ncols, NearK kc,
                                                         double fnear, double pnear, double ffar, double pfar,
                                                         float* __restrict__ fx, float* __restrict__ fy,
                                                         float* __restrict__ fz, float* __restrict__ pot) {
    __shared__ uint32_t heads_lds[MM_WAVES][2 * MM_STEPS];
    __shared__ __align__(16) float red_lds[MM_WAVES][MM_SINKS * MM_RED];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t* const heads = heads_lds[w];
    float* const red = red_lds[w];
    const int nc = 1 << lg, sh = 32 - lg, m = nc - 1;
    const uint32_t half = 1u << (sh - 1);
    const int total = *nitems;
    const unsigned blocks = ((unsigned)(total + MM_WAVES - 1) / MM_WAVES + 7u) & ~7u;
    const int dx = lane < ncols ? c_cols[lane][0] : 0, dy = lane < ncols ? c_cols[lane][1] : 0,
              hw = lane < ncols ? c_cols[lane][2] : 0;
    for (unsigned b = blockIdx.x; b < blocks; b += gridDim.x) {
        const int item = (int)xcd_contiguous(b, blocks) * MM_WAVES + w;
        if (item >= total) continue;
        const int it = __builtin_amdgcn_readfirstlane(items[item].x), first = __builtin_amdgcn_readfirstlane(items[item].y);
        const int cell = it & 0xffffff, back = it >> 24 & 7, ns = it >> 27;
        const int cx = cell >> 2 * lg, cy = cell >> lg & m, cz = cell & m;
        const uint4 own = P[first + min(lane, ns - 1)];
        // the lane's column
        const int* st = start + ((((cx + dx) & m) << lg | ((cy + dy) & m)) << lg);  // st[nc] is the end of the column
        const int za = cz - hw, zb = cz + hw + 1;
        const int end = st[nc], count = end - st[0];
        const int s0 = st[za & m];
        int len = st[zb > nc ? zb - nc : zb] - s0 + (za < 0 || zb > nc ? count : 0);
        if (lane >= ncols) len = 0;
        int upto = len;  // of the columns to this one
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(upto, d);
            if (lane >= d) upto += v;
        }
        const int W = __builtin_amdgcn_readlane(upto, 63), at = upto - len;
        // the columns that hold particles first: what a slot is more than its place in the list, and where the column ends
        const uint64_t some = __ballot(len > 0);
        const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(some >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0));
        const int rank = len > 0 ? below : __popcll(some) + lane - below;
        const int shift = __builtin_amdgcn_ds_permute(4 * rank, s0 - at);
        const bool wraps = cz < 3 || cz + 3 >= nc;  // uniform
        const int ends = __builtin_amdgcn_ds_permute(4 * rank, end), counts = __builtin_amdgcn_ds_permute(4 * rank, count);
        const uint32_t rx = ((uint32_t)cx << sh) + half, ry = ((uint32_t)cy << sh) + half, rz = ((uint32_t)(cz - back) << sh) + half;
        double sum = 0.0;
        for (int j0 = 0; j0 < W; j0 += 64 * MM_STEPS) {
            const int steps = min(MM_STEPS, (W - j0 + 63) / 64);
            heads[lane] = heads[64 + lane] = 0;
            wave_sync();
            if (len > 0 && at >= j0 && at < j0 + 64 * MM_STEPS) atomicOr(&heads[(at - j0) >> 5], 1u << (at & 31));
            wave_sync();
            const uint32_t hl = heads[2 * lane], hh = heads[2 * lane + 1];  // of step `lane`
            int run = __popcll(__ballot(len > 0 && at < j0));               // heads before the step
            const auto next = [&](int k, float& pad) {
                const uint64_t h = (uint64_t)__builtin_amdgcn_readlane(hh, k) << 32 | (uint32_t)__builtin_amdgcn_readlane(hl, k);
                const uint64_t up = h >> 1;
                const int r = run + (int)(h & 1) - 1 +
                              (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(up >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)up, 0));
                run += __popcll(h);
                const int j = j0 + 64 * k + lane;
                int slot = j + __builtin_amdgcn_ds_bpermute(4 * r, shift);
                if (wraps) {
                    const int e = __builtin_amdgcn_ds_bpermute(4 * r, ends), c = __builtin_amdgcn_ds_bpermute(4 * r, counts);
                    if (slot >= e) slot -= c;
                }
                pad = j < W ? 0.0f : __builtin_inff();
                return P[j < W ? slot : first];
            };
            switch (ns) {
#define CT2_MM_NS(NS) \
    case NS: near_sinks<KERNEL, EXACT, NS>(own, rx, ry, rz, steps, next, kc, lane, red); break;
                CT2_MM_NS(1) CT2_MM_NS(2) CT2_MM_NS(3) CT2_MM_NS(4) CT2_MM_NS(5) CT2_MM_NS(6) CT2_MM_NS(7) CT2_MM_NS(8)
                CT2_MM_NS(9) CT2_MM_NS(10)
#undef CT2_MM_NS
            }
            wave_sync();
            if (lane < 4 * ns) {  // sink lane / 4, component lane % 4
                const float4* r = (const float4*)(red + (lane >> 2) * MM_RED + 16 * (lane & 3));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 v = r[i];
                    sum += ((double)v.x + (double)v.y) + ((double)v.z + (double)v.w);
                }
            }
            wave_sync();
        }
        const uint32_t i = __shfl(own.w, lane >> 2);
        if (lane < 4 * ns) {
            const int q = lane & 3;
            float* const out = q == 0 ? fx : q == 1 ? fy : q == 2 ? fz : pot;
            out[i] = (float)(sum * (q < 3 ? fnear : pnear) + (double)far[4 * (size_t)first + lane] * (q < 3 ? ffar : pfar));
        }
    }
}

int mm_require() {
    CT2_TRY(require_particles());
    if (!g_mm.nc) return set_error(CT2_ERR_STATE, "ct2_mm_init has not been called");
    return CT2_OK;
}

int mm_forces() {
    Context& c = ctx();
    MMState& s = g_mm;
    const int n = (int)c.n, nc = s.nc, lg = ilog2(nc);
    const int n3 = nc * nc * nc;
    hipStream_t st = c.stream;
    CT2_TRY(ensure_scratch((void**)&s.other, &s.other_bytes, sizeof(uint4) * (size_t)n, "multipole-mesh sort"));
    CT2_TRY(ensure_scratch((void**)&s.Ps, &s.Ps_bytes, sizeof(uint4) * (size_t)n, "multipole-mesh particles"));
    CT2_TRY(ensure_scratch((void**)&s.start, &s.start_bytes, sizeof(int) * ((size_t)n3 + 1), "cell starts"));
    CT2_TRY(ensure_scratch((void**)&s.cnt, &s.cnt_bytes, (2 * sizeof(int) + sizeof(uint16_t)) * (size_t)n3, "item counts"));
    // a part of at most MM_SINKS - 1 sinks beyond full items in each cell and at each end of a run inside one
    const size_t max_items = (size_t)n / MM_SINKS + (size_t)std::min(n, n3) + (size_t)n / MM_RUN;
    CT2_TRY(ensure_scratch((void**)&s.items, &s.items_bytes, sizeof(int2) * max_items + sizeof(int), "work items"));
    int* const nitems = (int*)(s.items + max_items);
    const MMCellKey key{lg};
    CT2_TRY(cell_sort(c.x, c.y, c.z, n, key, 3 * lg, s.Ps, s.other, &s.sort_tmp, &s.sort_tmp_bytes, st));
    CT2_TRY(cell_starts(s.Ps, key, n, n3, PutCell{s.start}, st));
    int* first = s.cnt + n3;
    uint16_t* const part = (uint16_t*)(first + n3);
    mm_item_counts<<<(unsigned)(nc * nc / 4), 256, 0, st>>>(s.start, lg, mm_zspan(nc), s.cnt, part);
    CT2_LAUNCH_CHECK();
    size_t tmp = 0;
    CT2_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, s.cnt, first, n3, st));
    CT2_TRY(ensure_scratch(&s.scan_tmp, &s.scan_tmp_bytes, std::max<size_t>(tmp, 256), "item scan"));
    CT2_HIP(hipcub::DeviceScan::ExclusiveSum(s.scan_tmp, tmp, s.cnt, first, n3, st));
    mm_items<<<(unsigned)((n3 + 255) / 256), 256, 0, st>>>(s.start, s.cnt, part, first, n3, s.items, nitems);
    CT2_LAUNCH_CHECK();
    // far field
    mm_p2m<<<(unsigned)(n3 / MM_P2M_CELLS), 256, 0, st>>>(s.Ps, s.start, lg, s.P, s.K, (size_t)n3, s.Zm);
    CT2_LAUNCH_CHECK();
    CT2_TRY(fft3d_batch(s.Zm, nc, 1, false, s.nz));
#define CT2_MM_MG2L(PMAX, WAVES) \
    mm_mg2l<PMAX, WAVES><<<(unsigned)std::min(n3 / MM_QB, 256 * (16 / WAVES)), 64 * WAVES, 0, st>>>(s.Zm, s.Dt32, s.sched, nc, s.K, s.nz, s.Zl)
    if (s.P <= 4)
        CT2_MM_MG2L(4, 4);
    else if (s.P <= 6)
        CT2_MM_MG2L(6, 8);
    else
        CT2_MM_MG2L(MM_PMAX, 16);
#undef CT2_MM_MG2L
    CT2_LAUNCH_CHECK();
    CT2_TRY(fft3d_batch(s.Zl, nc, -1, false, s.nz));
    // L2P into the multipole grids, which the transforms are done with, where they hold every particle
    float4* far = (float4*)s.Zm;
    if (sizeof(float4) * (size_t)n > s.Z_bytes) {
        CT2_TRY(ensure_scratch((void**)&s.far, &s.far_bytes, sizeof(float4) * (size_t)n, "far field"));
        far = s.far;
    }
    switch (s.P) {
#define CT2_MM_L2P(P) \
    case P: mm_l2p<P><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(s.Ps, s.Zl, (int)n, lg, far); break;
        CT2_MM_L2P(1) CT2_MM_L2P(2) CT2_MM_L2P(3) CT2_MM_L2P(4) CT2_MM_L2P(5) CT2_MM_L2P(6) CT2_MM_L2P(7)
        default: mm_l2p<MM_PMAX><<<(unsigned)((n + 255) / 256), 256, 0, st>>>(s.Ps, s.Zl, (int)n, lg, far);
#undef CT2_MM_L2P
    }
    CT2_LAUNCH_CHECK();
    // near pairs
    const double two32 = 4294967296.0, h = c.opts.hsoft, hu = h * two32, gm = c.opts.GM;
    NearK kc;
    kc.eps2u = (float)(hu * hu);
    kc.h2u = kc.eps2u;
    kc.hinvu = (float)(1.0 / hu);
    kc.hinv3u = (float)(1.0 / (hu * hu * hu));
    const double fnear = gm * two32 * two32, pnear = gm * two32;
    const double ffar = gm * (double)nc * nc, pfar = gm * (double)nc;
    // a wave per work item (max_items bounds the count that the device computes; waves past it exit at once), as
    // far as a launch takes them: the waves of 2^31 threads go on with the rest
    const unsigned grid = (unsigned)std::min<size_t>((max_items + MM_WAVES - 1) / MM_WAVES + 7, (1u << 31) / (64 * MM_WAVES)) & ~7u;
    const bool plummer = c.opts.kernel == CT2_KERNEL_PLUMMER, exact = nc < 16;
#define CT2_MM_NEAR(KER, EX)                                                                                        \
    mm_near<KER, EX><<<grid, 64 * MM_WAVES, 0, st>>>(s.Ps, s.start, s.items, nitems, (const float*)far, lg, s.ncols, \
                                                     kc, fnear, pnear, ffar, pfar, c.fx, c.fy, c.fz, c.pot)
    if (plummer && exact)
        CT2_MM_NEAR(CT2_KERNEL_PLUMMER, true);
    else if (plummer)
        CT2_MM_NEAR(CT2_KERNEL_PLUMMER, false);
    else if (exact)
        CT2_MM_NEAR(CT2_KERNEL_CT2, true);
    else
        CT2_MM_NEAR(CT2_KERNEL_CT2, false);
#undef CT2_MM_NEAR
    CT2_LAUNCH_CHECK();
    c.forces_valid = true;
    return CT2_OK;
}

}  // namespace

void release_mm() {
    MMState& s = g_mm;
    for (void* p : {(void*)s.Dt, (void*)s.Dt32, (void*)s.Zm, (void*)s.Zl, (void*)s.other, s.sort_tmp, (void*)s.Ps, (void*)s.start,
                    (void*)s.items, (void*)s.cnt, s.scan_tmp, (void*)s.tabz, (void*)s.sched, (void*)s.far})
        dev_free(p);
    s = MMState();
}

}  // namespace ct2

using namespace ct2;

extern "C" int ct2_mm_init(int nc, int order) {
    CT2_TRY(require_init());
    if (!is_pow2(nc) || nc < 8 || nc > 256) return set_error(CT2_ERR_INVALID, "cell grid %d: a power of two in [8, 256]", nc);
    if (order < 1 || order > MM_PMAX) return set_error(CT2_ERR_INVALID, "expansion order %d outside [1, %d]", order, MM_PMAX);
    MMIndex I;
    I.init(order);
    const size_t n3 = (size_t)nc * nc * nc;
    const size_t dt_bytes = sizeof(double) * n3 * I.K;
    if (dt_bytes > ((size_t)8 << 30))
        return set_error(CT2_ERR_INVALID, "the derivative table of order %d on %d^3 cells (%zu bytes) exceeds 8 GiB", order,
                         nc, dt_bytes);
    Context& c = ctx();
    MMState& s = g_mm;
    hipStream_t st = c.stream;
    s.nc = 0;  // unusable until the table is complete
    const int nz = (I.K + 1) / 2;
    // column order: the components of one (a, b) in a row, by z exponent
    int col[MM_PMAX + 1][MM_PMAX + 1], row[MM_KMAX] = {}, rows = 0;
    for (int e = 0; e <= order; ++e)
        for (int a = e; a >= 0; --a) {
            col[a][e - a] = rows;
            for (int z = 0; z <= order - e; ++z) row[I.id[a][e - a][z]] = rows++;
        }
    // the MG2L outputs: pairs of z exponents (kz, kz + 1), with a run for every
    // (lx, ly), then the highest exponents left over (degree P) two by two; a
    // list per wave, each output to the shortest list, the longest first
    struct Output {
        uint32_t head;
        std::vector<uint32_t> runs;
        int cost;
    };
    std::vector<Output> outs;
    std::vector<int> single;  // grids in LocalGrids' order
    for (int e = 0; e <= order; ++e)
        for (int a = e; a >= 0; --a) {
            const int b = e - a;
            for (int kz = 0; kz + 1 <= order - e; kz += 2) {
                const int r = order - e - kz;
                Output o{(uint32_t)r | (uint32_t)outs.size() << 4 | (uint32_t)(e + kz) << 11, {}, 40};
                for (int le = 0, n = 0; le <= r; ++le)
                    for (int la = le; la >= 0; --la, ++n) {
                        const uint32_t w = mg2l_rows(col[la][le - la], col[a + la][b + le - la] + kz);
                        if (n & 1)
                            o.runs.back() |= w << 16;
                        else
                            o.runs.push_back(w);
                        o.cost += 10 * (r - le) + 15;  // about its share of the time
                    }
                outs.push_back(o);
            }
            if ((order - e) % 2 == 0) single.push_back(I.id[a][b][order - e]);
        }
    for (size_t k = 0; k < single.size(); k += 2) {
        const bool both = k + 1 < single.size();
        outs.push_back({(uint32_t)outs.size() << 4 | (uint32_t)order << 11,
                        {mg2l_rows(row[single[k]], both ? row[single[k + 1]] : (int)MG2L_NONE)}, 60});
    }
    if ((int)outs.size() != nz) return set_error(CT2_ERR_STATE, "%zu MG2L outputs for %d grids", outs.size(), nz);
    const int waves = order <= 4 ? 4 : order <= 6 ? 8 : 16;
    std::stable_sort(outs.begin(), outs.end(), [](const Output& x, const Output& y) { return x.cost > y.cost; });
    std::vector<uint32_t> sched((size_t)waves * MG2L_LIST, 0u);
    std::vector<int> load(waves, 0), count(waves, 0);
    std::vector<size_t> words(waves, 0);
    for (const Output& o : outs) {
        const int w = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        if (count[w] == MG2L_STEPS || words[w] + o.runs.size() > MG2L_STEPS)
            return set_error(CT2_ERR_STATE, "MG2L list longer than %d words", MG2L_STEPS);
        uint32_t* list = sched.data() + (size_t)w * MG2L_LIST;
        list[count[w]++] = o.head;
        std::copy(o.runs.begin(), o.runs.end(), list + MG2L_STEPS + words[w]);
        words[w] += o.runs.size();
        load[w] += o.cost;
    }
    const auto degree = [&](int c) { return (uint32_t)(I.e[c][0] + I.e[c][1] + I.e[c][2]); };
    for (int w = 0; w < waves; ++w) {
        uint32_t* stage = sched.data() + (size_t)w * MG2L_LIST + 2 * MG2L_STEPS;
        for (int i = 0, j = w; j < nz; ++i, j += waves) {
            stage[i] = (uint32_t)row[2 * j] | degree(2 * j) << 16;
            if (2 * j + 1 < I.K) stage[i] |= (uint32_t)row[2 * j + 1] << 8 | degree(2 * j + 1) << 24;
        }
        for (int i = 16, c = w; c < I.K; ++i, c += waves) stage[i] = (uint32_t)row[c] | (degree(c) & 2u) << 30;
        stage[MG2L_STEPS - 1] = (uint32_t)count[w];
    }
    int ce[MM_KMAX][3] = {};
    float cf[MM_KMAX] = {};
    for (int k = 0; k < I.K; ++k) {
        for (int q = 0; q < 3; ++q) ce[k][q] = I.e[k][q];
        cf[k] = (float)(1.0 / I.fact[k]);
    }
    // the near set |offset|^2 <= 10 as columns: (dx, dy) with dz in [-w, w]
    int cn[MM_COLS_MAX][3] = {};
    int ncols = 0;
    for (int a = -3; a <= 3; ++a)
        for (int b = -3; b <= 3; ++b)
            if (a * a + b * b <= MM_NEAR2) {
                int hw = 0;
                while (a * a + b * b + (hw + 1) * (hw + 1) <= MM_NEAR2) ++hw;
                cn[ncols][0] = a;
                cn[ncols][1] = b;
                cn[ncols][2] = hw;
                ++ncols;
            }
    CT2_HIP(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_e), ce, sizeof ce, 0, hipMemcpyHostToDevice, st));
    CT2_HIP(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_ifact), cf, sizeof cf, 0, hipMemcpyHostToDevice, st));
    CT2_HIP(hipMemcpyToSymbolAsync(HIP_SYMBOL(c_cols), cn, sizeof cn, 0, hipMemcpyHostToDevice, st));
    // buffers
    CT2_TRY(ensure_scratch((void**)&s.sched, &s.sched_bytes, sizeof(uint32_t) * sched.size(), "MG2L lists"));
    CT2_HIP(hipMemcpyAsync(s.sched, sched.data(), sizeof(uint32_t) * sched.size(), hipMemcpyHostToDevice, st));
    CT2_TRY(ensure_scratch((void**)&s.Dt, &s.Dt_bytes, dt_bytes, "multipole-mesh derivative table"));
    CT2_TRY(ensure_scratch((void**)&s.Dt32, &s.Dt32_bytes, dt_bytes / 2, "multipole-mesh FP32 table"));
    CT2_TRY(ensure_scratch((void**)&s.Zm, &s.Z_bytes, sizeof(float2) * n3 * nz, "multipole grids"));
    if (s.Zl) dev_free(s.Zl);
    s.Zl = nullptr;
    CT2_TRY(dev_alloc((void**)&s.Zl, sizeof(float2) * n3 * nz, "local-expansion grids"));
    CT2_TRY(ensure_scratch((void**)&s.tabz, &s.tabz_bytes, sizeof(double2) * n3, "table transform"));
    // the table: short-range samples on the host, one FP64 transform per component
    std::vector<double> S;
    short_samples(I, nc, S);
    std::vector<double> z(2 * n3);
    for (int k = 0; k < I.K; ++k) {
        for (size_t q = 0; q < n3; ++q) {
            z[2 * q] = S[(size_t)k * n3 + q];
            z[2 * q + 1] = 0.0;
        }
        CT2_HIP(hipMemcpyAsync(s.tabz, z.data(), sizeof(double2) * n3, hipMemcpyHostToDevice, st));
        CT2_TRY(fft3d(s.tabz, nc, 1, true));
        mm_table_finish<<<(unsigned)((n3 + 255) / 256), 256, 0, st>>>(s.tabz, nc, I.e[k][0], I.e[k][1], I.e[k][2],
                                                                       s.Dt + (size_t)k * n3, s.Dt32 + (size_t)k * n3);
        CT2_LAUNCH_CHECK();
        CT2_HIP(hipStreamSynchronize(st));  // z is refilled next
    }
    s.nc = nc;
    s.P = order;
    s.K = I.K;
    s.nz = nz;
    s.ncols = ncols;
    return CT2_OK;
}

extern "C" int ct2_mm_cells_for(size_t n, int particles_per_cell, int* nc) {
    if (!nc) return set_error(CT2_ERR_INVALID, "null output");
    if (particles_per_cell < 1) return set_error(CT2_ERR_INVALID, "particles per cell %d < 1", particles_per_cell);
    size_t g = 8;
    while (g < 256 && (2 * g) * (2 * g) * (2 * g) * (size_t)particles_per_cell <= n) g *= 2;
    *nc = (int)g;
    return CT2_OK;
}

extern "C" int ct2_mm_forces(void) {
    CT2_TRY(mm_require());
    CT2_TRY(mm_forces());
    ctx().last_path = CT2_PATH_MM;
    return CT2_OK;
}

extern "C" int ct2_kick_mm(const ct2_kick_params* p, unsigned flags, int* max_rung) {
    CT2_TRY(mm_require());
    CT2_TRY(check_kick_params(p));
    if (flags & ~(unsigned)CT2_KICK_STORE) return set_error(CT2_ERR_INVALID, "unknown flags 0x%x", flags);
    CT2_TRY(mm_forces());
    ctx().last_path = CT2_PATH_MM;
    return run_epilogue(p, max_rung);
}

extern "C" int ct2_mm_table_download(double* host) {
    CT2_TRY(require_init());
    if (!g_mm.nc) return set_error(CT2_ERR_STATE, "ct2_mm_init has not been called");
    if (!host) return set_error(CT2_ERR_INVALID, "null output");
    Context& c = ctx();
    CT2_HIP(hipMemcpyAsync(host, g_mm.Dt, sizeof(double) * (size_t)g_mm.K * g_mm.nc * g_mm.nc * g_mm.nc,
                           hipMemcpyDeviceToHost, c.stream));
    CT2_HIP(hipStreamSynchronize(c.stream));
    return CT2_OK;
}
