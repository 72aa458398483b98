// fft.hip -- 3-D FFTs for gfx950, complex and real, in passes over HBM.
//
// Each pass is one kernel that moves a batch of lines through a Stockham
// autosort radix-8 (mixed 2/4/8) transform (fft_stages.h): the first stage
// reads HBM straight into registers, the middle stages exchange through LDS,
// the last stage writes HBM from registers.  Natural order in and out, so no
// bit-reversal pass exists (the reference's scramble() step is absorbed).
//   z pass (contiguous lines): `fft_rows`, P lanes per line, LDS rows
//     padded by one element in eight to keep LDS accesses conflict-free;
//   y and x passes (stride n and n^2): `fft_cols`, C adjacent columns per
//     workgroup so that every HBM access is a C*sizeof(complex) segment
//     (128 bytes for FP32 at C=16).
// Cubes whose planes fit in LDS take the z and y passes, and the smallest all
// three, in one kernel (`fft_block`).  Real fields go through half spectra
// (`rfft_rows`, `half_cols`, `irfft_rows`): half the bytes of a complex
// transform per pass.
// Twiddles W_N^m are tabulated once per size on the host in FP64 libm
// (twiddles.cpp:6-54 computes the same table) and rounded to the working
// precision; each workgroup copies the table into LDS.
#include <cmath>
#include <map>
#include <utility>
#include <vector>

#include "fft_stages.h"
#include "internal.h"

namespace ct2 {
namespace {

template <typename T, int N, int NC = N>
constexpr int col_lanes() {
    return Cfg<T, N, NC>::P * Cfg<T, N, NC>::COLS;
}
template <typename T, int N>
constexpr int row_lanes() {
    return Cfg<T, N>::P * Cfg<T, N>::ROWS;
}

// z pass: lines of N contiguous elements; workgroup = ROWS lines; cube
// blockIdx.y of a batch.
template <typename T, int N, int DIR>
__global__ __launch_bounds__((row_lanes<T, N>())) void fft_rows(typename V2<T>::t* __restrict__ data,
                                                               const typename V2<T>::t* __restrict__ twg) {
    using T2 = typename V2<T>::t;
    using CF = Cfg<T, N>;
    __shared__ T2 sm[CF::ROWS * CF::ROWLEN];
    __shared__ T2 tw[N];
    load_twiddles<N>(tw, twg, row_lanes<T, N>());
    const int p = threadIdx.x % CF::P;
    const int c = threadIdx.x / CF::P;
    data += (size_t)blockIdx.y * ((size_t)N * N * N) + ((size_t)blockIdx.x * CF::ROWS + c) * N;
    run_stages<T, N, DIR, false, false>([&](int i, int) { return data[i]; }, [&](int i, int, T2 v) { data[i] = v; },
                                        [&](int i) { return c * CF::ROWLEN + i + (i >> 3); }, sm, tw, p);
}

// y / x pass: COLS adjacent columns (unit stride) of lines with stride
// stride_i; block b covers columns (b % inner)*COLS.. of slab b / inner, or
// with slab_fast columns (b / N)*COLS.. of slab b % N.
template <typename T, int N, int DIR>
__global__ __launch_bounds__((col_lanes<T, N>())) void fft_cols(typename V2<T>::t* __restrict__ data,
                                                               const typename V2<T>::t* __restrict__ twg,
                                                               long stride_i, long stride_outer, int inner,
                                                               bool slab_fast) {
    using T2 = typename V2<T>::t;
    using CF = Cfg<T, N>;
    __shared__ T2 sm[N * CF::COLS];
    __shared__ T2 tw[N];
    load_twiddles<N>(tw, twg, col_lanes<T, N>());
    const int c = threadIdx.x % CF::COLS;
    const int p = threadIdx.x / CF::COLS;
    const unsigned b = xcd_contiguous(blockIdx.x, gridDim.x);
    // y pass: the column groups of one slab side by side; x pass (lines at
    // stride n^2): slabs side by side, so that the workgroups in flight read
    // many slabs (512^3 forward transform 1.259 -> 1.242-1.257 ms; slab-fast
    // order in the y pass measured 1.311 ms)
    const long outer = slab_fast ? b % N : b / inner, in = slab_fast ? b / N : b % inner;
    data += (size_t)blockIdx.y * ((size_t)N * N * N) + outer * stride_outer + in * CF::COLS + c;
    run_stages<T, N, DIR, false, false>([&](int i, int) { return data[(long)i * stride_i]; },
                                        [&](int i, int, T2 v) { data[(long)i * stride_i] = v; },
                                        [&](int i) { return i * CF::COLS + c; }, sm, tw, p);
}

// The z and y passes of one x plane, or all three of a cube (N <= 16), in LDS:
// one read and one write of HBM for the axes it covers, and a launch fewer
// (small cubes are bound by launches of ~3 us).  A phase gives each line P
// lanes; the lanes of a column phase run over z.  Taken wherever a plane fits
// (FP32 N <= 128, FP64 N <= 64).  us per transform, one pass per axis -> this:
// FP32 8^3 8.0 -> 2.9, 16^3 8.1 -> 4.5, 32^3 8.0 -> 5.6, 64^3 10.3 -> 8.3, 128^3
// 34 -> 28 (128 workgroups, one per CU); FP64 8^3 7.7 -> 2.8, 64^3 14.1 -> 11.3;
// 83 FP32 cubes of 64^3 as the multipole mesh transforms them: 158 -> 107.
template <typename T, int N, bool CUBE>
struct Block {
    using CF = Cfg<T, N>;
    static constexpr int LINES = CUBE ? N * N : N;  // per phase
    static constexpr int ELEMS = LINES * CF::ROWLEN;
    static constexpr int TH = LINES * CF::P < 1024 ? LINES * CF::P : 1024;
    static constexpr int LPI = TH / CF::P;  // lines at a time
    static constexpr bool ok = (ELEMS + N) * (int)sizeof(typename V2<T>::t) <= 160 * 1024;
};

template <typename T, int N, int DIR, bool CUBE>
__global__ __launch_bounds__((Block<T, N, CUBE>::TH)) void fft_block(typename V2<T>::t* __restrict__ data,
                                                                    const typename V2<T>::t* __restrict__ twg) {
    using T2 = typename V2<T>::t;
    using CF = Cfg<T, N>;
    using BK = Block<T, N, CUBE>;
    __shared__ T2 sm[BK::ELEMS];
    __shared__ T2 tw[N];
    load_twiddles<N>(tw, twg, BK::TH);
    data += (size_t)blockIdx.x * BK::LINES * N;  // plane (or cube) blockIdx.x of the batch
    for (int l0 = 0; l0 < BK::LINES; l0 += BK::LPI) {  // z lines: line l holds (x, y)
        const int p = threadIdx.x % CF::P, l = l0 + threadIdx.x / CF::P;
        auto ix = [&](int i) { return l * CF::ROWLEN + i + (i >> 3); };
        run_stages<T, N, DIR, false, true>([&](int i, int) { return data[l * N + i]; },
                                           [&](int i, int, T2 v) { sm[ix(i)] = v; }, ix, sm, tw, p);
    }
    __syncthreads();
    const int p = threadIdx.x / BK::LPI;
    for (int l0 = 0; l0 < BK::LINES; l0 += BK::LPI) {  // y lines: line l holds (x, z)
        const int l = l0 + threadIdx.x % BK::LPI, z = l % N, x = l / N;
        auto ix = [&](int i) { return (x * N + i) * CF::ROWLEN + z + (z >> 3); };
        auto ld = [&](int i, int) { return sm[ix(i)]; };
        if constexpr (CUBE)
            run_stages<T, N, DIR, true, true>(ld, [&](int i, int, T2 v) { sm[ix(i)] = v; }, ix, sm, tw, p);
        else
            run_stages<T, N, DIR, true, false>(ld, [&](int i, int, T2 v) { data[i * N + z] = v; }, ix, sm, tw, p);
    }
    if constexpr (CUBE) {
        __syncthreads();
        for (int l0 = 0; l0 < BK::LINES; l0 += BK::LPI) {  // x lines: line l holds (y, z)
            const int l = l0 + threadIdx.x % BK::LPI, z = l % N, y = l / N;
            auto ix = [&](int i) { return (i * N + y) * CF::ROWLEN + z + (z >> 3); };
            run_stages<T, N, DIR, true, false>([&](int i, int) { return sm[ix(i)]; },
                                               [&](int i, int, T2 v) { data[(i * N + y) * N + z] = v; }, ix, sm, tw, p);
        }
    }
}

// ------------------------------------------------------------ real fields
//
// Half spectrum of an N^3 real field while it is transformed: the columns
// kz < N/2 as half[x][y][kz] (aligned rows of N/2) and kz = N/2 as
// nyq[y][x], so that both stay whole lines.

// A real field as the z pass reads it: samples 2i and 2i + 1 of a row.
struct RealField {
    const double* f;
    template <typename T2>
    __device__ __forceinline__ T2 pair(long at) const {
        return T2{f[at], f[at + 1]};
    }
};

struct DensityField {  // uint64 fixed point, 2^-32 units
    const unsigned long long* w;
    template <typename T2>
    __device__ __forceinline__ T2 pair(long at) const {
        using T = decltype(T2{}.x);
        const ulonglong2 v = *(const ulonglong2*)(w + at);
        return T2{(T)((double)v.x * 0x1p-32), (T)((double)v.y * 0x1p-32)};
    }
};

// Forward z pass of real rows: Z, the transform of the N/2 pairs
// (x_2i, x_2i+1), then F_k = (Z_k + conj Z_{N/2-k}) / 2 - i W_N^k (Z_k -
// conj Z_{N/2-k}) / 2.
template <typename T, int N, typename SRC>
__global__ __launch_bounds__((row_lanes<T, N / 2>())) void rfft_rows(SRC src, typename V2<T>::t* __restrict__ half,
                                                                    typename V2<T>::t* __restrict__ nyq,
                                                                    const typename V2<T>::t* __restrict__ twg) {
    using T2 = typename V2<T>::t;
    constexpr int H = N / 2;
    using CF = Cfg<T, H>;
    __shared__ T2 sm[CF::ROWS * CF::ROWLEN];
    __shared__ T2 tw[H];
    load_twiddles<H, 2>(tw, twg, row_lanes<T, H>());
    const int p = threadIdx.x % CF::P, c = threadIdx.x / CF::P;
    const long row0 = (long)blockIdx.x * CF::ROWS;
    auto ix = [&](int i) { return c * CF::ROWLEN + i + (i >> 3); };
    run_stages<T, H, 1, false, true>([&](int i, int) { return src.template pair<T2>((row0 + c) * N + 2 * i); },
                                     [&](int i, int, T2 v) { sm[ix(i)] = v; }, ix, sm, tw, p);
    __syncthreads();
    for (int e = threadIdx.x; e < CF::ROWS * H; e += row_lanes<T, H>()) {
        const int k = e % H, k2 = (H - k) % H;
        const T2* z = sm + e / H * CF::ROWLEN;
        const T2 a = z[k + (k >> 3)], b = z[k2 + (k2 >> 3)], w = twg[k];
        const long row = row0 + e / H;
        const T2 o = cmul(T2{a.x - b.x, a.y + b.y}, w);  // W (Z_k - conj Z_{N/2-k})
        half[row * H + k] = T2{(T)0.5 * (a.x + b.x + o.y), (T)0.5 * (a.y - b.y - o.x)};
        if (k == 0) nyq[(row % N) * N + row / N] = T2{a.x - a.y, (T)0};
    }
}

// Forward z and y passes of a plane of a real field in LDS, to its half spectrum:
// rfft_rows and half_cols in one kernel, a launch fewer.  Row y of the plane lies
// at sm[y ROW], kz = N/2 last in it.  FP64 round trips of two fields with it /
// without: 8^3 40 / 48 us, 64^3 57.5 / 59.2; a PM force on 128^3 loses 15 us to it.
template <typename T, int N>
struct HalfBlock {
    static constexpr int H = N / 2, P = Cfg<T, H>::P, PC = Cfg<T, N>::P;  // lanes per row / column
    static constexpr int ROW = Cfg<T, H>::ROWLEN + 1;
    static constexpr int TH = N * P < 1024 ? N * P : 1024;
    // at 128 a workgroup per plane leaves half of the chip idle
    static constexpr bool ok = N <= 64;
};

template <typename T, int N, typename SRC>
__global__ __launch_bounds__((HalfBlock<T, N>::TH)) void rfft_block(SRC src, typename V2<T>::t* __restrict__ half,
                                                                   typename V2<T>::t* __restrict__ nyq,
                                                                   const typename V2<T>::t* __restrict__ twg) {
    using T2 = typename V2<T>::t;
    using BK = HalfBlock<T, N>;
    constexpr int H = N / 2, ROW = BK::ROW, TH = BK::TH;
    __shared__ T2 sm[N * ROW];
    __shared__ T2 tw[N], twh[H];
    load_twiddles<N>(tw, twg, TH);
    load_twiddles<H, 2>(twh, twg, TH);
    const long x = blockIdx.x;
    for (int l0 = 0; l0 < N; l0 += TH / BK::P) {
        const int p = threadIdx.x % BK::P, y = l0 + threadIdx.x / BK::P;
        auto ix = [&](int i) { return y * ROW + i + (i >> 3); };
        run_stages<T, H, 1, false, true>([&](int i, int) { return src.template pair<T2>((x * N + y) * N + 2 * i); },
                                         [&](int i, int, T2 v) { sm[ix(i)] = v; }, ix, sm, twh, p);
    }
    __syncthreads();
    // Z to F as in rfft_rows, k and N/2 - k by one lane
    for (int e = threadIdx.x; e < N * (H / 2 + 1); e += TH) {
        const int k = e % (H / 2 + 1), k2 = (H - k) % H;
        T2* z = sm + e / (H / 2 + 1) * ROW;
        const T2 a = z[k + (k >> 3)], b = z[k2 + (k2 >> 3)];
        auto f = [&](T2 u, T2 v, T2 w) {
            const T2 o = cmul(T2{u.x - v.x, u.y + v.y}, w);
            return T2{(T)0.5 * (u.x + v.x + o.y), (T)0.5 * (u.y - v.y - o.x)};
        };
        z[k + (k >> 3)] = f(a, b, tw[k]);
        if (k == 0)
            z[H + (H >> 3)] = T2{a.x - a.y, (T)0};
        else if (k2 != k)
            z[k2 + (k2 >> 3)] = f(b, a, tw[k2]);
    }
    __syncthreads();
    for (int l0 = 0; l0 <= H; l0 += TH / BK::PC) {
        // lanes past the last column repeat it, and store nothing
        const int l = l0 + threadIdx.x % (TH / BK::PC), z = min(l, H), p = threadIdx.x / (TH / BK::PC);
        auto ix = [&](int i) { return i * ROW + z + (z >> 3); };
        run_stages<T, N, 1, true, false>([&](int i, int) { return sm[ix(i)]; },
                                         [&](int i, int, T2 v) {
                                             if (l < H)
                                                 half[(x * N + i) * H + z] = v;
                                             else if (l == H)
                                                 nyq[(long)i * N + x] = v;
                                         },
                                         ix, sm, tw, p);
    }
}

// Inverse z pass to real rows (the real part of the complex transform, so the
// imaginary parts of kz = 0 and N/2 do not enter).
template <typename T, int N>
__global__ __launch_bounds__((row_lanes<T, N / 2>())) void irfft_rows(const typename V2<T>::t* __restrict__ half,
                                                                     const typename V2<T>::t* __restrict__ nyq,
                                                                     T* __restrict__ out,
                                                                     const typename V2<T>::t* __restrict__ twg) {
    using T2 = typename V2<T>::t;
    constexpr int H = N / 2;
    using CF = Cfg<T, H>;
    __shared__ T2 sm[CF::ROWS * CF::ROWLEN];
    __shared__ T2 tw[H];
    load_twiddles<H, 2>(tw, twg, row_lanes<T, H>());
    const int p = threadIdx.x % CF::P, c = threadIdx.x / CF::P;
    const long row = (long)blockIdx.x * CF::ROWS + c;
    half += row * H;
    run_stages<T, H, -1, false, false>(
        [&](int k, int) {
            if (k == 0) {
                const T a = half[0].x, b = nyq[(row % N) * N + row / N].x;
                return T2{a + b, a - b};
            }
            const T2 a = half[k], b = half[H - k], w = twg[k];
            // (X_k + conj X_{H-k}) + i W^-k (X_k - conj X_{H-k})
            const T2 d = T2{a.x - b.x, a.y + b.y};
            const T2 o = T2{d.x * w.x + d.y * w.y, d.y * w.x - d.x * w.y};
            return T2{a.x + b.x - o.y, a.y - b.y + o.x};
        },
        [&](int i, int, T2 v) {
            out[row * N + 2 * i] = v.x;
            out[row * N + 2 * i + 1] = v.y;
        },
        [&](int i) { return c * CF::ROWLEN + i + (i >> 3); }, sm, tw, p);
}

// y / x pass over the half spectrum: blocks below N (N/2) / COLS take COLS
// columns of half, in fft_cols' order, the others COLS columns of nyq.  IO:
// 0 in place; the x pass may read (1) or write (2) the planar spectrum
// planar[(x N + y) (N/2 + 1) + kz] = Re, + N^2 (N/2 + 1) = Im instead.
template <typename T, int N, int DIR, bool XPASS, int IO>
__global__ __launch_bounds__((col_lanes<T, N, N / 2>())) void half_cols(typename V2<T>::t* __restrict__ half,
                                                                       typename V2<T>::t* __restrict__ nyq,
                                                                       const typename V2<T>::t* __restrict__ twg,
                                                                       const T* __restrict__ pin, T* __restrict__ pout) {
    static_assert(IO == 0 || XPASS, "the planar spectrum is the x pass's");
    using T2 = typename V2<T>::t;
    constexpr int H = N / 2, COLS = Cfg<T, N, H>::COLS, LANES = col_lanes<T, N, H>();
    constexpr unsigned MAIN = (unsigned)N * (H / COLS);
    constexpr long IMAG = (long)N * N * (H + 1);
    __shared__ T2 sm[N * COLS];
    __shared__ T2 tw[N];
    load_twiddles<N>(tw, twg, LANES);
    const int c = threadIdx.x % COLS, p = threadIdx.x / COLS;
    T2* d;
    long stride, q;  // q: the column's place in the planar spectrum's first x plane
    if (blockIdx.x < MAIN) {
        const unsigned b = xcd_contiguous(blockIdx.x, MAIN);
        const unsigned slab = XPASS ? b % N : b / (H / COLS), in = XPASS ? b / N : b % (H / COLS);
        const int k = in * COLS + c;
        d = half + (XPASS ? (long)slab * H : (long)slab * N * H) + k;
        stride = XPASS ? (long)N * H : H;
        q = (long)slab * (H + 1) + k;
    } else {
        const int j = (blockIdx.x - MAIN) * COLS + c;
        d = nyq + (XPASS ? (long)j * N : j);
        stride = XPASS ? 1 : N;
        q = (long)j * (H + 1) + H;
    }
    run_stages<T, N, DIR, false, false>(
        [&](int i, int) {
            const long e = q + (long)i * N * (H + 1);
            if constexpr (IO == 1) return T2{pin[e], pin[e + IMAG]};
            return d[(long)i * stride];
        },
        [&](int i, int, T2 v) {
            const long e = q + (long)i * N * (H + 1);
            if constexpr (IO == 2) {
                pout[e] = v.x;
                pout[e + IMAG] = v.y;
            } else {
                d[(long)i * stride] = v;
            }
        },
        [&](int i) { return i * COLS + c; }, sm, tw, p);
}

// ---- twiddle tables (device, per precision and size) ----
std::map<std::pair<int, int>, void*> g_tw;  // (bytes per real, N) -> W_N^m, m < N

template <typename T>
int twiddle_table(int N, const typename V2<T>::t** out) {
    const auto key = std::make_pair((int)sizeof(T), N);
    auto it = g_tw.find(key);
    if (it == g_tw.end()) {
        std::vector<typename V2<T>::t> h(N);
        const double twopi = 2.0 * M_PI;
        for (int m = 0; m < N; ++m) {
            h[m].x = (T)std::cos(-twopi * m / N);
            h[m].y = (T)std::sin(-twopi * m / N);
        }
        void* d = nullptr;
        CT2_TRY(dev_alloc(&d, sizeof(h[0]) * N, "FFT twiddles"));
        CT2_HIP(hipMemcpy(d, h.data(), sizeof(h[0]) * N, hipMemcpyHostToDevice));
        it = g_tw.emplace(key, d).first;
    }
    *out = (const typename V2<T>::t*)it->second;
    return CT2_OK;
}

// z and y passes of batch cubes of N^3, one after the other (each axis is
// independent, so they may also follow the x pass)
template <typename T, int N, int DIR>
int fft_zy(typename V2<T>::t* d, const typename V2<T>::t* tw, hipStream_t st, int batch) {
    if constexpr (Block<T, N, false>::ok) {
        fft_block<T, N, DIR, false><<<(unsigned)(N * batch), Block<T, N, false>::TH, 0, st>>>(d, tw);
        CT2_LAUNCH_CHECK();
    } else {
        using CF = Cfg<T, N>;
        constexpr int inner = N / CF::COLS;
        // Cubes of several times the Infinity Cache (256 MB) go in groups of planes
        // that it holds, the z pass of a group and then its y pass, which finds the
        // group there instead of in HBM.  us per transform, the passes whole /
        // groups of 64 / 128 / 192 MB: 512^3 FP32 1,223 / 1,237 / 1,167 / 1,173, FP64
        // 2,568 / 2,567 / 2,401 / 2,360, 1024^3 FP32 15,283 / - / 14,700 / 14,435;
        // 256^3 FP64 (268 MB) 239 / 258 / 247 / -: there the launches cost more.
        // (Pairing the z with the x pass, in groups of y: 512^3 FP32 1,134 at 128 MB,
        // but FP64 2,876.)
        constexpr size_t PLANE = sizeof(typename V2<T>::t) * N * N, GROUP = 192u << 20;
        const int planes = PLANE * N >= (1u << 30) ? (int)(GROUP / PLANE) : N * batch;
        for (long q = 0; q < (long)N * batch; q += planes) {
            const unsigned np = (unsigned)std::min<long>(planes, (long)N * batch - q);
            fft_rows<T, N, DIR><<<np * N / CF::ROWS, row_lanes<T, N>(), 0, st>>>(d + q * N * N, tw);
            CT2_LAUNCH_CHECK();
            // y: columns z, slabs x
            fft_cols<T, N, DIR><<<np * inner, col_lanes<T, N>(), 0, st>>>(d + q * N * N, tw, N, (long)N * N, inner, false);
            CT2_LAUNCH_CHECK();
        }
    }
    return CT2_OK;
}

// batch cubes of N^3 one after the other
template <typename T, int N, int DIR>
int fft3d_launch(typename V2<T>::t* d, hipStream_t st, int batch) {
    const typename V2<T>::t* tw = nullptr;
    CT2_TRY(twiddle_table<T>(N, &tw));
    if constexpr (N <= 16) {
        fft_block<T, N, DIR, true><<<(unsigned)batch, Block<T, N, true>::TH, 0, st>>>(d, tw);
        CT2_LAUNCH_CHECK();
    } else {
        CT2_TRY((fft_zy<T, N, DIR>(d, tw, st, batch)));
        // x: columns z, slabs y
        constexpr int inner = N / Cfg<T, N>::COLS;
        fft_cols<T, N, DIR><<<dim3((unsigned)(N * inner), batch), col_lanes<T, N>(), 0, st>>>(d, tw, (long)N * N, N,
                                                                                              inner, true);
        CT2_LAUNCH_CHECK();
    }
    return CT2_OK;
}

#define CT2_FFT_SIZES(CASE) CASE(8) CASE(16) CASE(32) CASE(64) CASE(128) CASE(256) CASE(512)

template <typename T, int DIR>
int fft3d_dispatch(void* data, int n, hipStream_t st, int batch = 1) {
    using T2 = typename V2<T>::t;
    T2* d = (T2*)data;
    switch (n) {
#define CT2_CASE(N) \
    case N: return fft3d_launch<T, N, DIR>(d, st, batch);
        CT2_FFT_SIZES(CT2_CASE)
#undef CT2_CASE
        case 1024:
            if constexpr (sizeof(T) == 4) return fft3d_launch<T, 1024, DIR>(d, st, batch);
            [[fallthrough]];
        default: return set_error(CT2_ERR_INVALID, "unsupported FFT size %d", n);
    }
}

template <typename T, int N, typename SRC>
int rfft_zy_launch(SRC src, typename V2<T>::t* half, hipStream_t st, const typename V2<T>::t** tw) {
    constexpr int COLS = Cfg<T, N, N / 2>::COLS;
    CT2_TRY(twiddle_table<T>(N, tw));
    typename V2<T>::t* nyq = half + (size_t)N * N * (N / 2);
    if constexpr (HalfBlock<T, N>::ok) {
        rfft_block<T, N, SRC><<<N, HalfBlock<T, N>::TH, 0, st>>>(src, half, nyq, *tw);
        CT2_LAUNCH_CHECK();
        return CT2_OK;
    }
    rfft_rows<T, N, SRC><<<N * N / Cfg<T, N / 2>::ROWS, row_lanes<T, N / 2>(), 0, st>>>(src, half, nyq, *tw);
    CT2_LAUNCH_CHECK();
    half_cols<T, N, 1, false, 0><<<N * (N / 2) / COLS + N / COLS, col_lanes<T, N, N / 2>(), 0, st>>>(half, nyq, *tw,
                                                                                                      nullptr, nullptr);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

template <int N>
int rfft3d_launch(const double* in, double* planar, double2* half, hipStream_t st) {
    constexpr int COLS = Cfg<double, N, N / 2>::COLS;
    const double2* tw = nullptr;
    CT2_TRY((rfft_zy_launch<double, N>(RealField{in}, half, st, &tw)));
    half_cols<double, N, 1, true, 2><<<N * (N / 2) / COLS + N / COLS, col_lanes<double, N, N / 2>(), 0, st>>>(
        half, half + (size_t)N * N * (N / 2), tw, nullptr, planar);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

template <int N>
int irfft3d_launch(const double* planar, double* out, double2* half, hipStream_t st) {
    constexpr int COLS = Cfg<double, N, N / 2>::COLS, BLOCKS = N * (N / 2) / COLS + N / COLS;
    constexpr int LANES = col_lanes<double, N, N / 2>();
    const double2* tw = nullptr;
    CT2_TRY(twiddle_table<double>(N, &tw));
    double2* nyq = half + (size_t)N * N * (N / 2);
    half_cols<double, N, -1, true, 1><<<BLOCKS, LANES, 0, st>>>(half, nyq, tw, planar, nullptr);
    CT2_LAUNCH_CHECK();
    half_cols<double, N, -1, false, 0><<<BLOCKS, LANES, 0, st>>>(half, nyq, tw, nullptr, nullptr);
    CT2_LAUNCH_CHECK();
    irfft_rows<double, N><<<N * N / Cfg<double, N / 2>::ROWS, row_lanes<double, N / 2>(), 0, st>>>(half, nyq, out, tw);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

}  // namespace

int fft_table_f32(int n, const float2** tw) { return twiddle_table<float>(n, tw); }

// The density W * 2^-32 (uint64 fixed point, n^3) through the z and y passes
// into its half spectrum (fft_half_elems(n) elements); the x pass is the
// caller's.
int rfft_zy_density(const unsigned long long* W, float2* half, int n) {
    CT2_TRY(require_init());
    if (!W || !half) return set_error(CT2_ERR_INVALID, "null FFT buffer");
    hipStream_t st = ctx().stream;
    const float2* tw = nullptr;
    switch (n) {
#define CT2_CASE(N) \
    case N: return rfft_zy_launch<float, N>(DensityField{W}, half, st, &tw);
        CT2_FFT_SIZES(CT2_CASE)
        CT2_CASE(1024)
#undef CT2_CASE
        default: return set_error(CT2_ERR_INVALID, "unsupported FFT size %d", n);
    }
}

// Inverse y and z passes of `batch` FP32 cubes.
int fft_inverse_yz(float2* data, int n, int batch) {
    CT2_TRY(require_init());
    if (!data) return set_error(CT2_ERR_INVALID, "null FFT buffer");
    hipStream_t st = ctx().stream;
    const float2* tw = nullptr;
    CT2_TRY(twiddle_table<float>(n, &tw));
    switch (n) {
#define CT2_CASE(N) \
    case N: return fft_zy<float, N, -1>(data, tw, st, batch);
        CT2_FFT_SIZES(CT2_CASE)
        CT2_CASE(1024)
#undef CT2_CASE
        default: return set_error(CT2_ERR_INVALID, "unsupported FFT size %d", n);
    }
}

// Real FP64 cube to the planar half spectrum, and back (unnormalised), through
// fft_half_elems(n) elements of scratch.  Three passes of 16 B per real sample
// each way, bound by HBM.  A round trip of 256^3 through the complex transform
// of the field (144 B a sample each way, with the conversions to and from
// complex as passes of their own) took 0.77 ms, now 0.34 (4.8 TB/s).
int rfft3d_f64(const double* in, double* planar, double2* half, int n) {
    hipStream_t st = ctx().stream;
    switch (n) {
#define CT2_CASE(N) \
    case N: return rfft3d_launch<N>(in, planar, half, st);
        CT2_FFT_SIZES(CT2_CASE)
#undef CT2_CASE
        default: return set_error(CT2_ERR_INVALID, "unsupported FFT size %d", n);
    }
}

int irfft3d_f64(const double* planar, double* out, double2* half, int n) {
    hipStream_t st = ctx().stream;
    switch (n) {
#define CT2_CASE(N) \
    case N: return irfft3d_launch<N>(planar, out, half, st);
        CT2_FFT_SIZES(CT2_CASE)
#undef CT2_CASE
        default: return set_error(CT2_ERR_INVALID, "unsupported FFT size %d", n);
    }
}

int fft3d_batch(void* data, int n, int dir, bool f64, int batch) {
    CT2_TRY(require_init());
    if (!data) return set_error(CT2_ERR_INVALID, "null FFT buffer");
    if (!is_pow2(n) || n < 8 || n > (f64 ? 512 : 1024))
        return set_error(CT2_ERR_INVALID, "FFT size %d is not a power of two in [8, %d]", n, f64 ? 512 : 1024);
    if (dir != 1 && dir != -1) return set_error(CT2_ERR_INVALID, "FFT direction must be +1 or -1");
    if (batch < 1 || batch > 65535) return set_error(CT2_ERR_INVALID, "FFT batch %d outside [1, 65535]", batch);
    hipStream_t st = ctx().stream;
    if (f64)
        return dir > 0 ? fft3d_dispatch<double, 1>(data, n, st, batch) : fft3d_dispatch<double, -1>(data, n, st, batch);
    return dir > 0 ? fft3d_dispatch<float, 1>(data, n, st, batch) : fft3d_dispatch<float, -1>(data, n, st, batch);
}

int fft3d(void* data, int n, int dir, bool f64) { return fft3d_batch(data, n, dir, f64, 1); }

void release_fft_plans() {
    for (auto& kv : g_tw) dev_free(kv.second);
    g_tw.clear();
}

}  // namespace ct2

using namespace ct2;

extern "C" int ct2_fft3d_c2c(void* data, int n, int dir) { return fft3d(data, n, dir, false); }
extern "C" int ct2_fft3d_c2c_f64(void* data, int n, int dir) { return fft3d(data, n, dir, true); }
