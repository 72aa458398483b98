// fft_ct2.hip -- ct2's own FFT entry points (fft.hpp:18-29) on the GPU, with
// ct2's data conventions, for callers that hold their data in device memory:
//
//   fft_complex (fft_complex_vector.cpp:9-65)  bit-reversed input, natural
//       output, FFTW_FORWARD sign for dir = +1 (dir = -1: the conjugate
//       transform, the evident intent of :57-58), unnormalised; `lanes`
//       interleaved transforms, element n lane l at re X[2 lanes n + l],
//       im X[2 lanes n + lanes + l] (complex<simd_f64>).
//   fft_real (fft_real_scalar.cpp:9-180, fft_real_vector.cpp:9-183)  real
//       bit-reversed input, half-complex output X[k] = Re F_k,
//       X[N-k] = Im F_k; lanes interleaved as [n][lane].
//   scramble (scramble.cpp:8-43), transpose_yz / transpose_r2c /
//       transpose_c2r (transpose.cpp:7-128, intended maps), and the 3-D
//       fft_r2c_3d / fft_c2r_3d (fft_r2c_3d.cpp, fft_c2r_3d.cpp: stubs in the
//       reference; here the planar layout out[(N/2+1)(N i + j) + k] = Re,
//       + N^2 (N/2+1) for Im, that transpose.cpp:36-56 prepares).
//
// The 1-D transforms sit in LDS as FP64 complex, several to a workgroup, and
// take radix-8 decimation-in-time steps in place (the input already is in
// bit-reversed order, so the output comes out in natural order), twiddles from
// an FP64 libm table, e^{-2 pi i m/N}; a real transform is a complex one of
// half the length.
// The 3-D transforms are fft.hip's real ones.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fft_radix.h"
#include "internal.h"

namespace ct2 {
namespace {

constexpr int F1_MAXN = 4096;

struct Twiddles {
    int n = 0;
    double2* d = nullptr;
};
std::vector<Twiddles> g_tw;
double2* g_half = nullptr;  // 3-D scratch: a half spectrum
size_t g_half_bytes = 0;

// Table W[m] = e^{-2 pi i m / N}, m < N, FP64 from libm.
int twiddles(int N, const double2** out) {
    for (const Twiddles& t : g_tw)
        if (t.n == N) {
            *out = t.d;
            return CT2_OK;
        }
    std::vector<double2> h(N);
    for (int m = 0; m < N; ++m) h[m] = make_double2(std::cos(2.0 * M_PI * m / N), -std::sin(2.0 * M_PI * m / N));
    Twiddles t;
    t.n = N;
    CT2_TRY(dev_alloc((void**)&t.d, h.size() * sizeof(double2), "1-D FFT twiddles"));
    CT2_HIP(hipMemcpy(t.d, h.data(), h.size() * sizeof(double2), hipMemcpyHostToDevice));
    g_tw.push_back(t);
    *out = t.d;
    return CT2_OK;
}

// One radix-R step (log2 R stages) of the transforms in LDS, T of M = 2^lm
// complex elements each, sub-transforms of 2^lh already done: outputs
// k + q h (q < R) of a group from its R sub-transforms' element k, which sit
// in bit-reversed order of the sub-transform.  W is the table of 2^(lm + 1)
// or 2^lm roots (ws = 1 or 0).
template <int R>
__device__ __forceinline__ void f1_step(double2* s, int threads, int T, int lm, int lh, int pitch,
                                        const double2* __restrict__ W, int ws) {
    constexpr int LR = R == 8 ? 3 : R == 4 ? 2 : 1;
    const int lq = lm - LR, nb = T << lq;
    for (int b = threadIdx.x; b < nb; b += threads) {
        const int q = b & ((1 << lq) - 1), k = q & ((1 << lh) - 1);
        const int base = ((q - k) << LR) + k;
        double2* row = s + (b >> lq) * pitch;
        double2 v[R];
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int rev = R == 8 ? ((j & 1) << 2 | (j & 2) | j >> 2) : R == 4 ? ((j & 1) << 1 | j >> 1) : j;
            const int i = base + (rev << lh);
            v[j] = row[i + (i >> 3)];
            if (lh > 0 && j > 0) v[j] = cmul(v[j], W[(j * k) << (lm - lh - LR + ws)]);
        }
        dft<R, 1>(v);
#pragma unroll
        for (int j = 0; j < R; ++j) {
            const int i = base + (j << lh);
            row[i + (i >> 3)] = v[j];
        }
    }
    __syncthreads();
}

// T <= E / M transforms per workgroup of E / 8 threads, in LDS: transform t,
// element e at t pitch + e + e/8 (the padding keeps the radix-8 steps' strided
// accesses, and the lanes of a group, off one bank group).  A transform holds 2 M doubles in memory, M = 2^lm:
//   complex (N = M): row r of a group's 2 M x L array is part r % 2 of element
//     r / 2;
//   real (N = 2 M): bit-reversed input holds the even samples in its first
//     half and the odd ones in its second, each again bit-reversed, so row r
//     is part r / M of element r % M of z = x_even + i x_odd, and
//     F_k = (Z_k + conj Z_{M-k}) / 2 - i W_N^k (Z_k - conj Z_{M-k}) / 2.
// dir = -1: the conjugate transform, as swapped parts in and out (complex) or
// the conjugate output (real).
// Bound by HBM (32 B per complex element, 16 B per real one) and the LDS
// passes: log8 M steps, one barrier each.  A group's L lanes stay in one
// workgroup wherever they fit (E up to 8192 elements, 148 KB), so that its
// interleaved lines are read once, eight reads of a thread in flight (one at a
// time, a group's reads alone cost as many trips to memory as it has doubles per
// thread: 27 x 4 real transforms of 2,048 with the caller's copy 19.1 us, now
// 15.9): 2,048 x 4 real transforms of 1,024 (67 MB each way) take 42 us.  One
// transform per workgroup with a radix-2
// stage per barrier, and every lane of a group read by another workgroup, took
// 121 us.
template <bool REAL, int L, int E>
__global__ __launch_bounds__(E / 8) void fft1d_ct2(double* __restrict__ X, int lm, long nt, int T, int dir,
                                                   const double2* __restrict__ W) {
    constexpr int TH = E / 8;
    __shared__ double2 s[E + E / 8 + E / 32];
    const int M = 1 << lm, pitch = M + (M >> 3) + (lm >= 5);
    const long t0 = (long)blockIdx.x * T;
    const int Lw = min(T, L);                     // lanes of a group in this workgroup
    const int ll = 31 - __clz(Lw);                // Lw is 1, 2 or 4
    const int have = (int)min((long)T, nt - t0);  // a multiple of Lw: nt and t0 are
    const int swap = !REAL && dir < 0;
    const int nd = have << (lm + 1);
    const long g0 = t0 / L, l0 = t0 % L;
    auto address = [&](int d) -> long {  // double d of the workgroup, in memory order
        const int l = d & (Lw - 1), r = (d >> ll) & (2 * M - 1), g = d >> (ll + lm + 1);
        return (((g0 + g) << (lm + 1)) + r) * L + l0 + l;
    };
#pragma unroll 8
    for (int d = threadIdx.x; d < nd; d += TH) {
        const int l = d & (Lw - 1), r = (d >> ll) & (2 * M - 1), g = d >> (ll + lm + 1);
        const int e = REAL ? r & (M - 1) : r >> 1;
        const int part = REAL ? r >> lm : (r & 1) ^ swap;
        ((double*)&s[((g << ll) + l) * pitch + e + (e >> 3)])[part] = X[address(d)];
    }
    __syncthreads();
    const int ws = REAL ? 1 : 0;
    int lh = lm % 3;
    if (lh == 1) f1_step<2>(s, TH, have, lm, 0, pitch, W, ws);
    if (lh == 2) f1_step<4>(s, TH, have, lm, 0, pitch, W, ws);
    for (; lh < lm; lh += 3) f1_step<8>(s, TH, have, lm, lh, pitch, W, ws);
#pragma unroll 4
    for (int d = threadIdx.x; d < nd; d += TH) {
        const int l = d & (Lw - 1), r = (d >> ll) & (2 * M - 1), g = d >> (ll + lm + 1);
        const double2* row = s + ((g << ll) + l) * pitch;
        if constexpr (REAL) {  // row r of the half-complex output: Re F_r, or Im F_{N-r} above N/2
            const bool im = r > M;
            const int k = im ? 2 * M - r : r;
            const int a = k & (M - 1), b = (M - k) & (M - 1);
            const double2 z1 = row[a + (a >> 3)], z2 = row[b + (b >> 3)], w = W[k];
            const double ox = 0.5 * (z1.x - z2.x), oy = 0.5 * (z1.y + z2.y);
            const double re = 0.5 * (z1.x + z2.x) + (w.x * oy + w.y * ox);
            const double mi = 0.5 * (z1.y - z2.y) - (w.x * ox - w.y * oy);
            X[address(d)] = im ? (dir < 0 ? -mi : mi) : re;
        } else {
            const int e = r >> 1;
            X[address(d)] = ((const double*)&row[e + (e >> 3)])[(r & 1) ^ swap];
        }
    }
}

// A transform per workgroup, log2 N radix-2 steps of a butterfly a thread: the
// shortest chain, for batches that leave the chip idle (a radix-8 step is three
// trips to LDS and the twiddles fewer, but a few waves' long arithmetic).  us per
// call in a row of them, of which 3.6 for the launch, this / fft1d_ct2: 100 real
// transforms of 256 4.0 / 9.1 (5.1 with one transform per workgroup there too),
// 1,000 complex ones of 512 7.6 / 8.4, 17 x 4 complex ones of 512 6.2 / 7.7.
constexpr int F1_FEW_MAXN = 1024;

// The rule: where this measured no slower (N = 8 to 1,024, 1 to 100,000 transforms).
constexpr bool fft1d_is_small(bool real, int lanes, int N, long nt) {
    const long elements = nt * (real ? N / 2 : N);
    return lanes == 1 ? N <= (real ? 512 : F1_FEW_MAXN) && nt <= (real ? 2048 : 4096) && elements <= 1L << 19
                      : N <= 512 && nt <= 512 && elements <= 1L << 16;
}

template <bool REAL>
__global__ __launch_bounds__(256) void fft1d_few(double* __restrict__ X, int N, int lanes, int dir,
                                                 const double2* __restrict__ W) {
    __shared__ double2 s[F1_FEW_MAXN];
    const int l = (int)(blockIdx.x % lanes), tid = threadIdx.x;
    X += (long)(blockIdx.x / lanes) * lanes * N * (REAL ? 1 : 2) + l;
    for (int n = tid; n < N; n += 256)
        s[n] = REAL ? make_double2(X[(long)lanes * n], 0.0)
                    : make_double2(X[2L * lanes * n], X[2L * lanes * n + lanes]);
    __syncthreads();
    for (int half = 1; half < N; half <<= 1) {
        const int stride = N / (2 * half);
        for (int q = tid; q < N / 2; q += 256) {
            const int k = q & (half - 1), i0 = ((q - k) << 1) + k, i1 = i0 + half;
            double2 w = W[k * stride];
            if (dir < 0) w.y = -w.y;
            const double2 a = s[i0], c = cmul(s[i1], w);
            s[i0] = cadd(a, c);
            s[i1] = csub(a, c);
        }
        __syncthreads();
    }
    if (REAL) {
        for (int k = tid; k <= N / 2; k += 256) {
            X[(long)lanes * k] = s[k].x;
            if (k > 0 && k < N / 2) X[(long)lanes * (N - k)] = s[k].y;
        }
    } else {
        for (int n = tid; n < N; n += 256) {
            X[2L * lanes * n] = s[n].x;
            X[2L * lanes * n + lanes] = s[n].y;
        }
    }
}

__device__ __forceinline__ int bitrev(int j, int bits) { return (int)(__brev((unsigned)j) >> (32 - bits)); }

// scramble: block j of N3 values <-> block bitrev(j), within each of N1 groups.
__global__ __launch_bounds__(256) void scramble_kernel(double* __restrict__ X, long total, int N2, int N3, int bits) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    const int t = (int)(e % N3);
    const long gj = e / N3;
    const int j = (int)(gj % N2);
    const long g = gj / N2;
    const int r = bits ? bitrev(j, bits) : 0;
    if (j < r) {
        double* base = X + g * (long)N2 * N3;
        const double a = base[(long)j * N3 + t];
        base[(long)j * N3 + t] = base[(long)r * N3 + t];
        base[(long)r * N3 + t] = a;
    }
}

__global__ __launch_bounds__(256) void transpose_yz_kernel(double* __restrict__ X, int N) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const long n3 = (long)N * N * N;
    if (e >= n3) return;
    const int z = (int)(e % N), y = (int)((e / N) % N);
    if (y < z) {
        const long x = e / ((long)N * N);
        const long j = (x * N + z) * N + y;
        const double a = X[e];
        X[e] = X[j];
        X[j] = a;
    }
}

// Half-complex rows along y of in[x][y][z] -> planar out[x][z][ky].
__global__ __launch_bounds__(256) void transpose_r2c_kernel(const double* __restrict__ in, double* __restrict__ out,
                                                            int N) {
    const int h = N / 2 + 1;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;  // over [x][iy < h][z]
    const long tot = (long)N * h * N;
    if (e >= tot) return;
    const int iz = (int)(e % N), iy = (int)((e / N) % h);
    const long ix = e / ((long)N * h);
    const long dimag = (long)N * N * h;
    const long jr = (ix * N + iz) * h + iy;
    out[jr] = in[(ix * N + iy) * N + iz];
    out[jr + dimag] = (iy == 0 || iy == N / 2) ? 0.0 : in[(ix * N + (N - iy)) * N + iz];
}

__global__ __launch_bounds__(256) void transpose_c2r_kernel(const double* __restrict__ in, double* __restrict__ out,
                                                            int N) {
    const int h = N / 2 + 1;
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const long tot = (long)N * h * N;
    if (e >= tot) return;
    const int iz = (int)(e % N), iy = (int)((e / N) % h);
    const long ix = e / ((long)N * h);
    const long dimag = (long)N * N * h;
    const long jr = (ix * N + iz) * h + iy;
    out[(ix * N + iy) * N + iz] = in[jr];
    if (iy != 0 && iy != N / 2) out[(ix * N + (N - iy)) * N + iz] = in[jr + dimag];
}

int check_1d(const void* X, int N, int dir, int lanes, size_t batch) {
    CT2_TRY(require_init());
    if (!X) return set_error(CT2_ERR_INVALID, "null data");
    if (!is_pow2(N) || N < 2 || N > F1_MAXN) return set_error(CT2_ERR_INVALID, "N = %d is not a power of two in [2, %d]", N, F1_MAXN);
    if (dir != 1 && dir != -1) return set_error(CT2_ERR_INVALID, "dir must be +1 or -1");
    if (lanes != 1 && lanes != 4) return set_error(CT2_ERR_INVALID, "lanes must be 1 or 4");
    if (batch == 0 || batch * (size_t)lanes > (size_t)1 << 30) return set_error(CT2_ERR_INVALID, "bad batch %zu", batch);
    return CT2_OK;
}

template <bool REAL, int L, int E>
int fft1d_launch(double* X, int N, int dir, size_t batch) {
    const double2* W;
    CT2_TRY(twiddles(N, &W));
    const int lm = ilog2(N) - (REAL ? 1 : 0);
    const long nt = (long)batch * L;
    // fewer to a workgroup where there would not be one for every CU (300 x 4 real
    // transforms of 128: 8.0 -> 4.7 us), but a group's lanes together unless the
    // data are small (17 x 4 complex ones of 2,048: 18.2 -> 12.7 us one by one;
    // 100 x 4: 19 -> 30)
    int T = E >> lm;
    while (T > 1 && (nt + T - 1) / T < 256 && (T > L || nt <= 128)) T /= 2;
    fft1d_ct2<REAL, L, E><<<(unsigned)((nt + T - 1) / T), E / 8, 0, ctx().stream>>>(X, lm, nt, T, dir, W);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

// 2048 elements per workgroup (256 threads, four workgroups per CU), more
// where a group's lanes or a single transform need it.
template <bool REAL, int L>
int fft1d_elements(double* X, int N, int dir, size_t batch) {
    if (fft1d_is_small(REAL, L, N, (long)batch * L)) {
        const double2* W;
        CT2_TRY(twiddles(N, &W));
        fft1d_few<REAL><<<(unsigned)(batch * L), 256, 0, ctx().stream>>>(X, N, L, dir, W);
        CT2_LAUNCH_CHECK();
        return CT2_OK;
    }
    const int need = (REAL ? N / 2 : N) * L;
    if (need <= 2048) return fft1d_launch<REAL, L, 2048>(X, N, dir, batch);
    if (need <= 4096) return fft1d_launch<REAL, L, 4096>(X, N, dir, batch);
    return fft1d_launch<REAL, L, 8192>(X, N, dir, batch);
}

int grid_1d(long total) { return (int)((total + 255) / 256); }

int check_3d(const void* a, const void* b, int N) {
    CT2_TRY(require_init());
    if (!a || !b) return set_error(CT2_ERR_INVALID, "null data");
    if (!is_pow2(N) || N < 8 || N > 512) return set_error(CT2_ERR_INVALID, "N = %d is not a power of two in [8, 512]", N);
    return CT2_OK;
}

}  // namespace

void release_fft_ct2() {
    for (Twiddles& t : g_tw) dev_free(t.d);
    g_tw.clear();
    dev_free(g_half);
    g_half = nullptr;
    g_half_bytes = 0;
}

}  // namespace ct2

using namespace ct2;

extern "C" int ct2_fft_complex_1d(double* X, int N, int dir, int lanes, size_t batch) {
    CT2_TRY(check_1d(X, N, dir, lanes, batch));
    return lanes == 1 ? fft1d_elements<false, 1>(X, N, dir, batch) : fft1d_elements<false, 4>(X, N, dir, batch);
}

extern "C" int ct2_fft_real_1d(double* X, int N, int dir, int lanes, size_t batch) {
    CT2_TRY(check_1d(X, N, dir, lanes, batch));
    return lanes == 1 ? fft1d_elements<true, 1>(X, N, dir, batch) : fft1d_elements<true, 4>(X, N, dir, batch);
}

extern "C" int ct2_scramble(double* X, int N1, int N2, int N3) {
    CT2_TRY(require_init());
    if (!X || N1 <= 0 || N3 <= 0 || !is_pow2(N2)) return set_error(CT2_ERR_INVALID, "bad scramble arguments");
    const long total = (long)N1 * N2 * N3;
    if (total > (1L << 33)) return set_error(CT2_ERR_INVALID, "scramble too large");
    scramble_kernel<<<grid_1d(total), 256, 0, ctx().stream>>>(X, total, N2, N3, ilog2(N2));
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

extern "C" int ct2_transpose_yz(double* X, int N) {
    CT2_TRY(require_init());
    if (!X || N <= 0 || N > 2048) return set_error(CT2_ERR_INVALID, "bad transpose arguments");
    transpose_yz_kernel<<<grid_1d((long)N * N * N), 256, 0, ctx().stream>>>(X, N);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

extern "C" int ct2_transpose_r2c(const double* in, double* out, int N) {
    CT2_TRY(require_init());
    if (!in || !out || N < 2 || N % 2 || N > 2048) return set_error(CT2_ERR_INVALID, "bad transpose arguments");
    transpose_r2c_kernel<<<grid_1d((long)N * (N / 2 + 1) * N), 256, 0, ctx().stream>>>(in, out, N);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

extern "C" int ct2_transpose_c2r(const double* in, double* out, int N) {
    CT2_TRY(require_init());
    if (!in || !out || N < 2 || N % 2 || N > 2048) return set_error(CT2_ERR_INVALID, "bad transpose arguments");
    transpose_c2r_kernel<<<grid_1d((long)N * (N / 2 + 1) * N), 256, 0, ctx().stream>>>(in, out, N);
    CT2_LAUNCH_CHECK();
    return CT2_OK;
}

// Both directions read all of `in` into the scratch before the first write of
// `out`, which may overlap it.
extern "C" int ct2_fft_r2c_3d(const double* in, double* out, int N) {
    CT2_TRY(check_3d(in, out, N));
    CT2_TRY(ensure_scratch((void**)&g_half, &g_half_bytes, fft_half_elems(N) * sizeof(double2), "3-D r2c scratch"));
    return rfft3d_f64(in, out, g_half, N);
}

extern "C" int ct2_fft_c2r_3d(const double* in, double* out, int N) {
    CT2_TRY(check_3d(in, out, N));
    CT2_TRY(ensure_scratch((void**)&g_half, &g_half_bytes, fft_half_elems(N) * sizeof(double2), "3-D c2r scratch"));
    return irfft3d_f64(in, out, g_half, N);
}

extern "C" int ct2_twiddles(int N, double* cosw, double* sinw, double* invsinw) {
    if (N <= 0 || !cosw || !sinw || !invsinw) return set_error(CT2_ERR_INVALID, "bad twiddle arguments");
    for (int n = 0; n < N; ++n) {
        const double a = 2.0 * M_PI * n / N;
        cosw[n] = std::cos(-a);
        sinw[n] = std::sin(-a);
        invsinw[n] = std::sin(a);
    }
    return CT2_OK;
}
