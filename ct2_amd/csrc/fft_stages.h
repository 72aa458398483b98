// fft_stages.h -- the transform of one line by the lanes of a workgroup, shared
// by the 3-D FFT passes (fft.hip) and the kernels that fuse work into one
// (pm.hip).
#pragma once

#include "fft_radix.h"

namespace ct2 {
namespace {

// Radix plan: N = prod radix(N, s); the largest radix is 8 except N <= 4 and 16.
__host__ __device__ constexpr int rmax_of(int N) { return N <= 4 ? N : (N == 16 ? 4 : 8); }
__host__ __device__ constexpr int nstages_of(int N) {
    int s = 0, m = 1;
    while (m < N) {
        m *= rmax_of(N);
        ++s;
    }
    return s;
}
// stage 0 carries the remainder radix, the later stages rmax
__host__ __device__ constexpr int radix_of(int N, int s) {
    int rest = N;
    for (int k = 1; k < nstages_of(N); ++k) rest /= rmax_of(N);
    return s == 0 ? rest : rmax_of(N);
}
__host__ __device__ constexpr int ns_of(int N, int s) {
    int m = 1;
    for (int k = 0; k < s; ++k) m *= radix_of(N, k);
    return m;
}

// Lines per workgroup for the row kernel and columns per workgroup for the
// column kernels (of NC columns), sized for <= 64 KB of LDS and >= 256 lanes
// where possible.
template <typename T, int N, int NC = N>
struct Cfg {
    static constexpr int RM = rmax_of(N);
    static constexpr int P = N / RM;  // lanes per line, RM elements each
    static constexpr int ELEM = (int)sizeof(T) * 2;
    static constexpr int want_cols = (256 / P) > 16 ? (256 / P) : 16;
    static constexpr int lds_cols = (65536 / (N * ELEM)) > 0 ? (65536 / (N * ELEM)) : 1;
    static constexpr int C0 = want_cols < lds_cols ? want_cols : lds_cols;
    static constexpr int COLS = C0 < NC ? C0 : NC;
    static constexpr int want_rows = (256 / P) > 1 ? (256 / P) : 1;
    static constexpr int ROWS = want_rows < N * N ? want_rows : N * N;
    static constexpr int ROWLEN = N + N / 8;  // padded LDS row
};

// Stockham autosort stages of one line of N elements by its P lanes (this one
// is lane p).  ld(i, m) gives element i, st(i, m, v) takes output i; the lane
// touches i = p + m P only (m < RM, a constant once unrolled) in both, so a
// line's output can stay in registers as the next transform's input.  The
// stages exchange through LDS at sm[ix(i)].  LIN / LOUT: ld reads / st writes
// that LDS too, and a barrier keeps the two apart.  tw: the forward table.
template <typename T, int N, int DIR, bool LIN, bool LOUT, int S = 0, typename LD, typename ST, typename IX>
__device__ __forceinline__ void run_stages(const LD& ld, const ST& st, const IX& ix, typename V2<T>::t* sm,
                                           const typename V2<T>::t* tw, int p) {
    using T2 = typename V2<T>::t;
    using CF = Cfg<T, N>;
    constexpr int NS = nstages_of(N);
    constexpr int R = radix_of(N, S);
    constexpr int Ns = ns_of(N, S);
    constexpr int L = N / R;
    constexpr int NB = CF::RM / R;  // butterflies per lane in this stage
    constexpr bool FIRST = S == 0, LAST = S == NS - 1;
    T2 v[CF::RM];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int b = p + u * CF::P;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = b + r * L;
            if constexpr (FIRST)
                v[u * R + r] = ld(i, (u * CF::P + r * L) / CF::P);
            else
                v[u * R + r] = sm[ix(i)];
        }
        if constexpr (!FIRST) {
            const int k = b & (Ns - 1);
#pragma unroll
            for (int r = 1; r < R; ++r) {
                T2 w = tw[r * k * (N / (Ns * R))];
                if constexpr (DIR < 0) w.y = -w.y;
                v[u * R + r] = cmul(v[u * R + r], w);
            }
        }
        dft<R, DIR>(&v[u * R]);
    }
    if constexpr (LAST) {
        if constexpr (LOUT && (!FIRST || LIN)) __syncthreads();
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int r = 0; r < R; ++r)
                st(p + u * CF::P + r * L, (u * CF::P + r * L) / CF::P, v[u * R + r]);
    } else {
        if constexpr (!FIRST || LIN) __syncthreads();
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int b = p + u * CF::P;
            const int k = b & (Ns - 1);
            const int o = (b / Ns) * Ns * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) sm[ix(o + r * Ns)] = v[u * R + r];
        }
        __syncthreads();
        run_stages<T, N, DIR, LIN, LOUT, S + 1>(ld, st, ix, sm, tw, p);
    }
}

// The workgroup's copy of a table of N roots, every STEP-th of twg.
template <int N, int STEP = 1, typename T2>
__device__ __forceinline__ void load_twiddles(T2* tw, const T2* __restrict__ twg, int lanes) {
    for (int m = threadIdx.x; m < N; m += lanes) tw[m] = twg[m * STEP];
}

// Workgroups are dealt to the 8 XCDs in turn: XCD x takes the contiguous
// blocks [x G/8, (x+1) G/8) of G, so that neighbouring lines share its L2.
__device__ __forceinline__ unsigned xcd_contiguous(unsigned b, unsigned G) {
    return G % 8u == 0u ? (b % 8u) * (G / 8u) + b / 8u : b;
}

}  // namespace
}  // namespace ct2
