// fft_radix.h -- complex arithmetic and the small DFTs the transforms of
// fft.hip and fft_ct2.hip are built from.
#pragma once

#include <hip/hip_runtime.h>

namespace ct2 {
namespace {

template <typename T>
struct V2;
template <>
struct V2<float> {
    using t = float2;
};
template <>
struct V2<double> {
    using t = double2;
};

template <typename T2>
__device__ __forceinline__ T2 cadd(T2 a, T2 b) {
    return T2{a.x + b.x, a.y + b.y};
}
template <typename T2>
__device__ __forceinline__ T2 csub(T2 a, T2 b) {
    return T2{a.x - b.x, a.y - b.y};
}
template <typename T2>
__device__ __forceinline__ T2 cmul(T2 a, T2 b) {
    return T2{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
// a * (-i * DIR)
template <int DIR, typename T2>
__device__ __forceinline__ T2 mul_mi(T2 a) {
    if constexpr (DIR > 0)
        return T2{a.y, -a.x};
    else
        return T2{-a.y, a.x};
}

// In-register DFT of R points, X_k = sum_j v_j e^{-2 pi i DIR jk/R}.
template <int R, int DIR, typename T2>
__device__ __forceinline__ void dft(T2* v) {
    if constexpr (R == 2) {
        const T2 a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    } else if constexpr (R == 4) {
        const T2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
        const T2 c = cadd(v[1], v[3]), d = mul_mi<DIR>(csub(v[1], v[3]));
        v[0] = cadd(a, c);
        v[1] = cadd(b, d);
        v[2] = csub(a, c);
        v[3] = csub(b, d);
    } else {
        static_assert(R == 8, "radix");
        using T = decltype(v[0].x);
        T2 e[4] = {v[0], v[2], v[4], v[6]};
        T2 o[4] = {v[1], v[3], v[5], v[7]};
        dft<4, DIR>(e);
        dft<4, DIR>(o);
        const T s = (T)0.70710678118654752440;
        // o1 *= (1 - i DIR)/sqrt2 ; o2 *= -i DIR ; o3 *= (-1 - i DIR)/sqrt2
        o[1] = T2{(o[1].x + DIR * o[1].y) * s, (o[1].y - DIR * o[1].x) * s};
        o[2] = mul_mi<DIR>(o[2]);
        o[3] = T2{(-o[3].x + DIR * o[3].y) * s, (-o[3].y - DIR * o[3].x) * s};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = cadd(e[k], o[k]);
            v[k + 4] = csub(e[k], o[k]);
        }
    }
}

}  // namespace
}  // namespace ct2
