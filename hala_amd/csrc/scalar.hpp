// scalar.hpp -- the four scalar types' arithmetic, under one set of names.
//
// Complex values have the std::complex layout.  Never fused (-ffp-contract=off):
//   a * b = (ar br - ai bi, ar bi + ai br)
//   a / b = ((ar br + ai bi) / d, (ai br - ar bi) / d),  d = br br + bi bi
#pragma once
#include <hip/hip_runtime.h>

namespace hala_amd {

template <class R>
struct cx {
    R re, im;
};
template <class R>
__device__ __forceinline__ cx<R> cadd(cx<R> a, cx<R> b) {
    return {a.re + b.re, a.im + b.im};
}
template <class R>
__device__ __forceinline__ cx<R> csub(cx<R> a, cx<R> b) {
    return {a.re - b.re, a.im - b.im};
}
template <class R>
__device__ __forceinline__ cx<R> cmul(cx<R> a, cx<R> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <class R>
__device__ __forceinline__ cx<R> cdiv(cx<R> a, cx<R> b) {
    const R d = b.re * b.re + b.im * b.im;
    return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}
template <class R>
__device__ __forceinline__ cx<R> cconj(cx<R> a) {
    return {a.re, -a.im};
}
template <class R>
__device__ __forceinline__ bool czero(cx<R> a) {
    return a.re == R(0) && a.im == R(0);
}

__device__ __forceinline__ double cadd(double a, double b) { return a + b; }
__device__ __forceinline__ float cadd(float a, float b) { return a + b; }
__device__ __forceinline__ double cmul(double a, double b) { return a * b; }
__device__ __forceinline__ float cmul(float a, float b) { return a * b; }
__device__ __forceinline__ double cconj(double a) { return a; }
__device__ __forceinline__ float cconj(float a) { return a; }
__device__ __forceinline__ bool czero(double a) { return a == 0.0; }
__device__ __forceinline__ bool czero(float a) { return a == 0.0f; }

template <class S>
struct is_complex {
    static constexpr bool value = false;
};
template <class R>
struct is_complex<cx<R>> {
    static constexpr bool value = true;
};

}  // namespace hala_amd
