// hbem_complex.hpp -- complex arithmetic of the dense kernels (LU, solves,
// randomized SVD), in double and single precision.
#pragma once
#include <type_traits>

#include "hbem_internal.hpp"

namespace hbem {

constexpr int kMaxNc = 8;                     // most right-hand sides of the randomized SVD

template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(const F& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// Reciprocal and product with every multiply-add an explicit fma: the LU's
// arithmetic per matrix entry is then fixed by the source, whichever kernel
// instantiation (rows per thread, chunk width) performs it, so a matrix
// factorised inside a larger zero-padded one gives the same bits.
__device__ __forceinline__ cdbl crecip(cdbl d) {
    const double s = 1.0 / fma(d.x, d.x, d.y * d.y);
    return mk(d.x * s, -d.y * s);
}
__device__ __forceinline__ cdbl cmulx(cdbl a, cdbl b) { return mk(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x)); }
__device__ __forceinline__ void cfms(cdbl& acc, cdbl a, cdbl b) {   // acc -= a * b
    acc.x = fma(-a.x, b.x, fma(a.y, b.y, acc.x));
    acc.y = fma(-a.x, b.y, fma(-a.y, b.x, acc.y));
}
__device__ __forceinline__ void cfma(cdbl& acc, cdbl a, cdbl b) {   // acc += a * b
    acc.x = fma(a.x, b.x, fma(-a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(a.y, b.x, acc.y));
}
__device__ __forceinline__ cdbl shfl_c(cdbl v, int src) {
    return mk(__shfl(v.x, src, 64), __shfl(v.y, src, 64));
}
// lane src's value in every lane, src the same for the whole wavefront:
// v_readlane through a scalar register, no LDS round trip
__device__ __forceinline__ double bcast_lane(double v, int src) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ cdbl bcast_lane(cdbl v, int src) { return mk(bcast_lane(v.x, src), bcast_lane(v.y, src)); }

// The same operations on single-precision complex values (the factors of the
// mixed-precision LU).
__device__ __forceinline__ float cabs2(cflt a) { return a.x * a.x + a.y * a.y; }
__device__ __forceinline__ cflt operator*(cflt a, cflt b) { return cflt{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ __forceinline__ cflt crecip(cflt d) {
    const float s = 1.0f / fmaf(d.x, d.x, d.y * d.y);
    return cflt{d.x * s, -d.y * s};
}
__device__ __forceinline__ cflt cmulx(cflt a, cflt b) {
    return cflt{fmaf(a.x, b.x, -(a.y * b.y)), fmaf(a.x, b.y, a.y * b.x)};
}
__device__ __forceinline__ void cfms(cflt& acc, cflt a, cflt b) {   // acc -= a * b
    acc.x = fmaf(-a.x, b.x, fmaf(a.y, b.y, acc.x));
    acc.y = fmaf(-a.x, b.y, fmaf(-a.y, b.x, acc.y));
}
__device__ __forceinline__ cflt shfl_c(cflt v, int src) { return cflt{__shfl(v.x, src, 64), __shfl(v.y, src, 64)}; }
// widening load of a factor entry for double-precision arithmetic
__device__ __forceinline__ cdbl to_cdbl(cdbl v) { return v; }
__device__ __forceinline__ cdbl to_cdbl(cflt v) { return mk((double)v.x, (double)v.y); }

}  // namespace hbem
