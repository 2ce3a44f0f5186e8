// scalars.hpp — the number systems H(k) lives in, for the kernels of the
// eigen-solve (one template, three element types):
//
//   r1<R>  real        H(k) of a crystal with an inversion centre, no spin-orbit
//   c2<R>  complex     any H(k)
//   q4<R>  quaternion  H(k) of a crystal with an inversion centre and spin-orbit:
//                      the 2 x 2 spinor block of a pair of basis vectors is
//                      [[u, -conj(d)], [d, conj(u)]], u = x + i y, d = z + i w
//
// A real number costs a quarter of a complex one's multiply-adds, and a
// quaternion matrix of half the dimension half of the complex one's.  Products
// keep their order (quaternions do not commute).
#pragma once
#include <hip/hip_runtime.h>

namespace uepm {

template <typename R_>
struct r1 {
    using R = R_;
    static constexpr int NC = 1;
    R x;
};
template <typename R_>
struct c2 {
    using R = R_;
    static constexpr int NC = 2;
    R x, y;
};
template <typename R_>
struct alignas(4 * sizeof(R_)) q4 {
    using R = R_;
    static constexpr int NC = 4;
    R x, y, z, w;
};

#define UEPM_SC template <typename R> __device__ __forceinline__

// zero, one, and a real number as a scalar of type S
template <typename S>
__device__ __forceinline__ S sc_real(typename S::R a) {
    S s{};
    s.x = a;
    return s;
}
UEPM_SC r1<R> add(r1<R> a, r1<R> b) { return {a.x + b.x}; }
UEPM_SC c2<R> add(c2<R> a, c2<R> b) { return {a.x + b.x, a.y + b.y}; }
UEPM_SC q4<R> add(q4<R> a, q4<R> b) { return {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }

// f a for a real f
UEPM_SC r1<R> scale(r1<R> a, R f) { return {f * a.x}; }
UEPM_SC c2<R> scale(c2<R> a, R f) { return {f * a.x, f * a.y}; }
UEPM_SC q4<R> scale(q4<R> a, R f) { return {f * a.x, f * a.y, f * a.z, f * a.w}; }

// conj(a) where c, else a
UEPM_SC r1<R> conj_if(r1<R> a, bool) { return a; }
UEPM_SC c2<R> conj_if(c2<R> a, bool c) { return {a.x, c ? -a.y : a.y}; }
UEPM_SC q4<R> conj_if(q4<R> a, bool c) { return {a.x, c ? -a.y : a.y, c ? -a.z : a.z, c ? -a.w : a.w}; }

// a b
UEPM_SC r1<R> mul(r1<R> a, r1<R> b) { return {a.x * b.x}; }
UEPM_SC c2<R> mul(c2<R> a, c2<R> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
UEPM_SC q4<R> mul(q4<R> a, q4<R> b) {
    return {a.x * b.x - a.y * b.y - a.z * b.z - a.w * b.w, a.x * b.y + a.y * b.x - a.z * b.w + a.w * b.z,
            a.x * b.z + a.y * b.w + a.z * b.x - a.w * b.y, a.x * b.w - a.y * b.z + a.z * b.y + a.w * b.x};
}

// c ? a : b per component (a select of the whole struct would go through memory)
UEPM_SC r1<R> sel(bool c, r1<R> a, r1<R> b) { return {c ? a.x : b.x}; }
UEPM_SC c2<R> sel(bool c, c2<R> a, c2<R> b) { return {c ? a.x : b.x, c ? a.y : b.y}; }
UEPM_SC q4<R> sel(bool c, q4<R> a, q4<R> b) {
    return {c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w};
}

// acc + |a|^2, acc + Re(conj(a) b), |imaginary part|^2
UEPM_SC R norm2(r1<R> a) { return a.x * a.x; }
UEPM_SC R norm2(c2<R> a) { return fma(a.x, a.x, a.y * a.y); }
UEPM_SC R norm2(q4<R> a) { return fma(a.x, a.x, fma(a.y, a.y, fma(a.z, a.z, a.w * a.w))); }
UEPM_SC R dot_acc(r1<R> a, r1<R> b, R acc) { return fma(a.x, b.x, acc); }
UEPM_SC R dot_acc(c2<R> a, c2<R> b, R acc) { return fma(a.x, b.x, fma(a.y, b.y, acc)); }
UEPM_SC R dot_acc(q4<R> a, q4<R> b, R acc) {
    return fma(a.x, b.x, fma(a.y, b.y, fma(a.z, b.z, fma(a.w, b.w, acc))));
}
UEPM_SC R imag2(r1<R>) { return R(0); }
UEPM_SC R imag2(c2<R> a) { return a.y * a.y; }
UEPM_SC R imag2(q4<R> a) { return fma(a.y, a.y, fma(a.z, a.z, a.w * a.w)); }
// Whether a column whose elements below its first one, al, have the squared norm xn2
// takes a reflector: not when they are all below 1e-15 (FP64: 1e-145), far under the
// rounding of any matrix here, where 1 / |x|^2 (and |x|^2) would leave the range.  (NaN does.)
template <typename S>
__device__ __forceinline__ bool reflects(typename S::R xn2, S al) {
    using R = typename S::R;
    return !(xn2 + imag2(al) <= (sizeof(R) == 4 ? R(1e-30) : R(1e-290)));
}

// f a + b for a real f
UEPM_SC r1<R> axpy(R f, r1<R> a, r1<R> b) { return {fma(f, a.x, b.x)}; }
UEPM_SC c2<R> axpy(R f, c2<R> a, c2<R> b) { return {fma(f, a.x, b.x), fma(f, a.y, b.y)}; }
UEPM_SC q4<R> axpy(R f, q4<R> a, q4<R> b) {
    return {fma(f, a.x, b.x), fma(f, a.y, b.y), fma(f, a.z, b.z), fma(f, a.w, b.w)};
}

// acc += a b
UEPM_SC void fma_ab(r1<R>& acc, r1<R> a, r1<R> b) { acc.x = fma(a.x, b.x, acc.x); }
UEPM_SC void fma_ab(c2<R>& acc, c2<R> a, c2<R> b) {
    acc.x = fma(a.x, b.x, fma(-a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(a.y, b.x, acc.y));
}
UEPM_SC void fma_ab(q4<R>& acc, q4<R> a, q4<R> b) {
    acc.x = fma(a.x, b.x, fma(-a.y, b.y, fma(-a.z, b.z, fma(-a.w, b.w, acc.x))));
    acc.y = fma(a.x, b.y, fma(a.y, b.x, fma(-a.z, b.w, fma(a.w, b.z, acc.y))));
    acc.z = fma(a.x, b.z, fma(a.y, b.w, fma(a.z, b.x, fma(-a.w, b.y, acc.z))));
    acc.w = fma(a.x, b.w, fma(-a.y, b.z, fma(a.z, b.y, fma(a.w, b.x, acc.w))));
}
// acc += conj(a) b
UEPM_SC void fma_cab(r1<R>& acc, r1<R> a, r1<R> b) { acc.x = fma(a.x, b.x, acc.x); }
UEPM_SC void fma_cab(c2<R>& acc, c2<R> a, c2<R> b) {
    acc.x = fma(a.x, b.x, fma(a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(-a.y, b.x, acc.y));
}
UEPM_SC void fma_cab(q4<R>& acc, q4<R> a, q4<R> b) {
    acc.x = fma(a.x, b.x, fma(a.y, b.y, fma(a.z, b.z, fma(a.w, b.w, acc.x))));
    acc.y = fma(a.x, b.y, fma(-a.y, b.x, fma(a.z, b.w, fma(-a.w, b.z, acc.y))));
    acc.z = fma(a.x, b.z, fma(-a.y, b.w, fma(-a.z, b.x, fma(a.w, b.y, acc.z))));
    acc.w = fma(a.x, b.w, fma(a.y, b.z, fma(-a.z, b.y, fma(-a.w, b.x, acc.w))));
}
// acc -= a conj(b)
UEPM_SC void fms_abc(r1<R>& acc, r1<R> a, r1<R> b) { acc.x = fma(-a.x, b.x, acc.x); }
UEPM_SC void fms_abc(c2<R>& acc, c2<R> a, c2<R> b) {
    acc.x = fma(-a.x, b.x, acc.x);
    acc.x = fma(-a.y, b.y, acc.x);
    acc.y = fma(-a.y, b.x, acc.y);
    acc.y = fma(a.x, b.y, acc.y);
}
UEPM_SC void fms_abc(q4<R>& acc, q4<R> a, q4<R> b) {
    acc.x = fma(-a.x, b.x, fma(-a.y, b.y, fma(-a.z, b.z, fma(-a.w, b.w, acc.x))));
    acc.y = fma(a.x, b.y, fma(-a.y, b.x, fma(-a.z, b.w, fma(a.w, b.z, acc.y))));
    acc.z = fma(a.x, b.z, fma(a.y, b.w, fma(-a.z, b.x, fma(-a.w, b.y, acc.z))));
    acc.w = fma(a.x, b.w, fma(-a.y, b.z, fma(a.z, b.y, fma(-a.w, b.x, acc.w))));
}
#undef UEPM_SC

// Element types in memory: float / double, float2 / double2, q4<float> / q4<double>.
template <typename S>
struct ScMem;
template <>
struct ScMem<r1<float>> { using T = float; };
template <>
struct ScMem<r1<double>> { using T = double; };
template <>
struct ScMem<c2<float>> { using T = float2; };
template <>
struct ScMem<c2<double>> { using T = double2; };
template <>
struct ScMem<q4<float>> { using T = q4<float>; };
template <>
struct ScMem<q4<double>> { using T = q4<double>; };

// the scalar of type S held by a memory element (converted to S's precision)
template <typename S, typename T>
__device__ __forceinline__ S sc_load(const T& h) {
    using R = typename S::R;
    if constexpr (S::NC == 1) return S{(R)h};
    else if constexpr (S::NC == 2) return S{(R)h.x, (R)h.y};
    else return S{(R)h.x, (R)h.y, (R)h.z, (R)h.w};
}
template <typename S>
__device__ __forceinline__ typename ScMem<S>::T sc_store(S a) {
    typename ScMem<S>::T v;
    if constexpr (S::NC == 1) v = a.x;
    else if constexpr (S::NC == 2) {
        v.x = a.x;
        v.y = a.y;
    } else v = a;
    return v;
}

}  // namespace uepm
