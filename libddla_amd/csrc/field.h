// Element types of the factorization kernels (device code): real elements (R)
// and complex ones (Cx<R>, the interleaved layout of std::complex<R>).  In LDS
// and in registers a complex block is two planes of real numbers, so that the
// matrix-core products are products of planes; a real block is one plane.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_tile.h"

namespace ddla {
namespace kern {

template <class R>
struct Cx {
    R re, im;
};

template <class T>
struct Field {
    using real = T;
    static constexpr int planes = 1;
};
template <class R>
struct Field<Cx<R>> {
    using real = R;
    static constexpr int planes = 2;
};
template <class T>
using real_t = typename Field<T>::real;

namespace field {

using gemm_detail::Mfma;

// Element operations (real y): x y, x - a b, x - a conj(b), d - |l|^2.
template <class R>
__device__ __forceinline__ R scale(R x, R y)
{
    return x * y;
}
template <class R>
__device__ __forceinline__ Cx<R> scale(Cx<R> x, R y)
{
    return {x.re * y, x.im * y};
}
template <class R>
__device__ __forceinline__ R sub_mul(R x, R a, R b)
{
    return fma(-a, b, x);
}
template <class R>
__device__ __forceinline__ Cx<R> sub_mul(Cx<R> x, Cx<R> a, Cx<R> b)
{
    return {fma(a.im, b.im, fma(-a.re, b.re, x.re)), fma(-a.im, b.re, fma(-a.re, b.im, x.im))};
}
template <class R>
__device__ __forceinline__ R sub_mul_conj(R x, R a, R b)
{
    return fma(-a, b, x);
}
template <class R>
__device__ __forceinline__ Cx<R> sub_mul_conj(Cx<R> x, Cx<R> a, Cx<R> b)
{
    return {fma(-a.im, b.im, fma(-a.re, b.re, x.re)), fma(-a.im, b.re, fma(a.re, b.im, x.im))};
}
template <class R>
__device__ __forceinline__ R sub_norm(R d, R l)
{
    return fma(-l, l, d);
}
template <class R>
__device__ __forceinline__ R sub_norm(R d, Cx<R> l)
{
    return fma(-l.im, l.im, fma(-l.re, l.re, d));
}

template <class T>
__device__ __forceinline__ real_t<T> plane(const T& x, int p)
{
    if constexpr (Field<T>::planes == 1) return x;
    else return p == 0 ? x.re : x.im;
}
template <class T>
__device__ __forceinline__ T element(real_t<T> re, real_t<T> im)
{
    if constexpr (Field<T>::planes == 1) return re;
    else return T{re, im};
}

// One 16x16x4 step of a product on the matrix cores for planes a[P] (left
// operand), b[P] (right), acc[P]:
//   mma_add:       acc += a b
//   mma_add_conj:  acc += a conj(b)
//   mma_sub_conj:  acc -= a conj(b)
//   mma_conj_add:  acc += conj(a) b
template <class R>
using acc_t = typename Mfma<R>::acc_t;

template <class R>
__device__ __forceinline__ void mma_add(const R (&a)[1], const R (&b)[1], acc_t<R> (&acc)[1])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
}
template <class R>
__device__ __forceinline__ void mma_add(const R (&a)[2], const R (&b)[2], acc_t<R> (&acc)[2])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
    acc[1] = Mfma<R>::mma(a[0], b[1], acc[1]);
    acc[0] = Mfma<R>::mma(-a[1], b[1], acc[0]);
    acc[1] = Mfma<R>::mma(a[1], b[0], acc[1]);
}
template <class R>
__device__ __forceinline__ void mma_sub_conj(const R (&a)[1], const R (&b)[1], acc_t<R> (&acc)[1])
{
    acc[0] = Mfma<R>::mma(-a[0], b[0], acc[0]);
}
template <class R>
__device__ __forceinline__ void mma_sub_conj(const R (&a)[2], const R (&b)[2], acc_t<R> (&acc)[2])
{
    acc[0] = Mfma<R>::mma(-a[0], b[0], acc[0]);
    acc[1] = Mfma<R>::mma(a[0], b[1], acc[1]);
    acc[0] = Mfma<R>::mma(-a[1], b[1], acc[0]);
    acc[1] = Mfma<R>::mma(-a[1], b[0], acc[1]);
}
template <class R>
__device__ __forceinline__ void mma_add_conj(const R (&a)[1], const R (&b)[1], acc_t<R> (&acc)[1])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
}
template <class R>
__device__ __forceinline__ void mma_add_conj(const R (&a)[2], const R (&b)[2], acc_t<R> (&acc)[2])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
    acc[1] = Mfma<R>::mma(-a[0], b[1], acc[1]);
    acc[0] = Mfma<R>::mma(a[1], b[1], acc[0]);
    acc[1] = Mfma<R>::mma(a[1], b[0], acc[1]);
}
template <class R>
__device__ __forceinline__ void mma_conj_add(const R (&a)[1], const R (&b)[1], acc_t<R> (&acc)[1])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
}
template <class R>
__device__ __forceinline__ void mma_conj_add(const R (&a)[2], const R (&b)[2], acc_t<R> (&acc)[2])
{
    acc[0] = Mfma<R>::mma(a[0], b[0], acc[0]);
    acc[1] = Mfma<R>::mma(a[0], b[1], acc[1]);
    acc[0] = Mfma<R>::mma(a[1], b[1], acc[0]);
    acc[1] = Mfma<R>::mma(-a[1], b[0], acc[1]);
}

} // namespace field
} // namespace kern
} // namespace ddla
