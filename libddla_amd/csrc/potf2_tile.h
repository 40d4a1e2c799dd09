// Cholesky factorization and triangular inverse of one 64 x 64 diagonal block
// held in LDS, for a 256-thread workgroup on gfx950 (device code, included by
// kernels.hip).
//
// The block S is column-major in LDS with column stride kL (S[c * kL + r] =
// A(r, c)) and only its lower triangle is referenced.  It is factored in
// 16-column strips, the inverse X = L^-1 growing beside it:
//   * a strip is factored four columns at a time on the matrix cores
//     (factor_strip).  Every wavefront keeps the strip's 16 x 16 diagonal
//     block and one 16 x 16 block of its own (rows below; wavefront 0: the
//     identity) in the accumulator layout, in which the four columns of a step
//     are one register and, as they stand, both operands of the 16x16x4
//     product that applies them to the later columns.  The step's 4 x 4
//     diagonal block is factored and inverted by every lane redundantly, so
//     neither a pivot's chain to the next one nor the strip has any exchange
//     between wavefronts in it, and the pass turns the identity into
//     L(b, b)^-T, the inverse of the strip's diagonal block;
//   * between two passes the strip is applied to the next strip's columns
//     (update_tile), and to the columns beyond while the next pass runs; the
//     wavefronts that have no rows left in a strip also form, during the
//     passes, the 16 x 16 products of the inverse, X(r, c) = -D(r) sum_k
//     L(r, k) X(k, c).
// What bounds it is the dependency chain of 64 pivots; after the last strip
// only one 16 x 16 product is left of the inverse.  Measured on one workgroup,
// factor and inverse of a block: FP64 13.4 -> 7.3 us, FP32 9.6 -> 5.1 us against
// strips factored column by column in one wavefront (pivots and multipliers
// through v_readlane) with the inverse formed afterwards.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_tile.h"

namespace ddla {
namespace kern {
namespace potf2_detail {

using gemm_detail::Mfma;

constexpr int kB = 64;  // block order
constexpr int kL = 65;  // LDS column stride, in elements
constexpr int kW = 16;  // strip width

template <int i>
struct Const {
    static constexpr int value = i;
};

__device__ inline double lane_value(double x, int l)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ inline float lane_value(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// x where mask is all ones, zero where it is zero (whatever x is).
__device__ inline double masked(double x, int mask)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)b & (unsigned)mask, hi = (unsigned)(b >> 32) & (unsigned)mask;
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ inline float masked(float x, int mask) { return __int_as_float(__float_as_int(x) & mask); }

// The bits of x and y together (one of them masked to zero).
__device__ inline double merged(double x, double y)
{
    return __longlong_as_double(__double_as_longlong(x) | __double_as_longlong(y));
}

__device__ inline float merged(float x, float y) { return __int_as_float(__float_as_int(x) | __float_as_int(y)); }

// 1 / sqrt(d) for d > 0: the hardware estimate and one third-order step (FP64:
// with e = 1 - d y^2, y (1 + e/2 + 3 e^2 / 8); the estimate's ~2^-23 becomes
// ~2^-67, rounding aside) or one Newton step (FP32).
__device__ inline double rsqrt_refined(double d)
{
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-(d * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

__device__ inline float rsqrt_refined(float d)
{
    float y = __builtin_amdgcn_rsqf(d);
    const float h = 0.5f * d;
    const float e = fmaf(-h * y, y, 0.5f);
    return fmaf(y, e, y);
}

// Row of the diagonal block that lane l % 16 holds, and the lane that holds
// row r of it: chosen so that register q of the accumulator layout holds
// columns 4q .. 4q + 3 (column 4q + lane / 16) and can serve as the product's
// left operand too.  FP64 accumulators are D[l / 16 + 4r][l % 16], FP32 ones
// D[4 (l / 16) + r][l % 16].
template <class T>
__device__ constexpr int diag_row(int i)
{
    return sizeof(T) == 8 ? i : (i >> 2) + 4 * (i & 3);  // its own inverse
}

// One wavefront's share of strip b (columns 16b .. 16b+15): wavefront w < 4 - b
// takes, beside the diagonal block, the rows 16 (b + w) .. below it, or for w =
// 0 the identity.  Rows below are written back to S, D(b) = L(b, b)^-1 to X's
// block (b, b), zeros above its diagonal; the diagonal block of L stays in diag
// (the other wavefronts still read S's when this one is done: store_diagonal
// after a barrier).  Returns 0, or the 1-based block index of the first pivot
// that is not positive (or is NaN); the columns from that pivot on then hold no
// meaningful values.  No branch depends on a pivot (a failed one is recorded,
// not acted on).
template <class T, int b>
__device__ __attribute__((always_inline)) inline int factor_strip(T* S, T* X, T (&diag)[4])
{
    using Op = Mfma<T>;
    using acc_t = typename Op::acc_t;
    constexpr int r0 = kW * b;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int pr = diag_row<T>(li);
    acc_t d, x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = g + 4 * r;
        d[r] = masked(S[(r0 + c) * kL + r0 + pr], -(int)(pr >= c));
        x[r] = wave == 0 ? (li == c ? T(1) : T(0)) : S[(r0 + c) * kL + r0 + kW * wave + li];
    }
    const T u0 = g == 0 ? T(1) : T(0), u1 = g == 1 ? T(1) : T(0), u2 = g == 2 ? T(1) : T(0), u3 = g == 3 ? T(1) : T(0);
    T below[4];                  // the finished columns of x
    unsigned long long bad = 0;  // bit j: the pivot of column j is not positive
    auto check = [&](T p, int j) { bad |= __ballot(!(p > T(0))) & (1ull << j); };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        auto at = [&](int r, int c) { return lane_value(d[q], 16 * c + diag_row<T>(4 * q + r)); };
        const T a00 = at(0, 0), a10 = at(1, 0), a20 = at(2, 0), a30 = at(3, 0), a11 = at(1, 1);
        const T a21 = at(2, 1), a31 = at(3, 1), a22 = at(2, 2), a32 = at(3, 2), a33 = at(3, 3);
        const T y0 = rsqrt_refined(a00);
        const T l10 = a10 * y0, l20 = a20 * y0, l30 = a30 * y0;
        const T d1 = fma(-l10, l10, a11), y1 = rsqrt_refined(d1);
        const T l21 = fma(-l20, l10, a21) * y1, l31 = fma(-l30, l10, a31) * y1;
        const T d2 = fma(-l21, l21, fma(-l20, l20, a22)), y2 = rsqrt_refined(d2);
        const T l32 = fma(-l31, l21, fma(-l30, l20, a32)) * y2;
        const T d3 = fma(-l32, l32, fma(-l31, l31, fma(-l30, l30, a33))), y3 = rsqrt_refined(d3);
        check(a00, 4 * q);
        check(d1, 4 * q + 1);
        check(d2, 4 * q + 2);
        check(d3, 4 * q + 3);
        // column g of the 4 x 4 inverse, then its row diag_row(l % 16) as the left operand
        const T e0 = u0 * y0, e1 = fma(-l10, e0, u1) * y1;
        const T e2 = fma(-l21, e1, fma(-l20, e0, u2)) * y2;
        const T e3 = fma(-l32, e2, fma(-l31, e1, fma(-l30, e0, u3))) * y3;
        const T inv = merged(merged(masked(e0, -(int)(pr == 0)), masked(e1, -(int)(pr == 1))),
                             merged(masked(e2, -(int)(pr == 2)), masked(e3, -(int)(pr == 3))));
        const acc_t zero = {0, 0, 0, 0};
        diag[q] = Op::mma(inv, d[q], zero)[0];
        if (q < 3) d = Op::mma(masked(-diag[q], -(int)(pr >= 4 * q + 4)), diag[q], d);
        below[q] = Op::mma(inv, x[q], zero)[0];
        if (q < 3) x = Op::mma(masked(-diag[q], -(int)(pr >= 4 * q + 4)), below[q], x);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = g + 4 * r;
        if (wave == 0) X[(r0 + li) * kL + r0 + c] = below[r];
        else S[(r0 + c) * kL + r0 + kW * wave + li] = below[r];
    }
    return bad == 0 ? 0 : r0 + (int)__ffsll(bad);
}

// L(b, b), as factor_strip left it in a wavefront's diag, to S.
template <class T>
__device__ __attribute__((always_inline)) inline void store_diagonal(const T (&diag)[4], int b, T* S)
{
    const int lane = threadIdx.x & 63, pr = diag_row<T>(lane & 15);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int c = (lane >> 4) + 4 * r;
        if (pr >= c) S[(kW * b + c) * kL + kW * b + pr] = diag[r];
    }
}

// S(16r.., 16c..) -= L(16r.., strip b) L(16c.., strip b)^T, one 16 x 16 tile by
// one wavefront.
template <class T>
__device__ __attribute__((always_inline)) inline void update_tile(T* S, int b, int r, int c)
{
    using Op = Mfma<T>;
    const int lane = threadIdx.x & 63, li = lane & 15;
    T* C = S + (kW * c + li) * kL + kW * r;
    typename Op::acc_t acc;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = C[Op::row(lane, e)];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const T* k = S + (kW * b + Op::row(lane, s)) * kL + li;
        acc = Op::mma(-k[kW * r], k[kW * c], acc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) C[Op::row(lane, e)] = acc[e];
}

// acc + A B of two 16 x 16 tiles given by their first elements.  The product
// steps take the inner index in the order of the accumulator's rows
// (Op::row(lane, s) in step s), so that an accumulator can be the right
// operand of a following product as it stands (left_product).
template <class T>
__device__ __attribute__((always_inline)) inline typename Mfma<T>::acc_t tile_product(
    const T* A, const T* B, typename Mfma<T>::acc_t acc)
{
    using Op = Mfma<T>;
    const int lane = threadIdx.x & 63, li = lane & 15;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int k = Op::row(lane, s);
        acc = Op::mma(A[k * kL + li], B[li * kL + k], acc);
    }
    return acc;
}

// C = -D t: D and C 16 x 16 tiles in LDS, t an accumulator.
template <class T>
__device__ __attribute__((always_inline)) inline void left_product(const T* D, const typename Mfma<T>::acc_t& t, T* C)
{
    using Op = Mfma<T>;
    const int lane = threadIdx.x & 63, li = lane & 15;
    typename Op::acc_t acc = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = Op::mma(-D[Op::row(lane, s) * kL + li], t[s], acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) C[li * kL + Op::row(lane, e)] = acc[e];
}

// X = L^-1 for the lower triangle of S, rdiag[i] = 1 / L(i, i).  The lower
// triangle of X is complete on return; its strict upper triangle holds
// scratch (callers write zeros there when they store X).
template <class T>
__device__ __attribute__((always_inline)) inline void invert_lower(const T* S, const T* rdiag, T* X)
{
    using Op = Mfma<T>;
    using acc_t = typename Op::acc_t;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    // diagonal 16 x 16 inverses; in wavefront p, lane c < 16 owns column c of D(p)
    {
        const int o = kW * wave;
        T x[kW];
#pragma unroll
        for (int i = 0; i < kW; ++i) {
            T t = (i == lane) ? T(1) : T(0);
#pragma unroll
            for (int k = 0; k < i; ++k) t = fma(-S[(o + k) * kL + o + i], x[k], t);
            x[i] = t * rdiag[o + i];
        }
        if (lane < kW) {
#pragma unroll
            for (int i = 0; i < kW; ++i) X[(o + lane) * kL + o + i] = x[i];
        }
    }
    __syncthreads();
    // X(r, c) = -D(r) L(r, c) D(c) for (r, c) = (1, 0), (3, 2); T = L(r, c) D(c)
    // is staged in the unused block X(c, r)
    const int r2 = 2 * wave + 1, c2 = 2 * wave;
    if (wave < 2) {
        acc_t acc = {0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < kW; ks += 4) {
            const int kk = ks + lk;
            acc = Op::mma(S[(kW * c2 + kk) * kL + kW * r2 + li], X[(kW * c2 + li) * kL + kW * c2 + kk], acc);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) X[(kW * r2 + li) * kL + kW * c2 + Op::row(lane, e)] = acc[e];
    }
    __syncthreads();
    if (wave < 2) {
        acc_t acc = {0, 0, 0, 0};
#pragma unroll
        for (int ks = 0; ks < kW; ks += 4) {
            const int kk = ks + lk;
            acc = Op::mma(-X[(kW * r2 + kk) * kL + kW * r2 + li], X[(kW * r2 + li) * kL + kW * c2 + kk], acc);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) X[(kW * c2 + li) * kL + kW * r2 + Op::row(lane, e)] = acc[e];
    }
    __syncthreads();
    // X21 = -X22 (L21 X11) on 32-row halves; wavefront w owns 16 x 16 tile
    // (a, bc) = (w / 2, w % 2); T = L21 X11 is staged in the unused X[0:32, 32:64]
    const int a = wave >> 1, bc = wave & 1;
    {
        acc_t acc = {0, 0, 0, 0};
        for (int kb = bc; kb < 2; ++kb) {
#pragma unroll
            for (int ks = 0; ks < kW; ks += 4) {
                const int kk = kW * kb + ks + lk;
                acc = Op::mma(S[kk * kL + 32 + kW * a + li], X[(kW * bc + li) * kL + kk], acc);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) X[(32 + kW * bc + li) * kL + kW * a + Op::row(lane, e)] = acc[e];
    }
    __syncthreads();
    {
        acc_t acc = {0, 0, 0, 0};
        for (int kb = 0; kb <= a; ++kb) {
#pragma unroll
            for (int ks = 0; ks < kW; ks += 4) {
                const int kk = kW * kb + ks + lk;
                acc = Op::mma(-X[(32 + kk) * kL + 32 + kW * a + li], X[(32 + kW * bc + li) * kL + kk], acc);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) X[(kW * bc + li) * kL + 32 + kW * a + Op::row(lane, e)] = acc[e];
    }
    __syncthreads();
}

// Factorization of the lower triangle of S in place and, when it succeeds,
// X = L^-1 (its lower triangle; the 16 x 16 blocks above the diagonal are not
// written).  Returns 0 or the 1-based index of the first failed pivot (uniform
// over the workgroup).  Every thread of the workgroup must call it, and it
// ends with a barrier.
template <class T>
__device__ __attribute__((always_inline)) inline int factor_invert64(T* S, T* X, int* s_flag)
{
    const int wave = threadIdx.x >> 6;
    auto s_at = [&](int r, int c) { return S + kW * c * kL + kW * r; };
    auto x_at = [&](int r, int c) { return X + kW * c * kL + kW * r; };
    const typename Mfma<T>::acc_t zero = {0, 0, 0, 0};
    typename Mfma<T>::acc_t t = zero;  // L X product of the block of X that the wavefront forms next
    // strip b beside work() on the wavefronts that have no rows in it; 0 or the failed pivot
    auto pass = [&](auto strip, auto work) -> int {
        constexpr int b = decltype(strip)::value;
        T diag[4];
        if (wave < 4 - b) {
            const int f = factor_strip<T, b>(S, X, diag);
            if (threadIdx.x == 0) *s_flag = f;
        } else {
            work();
        }
        __syncthreads();
        if (wave == 0) store_diagonal<T>(diag, b, S);
        const int f = *s_flag;
        if (f != 0) __syncthreads();
        return f;
    };
    int f = pass(Const<0>(), [] {});
    if (f != 0) return f;
    if (wave < 3) update_tile<T>(S, 0, 1 + wave, 1);
    else t = tile_product<T>(s_at(1, 0), x_at(0, 0), zero);
    __syncthreads();
    f = pass(Const<1>(), [&] {
        update_tile<T>(S, 0, 2, 2);
        update_tile<T>(S, 0, 3, 2);
        update_tile<T>(S, 0, 3, 3);
    });
    if (f != 0) return f;
    if (wave < 2) update_tile<T>(S, 1, 2 + wave, 2);
    else if (wave == 3) left_product<T>(x_at(1, 1), t, x_at(1, 0));
    __syncthreads();
    f = pass(Const<2>(), [&] {
        if (wave == 2) {
            t = tile_product<T>(s_at(2, 1), x_at(1, 0), tile_product<T>(s_at(2, 0), x_at(0, 0), zero));
        } else {
            update_tile<T>(S, 1, 3, 3);
            t = tile_product<T>(s_at(2, 1), x_at(1, 1), zero);
        }
    });
    if (f != 0) return f;
    if (wave == 0) update_tile<T>(S, 2, 3, 3);
    else if (wave > 1) left_product<T>(x_at(2, 2), t, x_at(2, wave - 2));
    __syncthreads();
    f = pass(Const<3>(), [&] {
        t = zero;
        for (int k = wave - 1; k < 3; ++k) t = tile_product<T>(s_at(3, k), x_at(k, wave - 1), t);
    });
    if (f != 0) return f;
    if (wave > 0) left_product<T>(x_at(3, 3), t, x_at(3, wave - 1));
    __syncthreads();
    return 0;
}

// The same as an out-of-line function, for kernels whose register budget
// cannot hold it inlined (it would spill there).
template <class T>
__device__ __attribute__((noinline)) int factor_invert64_call(T* S, T* X, int* s_flag)
{
    return factor_invert64<T>(S, X, s_flag);
}

// Copies the referenced triangle of the w x w diagonal block at A (uplo
// L: A[r + c * lda], r >= c; uplo U: A[c + r * lda]) into the lower triangle
// of S, zeros above it and the identity beyond order w.
template <class T>
__device__ void load_block(bool upper, int w, const T* A, long long lda, T* S)
{
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int fast = idx & (kB - 1), slow = idx >> 6;
        const int r = upper ? slow : fast, c = upper ? fast : slow;
        T v = T(0);
        if (r < w && c < w) {
            if (r >= c) v = upper ? A[c + (long long)r * lda] : A[r + (long long)c * lda];
        } else if (r == c) {
            v = T(1);
        }
        S[c * kL + r] = v;
    }
}

// Writes the lower triangle of S (order w) back to the referenced triangle at A.
template <class T>
__device__ void store_factor(bool upper, int w, const T* S, T* A, long long lda)
{
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int fast = idx & (kB - 1), slow = idx >> 6;
        const int r = upper ? slow : fast, c = upper ? fast : slow;
        if (r < w && c < w && r >= c) {
            if (upper) A[c + (long long)r * lda] = S[c * kL + r];
            else A[r + (long long)c * lda] = S[c * kL + r];
        }
    }
}

// Stores X as a full 64 x 64 column-major block (leading dimension 64) with
// exact zeros above the diagonal.
template <class T>
__device__ void store_inverse(const T* X, T* inv)
{
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int r = idx & (kB - 1), c = idx >> 6;
        inv[idx] = r >= c ? X[c * kL + r] : T(0);
    }
}

} // namespace potf2_detail
} // namespace kern
} // namespace ddla
