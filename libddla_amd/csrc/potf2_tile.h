// Cholesky factorization and triangular inverse of one 64 x 64 diagonal block
// held in LDS, for a 256-thread workgroup on gfx950 (device code, included by
// kernels.hip and zkernels.hip), real or complex Hermitian.
//
// The block S is column-major in LDS with column stride kL (S[c * kL + r] =
// A(r, c); of a complex block the real parts, kPlane elements before the
// imaginary ones) and only its lower triangle is referenced, of its diagonal
// only the real part.  It is factored in
// 16-column strips, the inverse X = L^-1 growing beside it:
//   * a strip is factored four columns at a time on the matrix cores
//     (factor_strip).  Every wavefront keeps the strip's 16 x 16 diagonal
//     block and one 16 x 16 block of its own (rows below; wavefront 0: the
//     identity) in the accumulator layout, in which the four columns of a step
//     are one register and, as they stand, both operands of the 16x16x4
//     product that applies them to the later columns.  The step's 4 x 4
//     diagonal block is factored by every lane redundantly, and every lane
//     finishes the four columns of its row by substitution, so neither a pivot's
//     chain to the next one nor the strip has any exchange between wavefronts in
//     it, and the pass turns the identity into L(b, b)^-T, the inverse of the
//     strip's diagonal block (multiplied by an explicit inverse of the 4 x 4
//     block instead, in 7.3 and 5.1 us a block, the columns of a nearly singular one were
//     off by 47 n eps instead of 0.5, pivots among them down to negative ones in
//     a factor reported complete, and a NaN pivot reached the columns before it);
//   * between two passes the strip is applied to the next strip's columns
//     (update_tile), and to the columns beyond while the next pass runs; the
//     wavefronts that have no rows left in a strip also form, during the
//     passes, the 16 x 16 products of the inverse, X(r, c) = -D(r) sum_k
//     L(r, k) X(k, c).
// What bounds it is the dependency chain of 64 pivots; after the last strip
// only one 16 x 16 product is left of the inverse.  Measured on one workgroup,
// factor and inverse of a block: FP64 13.4 -> 7.6 us, FP32 9.6 -> 5.4 us against
// strips factored column by column in one wavefront (pivots and multipliers
// through v_readlane) with the inverse formed afterwards.
#pragma once
#include <hip/hip_runtime.h>

#include "field.h"
#include "gemm_tile.h"

namespace ddla {
namespace kern {
namespace potf2_detail {

using gemm_detail::Mfma;
using namespace field;

constexpr int kB = 64;           // block order
constexpr int kL = 65;           // LDS column stride, in elements
constexpr int kPlane = kB * kL;  // one plane of a block in LDS
constexpr int kW = 16;           // strip width

// A wavefront's accumulators of one 16 x 16 tile of T.
template <class T>
using tile_acc = acc_t<real_t<T>>[Field<T>::planes];

template <class T>
__device__ __forceinline__ void clear(tile_acc<T>& acc)
{
#pragma unroll
    for (int p = 0; p < Field<T>::planes; ++p) acc[p] = acc_t<real_t<T>>{0, 0, 0, 0};
}

// Element idx of a block in LDS, of every plane.
template <class T>
__device__ __forceinline__ void load_planes(const real_t<T>* S, real_t<T> (&v)[Field<T>::planes])
{
#pragma unroll
    for (int p = 0; p < Field<T>::planes; ++p) v[p] = S[p * kPlane];
}

template <int i>
struct Const {
    static constexpr int value = i;
};

__device__ __forceinline__ double lane_value(double x, int l)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ float lane_value(float x, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}

// x where mask is all ones, zero where it is zero (whatever x is).
__device__ __forceinline__ double masked(double x, int mask)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)b & (unsigned)mask, hi = (unsigned)(b >> 32) & (unsigned)mask;
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ float masked(float x, int mask) { return __int_as_float(__float_as_int(x) & mask); }

// x[c] = the v of lane 16 c + l % 16, for every lane l.
__device__ __forceinline__ void gather_columns(unsigned v, unsigned (&x)[4])
{
    // odd rows of sixteen lanes of the first operand against even ones of the second, then the halves likewise
    const auto pairs = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    const auto even = __builtin_amdgcn_permlane32_swap(pairs[0], pairs[0], false, false);
    const auto odd = __builtin_amdgcn_permlane32_swap(pairs[1], pairs[1], false, false);
    x[0] = even[0];
    x[1] = odd[0];
    x[2] = even[1];
    x[3] = odd[1];
}

__device__ __forceinline__ void gather_columns(float v, float (&x)[4])
{
    unsigned u[4];
    gather_columns(__float_as_uint(v), u);
#pragma unroll
    for (int c = 0; c < 4; ++c) x[c] = __uint_as_float(u[c]);
}

__device__ __forceinline__ void gather_columns(double v, double (&x)[4])
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    unsigned lo[4], hi[4];
    gather_columns((unsigned)b, lo);
    gather_columns((unsigned)(b >> 32), hi);
#pragma unroll
    for (int c = 0; c < 4; ++c)
        x[c] = __longlong_as_double((long long)(((unsigned long long)hi[c] << 32) | lo[c]));
}

// 1 / sqrt(d) for d > 0: the hardware estimate and one third-order step (FP64:
// with e = 1 - d y^2, y (1 + e/2 + 3 e^2 / 8); the estimate's ~2^-23 becomes
// ~2^-67, rounding aside) or one Newton step (FP32).
__device__ __forceinline__ double rsqrt_refined(double d)
{
    const double y = __builtin_amdgcn_rsq(d);
    const double e = fma(-(d * y), y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

__device__ __forceinline__ float rsqrt_refined(float d)
{
    float y = __builtin_amdgcn_rsqf(d);
    const float h = 0.5f * d;
    const float e = fmaf(-h * y, y, 0.5f);
    return fmaf(y, e, y);
}

// acc += conj(a) b, one 16x16x4 product.  A complex one adds up by itself first, so
// that acc's scale rounds once a step and not at each of its eight terms: factors of
// order 64 to 1300 are off by 1.2 to 1.6e-16 (complex128) and 6.1 to 8.8e-8
// (complex64) so, by 2.5 to 2.7e-16 and 1.3 to 1.5e-7 otherwise.  (Column by column,
// with one rounding each, 1.8 to 2.1e-16 and 1.0 to 1.1e-7.)  It costs 0.8 % of a
// complex pposv of order 1999.
template <class T>
__device__ __forceinline__ void add_product(const real_t<T> (&a)[Field<T>::planes],
                                            const real_t<T> (&b)[Field<T>::planes], tile_acc<T>& acc)
{
    if constexpr (Field<T>::planes == 1) {
        mma_conj_add(a, b, acc);
    } else {
        tile_acc<T> sum;
        clear<T>(sum);
        mma_conj_add(a, b, sum);
#pragma unroll
        for (int p = 0; p < Field<T>::planes; ++p) acc[p] += sum[p];
    }
}

// Row of the diagonal block that lane l % 16 holds, and the lane that holds
// row r of it: chosen so that register q of the accumulator layout holds
// columns 4q .. 4q + 3 (column 4q + lane / 16) and can serve as the product's
// left operand too.  FP64 accumulators are D[l / 16 + 4r][l % 16], FP32 ones
// D[4 (l / 16) + r][l % 16].
template <class R>
__device__ constexpr int diag_row(int i)
{
    return sizeof(R) == 8 ? i : (i >> 2) + 4 * (i & 3);  // its own inverse
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
__device__ __forceinline__ int factor_strip(real_t<T>* S, real_t<T>* X,
                                                                  real_t<T> (&diag)[4][Field<T>::planes])
{
    using R = real_t<T>;
    constexpr int P = Field<T>::planes;
    constexpr int r0 = kW * b;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int pr = diag_row<R>(li);
    tile_acc<T> d, x;
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = g + 4 * r;
            d[p][r] = masked(S[p * kPlane + (r0 + c) * kL + r0 + pr], -(int)(p == 0 ? pr >= c : pr > c));
            x[p][r] = wave == 0 ? (p == 0 && li == c ? R(1) : R(0))
                                : S[p * kPlane + (r0 + c) * kL + r0 + kW * wave + li];
        }
    R below[4][P];               // the finished columns of x
    unsigned long long bad = 0;  // bit j: the pivot of column j is not positive
    auto check = [&](R v, int j) { bad |= __ballot(!(v > R(0))) & (1ull << j); };
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        auto real_at = [&](int c) { return lane_value(d[0][q], 16 * c + diag_row<R>(4 * q + c)); };
        auto at = [&](int r, int c) {
            const int l = 16 * c + diag_row<R>(4 * q + r);
            return element<T>(lane_value(d[0][q], l), lane_value(d[P - 1][q], l));
        };
        const R a00 = real_at(0), a11 = real_at(1), a22 = real_at(2), a33 = real_at(3);
        const T a10 = at(1, 0), a20 = at(2, 0), a30 = at(3, 0), a21 = at(2, 1), a31 = at(3, 1), a32 = at(3, 2);
        const R y0 = rsqrt_refined(a00);
        const T l10 = scale(a10, y0), l20 = scale(a20, y0), l30 = scale(a30, y0);
        const R d1 = sub_norm(a11, l10), y1 = rsqrt_refined(d1);
        const T l21 = scale(sub_mul_conj(a21, l20, l10), y1), l31 = scale(sub_mul_conj(a31, l30, l10), y1);
        const R d2 = sub_norm(sub_norm(a22, l20), l21), y2 = rsqrt_refined(d2);
        const T l32 = scale(sub_mul_conj(sub_mul_conj(a32, l30, l20), l31, l21), y2);
        const R d3 = sub_norm(sub_norm(sub_norm(a33, l30), l31), l32), y3 = rsqrt_refined(d3);
        check(a00, 4 * q);
        check(d1, 4 * q + 1);
        check(d2, 4 * q + 2);
        check(d3, 4 * q + 3);
        // the four finished columns of every row, W = A L44^-H by substitution: a lane
        // takes the step's elements of its row from the four lanes that hold them
        auto substitute = [&](const tile_acc<T>& block, R (&column)[P]) __attribute__((always_inline)) {
            R v[P][4];
#pragma unroll
            for (int p = 0; p < P; ++p) gather_columns(block[p][q], v[p]);
            auto at = [&](int c) { return element<T>(v[0][c], v[P - 1][c]); };
            const T w0 = scale(at(0), y0);
            const T w1 = scale(sub_mul_conj(at(1), w0, l10), y1);
            const T w2 = scale(sub_mul_conj(sub_mul_conj(at(2), w0, l20), w1, l21), y2);
            const T w3 = scale(sub_mul_conj(sub_mul_conj(sub_mul_conj(at(3), w0, l30), w1, l31), w2, l32), y3);
#pragma unroll
            for (int p = 0; p < P; ++p)
                column[p] = g < 2 ? (g == 0 ? plane(w0, p) : plane(w1, p)) : (g == 2 ? plane(w2, p) : plane(w3, p));
        };
        R next[P];
        substitute(d, diag[q]);
#pragma unroll
        for (int p = 0; p < P; ++p)
            next[p] = masked(-diag[q][p], -(int)(pr >= 4 * q + 4));  // the rows that later columns multiply
        if (q < 3) add_product<T>(next, diag[q], d);
        substitute(x, below[q]);
        if (q < 3) add_product<T>(next, below[q], x);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = g + 4 * r;
            if (wave == 0) X[p * kPlane + (r0 + li) * kL + r0 + c] = p == 0 ? below[r][p] : -below[r][p];
            else S[p * kPlane + (r0 + c) * kL + r0 + kW * wave + li] = below[r][p];
        }
    return bad == 0 ? 0 : r0 + (int)__ffsll(bad);
}

// L(b, b), as factor_strip left it in a wavefront's diag, to S.
template <class T>
__device__ __forceinline__ void store_diagonal(const real_t<T> (&diag)[4][Field<T>::planes],
                                                                     int b, real_t<T>* S)
{
    const int lane = threadIdx.x & 63, pr = diag_row<real_t<T>>(lane & 15);
#pragma unroll
    for (int p = 0; p < Field<T>::planes; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = (lane >> 4) + 4 * r;
            if (pr >= c)
                S[p * kPlane + (kW * b + c) * kL + kW * b + pr] = p == 1 && pr == c ? real_t<T>(0) : diag[r][p];
        }
}

// S(16r.., 16c..) -= L(16r.., strip b) L(16c.., strip b)^H, one 16 x 16 tile by
// one wavefront; of complex elements the strip's terms as one sum (add_product).
template <class T>
__device__ __forceinline__ void update_tile(real_t<T>* S, int b, int r, int c)
{
    using R = real_t<T>;
    using Op = Mfma<R>;
    constexpr int P = Field<T>::planes;
    const int lane = threadIdx.x & 63, li = lane & 15;
    R* C = S + (kW * c + li) * kL + kW * r;
    tile_acc<T> acc, sum;
    clear<T>(sum);
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[p][e] = C[p * kPlane + Op::row(lane, e)];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const R* k = S + (kW * b + Op::row(lane, s)) * kL + li;
        R left[P], right[P];
        load_planes<T>(k + kW * r, left);
        load_planes<T>(k + kW * c, right);
        mma_sub_conj(left, right, P == 1 ? acc : sum);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) C[p * kPlane + Op::row(lane, e)] = P == 1 ? acc[p][e] : acc[p][e] + sum[p][e];
}

// acc += A B of two 16 x 16 tiles given by their first elements.  The product
// steps take the inner index in the order of the accumulator's rows
// (Op::row(lane, s) in step s), so that an accumulator can be the right
// operand of a following product as it stands (left_product).
template <class T>
__device__ __forceinline__ void tile_product(const real_t<T>* A, const real_t<T>* B,
                                                                   tile_acc<T>& acc)
{
    using R = real_t<T>;
    constexpr int P = Field<T>::planes;
    const int lane = threadIdx.x & 63, li = lane & 15;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int k = Mfma<R>::row(lane, s);
        R left[P], right[P];
        load_planes<T>(A + k * kL + li, left);
        load_planes<T>(B + li * kL + k, right);
        mma_add(left, right, acc);
    }
}

// C = -D t: D and C 16 x 16 tiles in LDS, t an accumulator.
template <class T>
__device__ __forceinline__ void left_product(const real_t<T>* D, const tile_acc<T>& t,
                                                                   real_t<T>* C)
{
    using R = real_t<T>;
    using Op = Mfma<R>;
    constexpr int P = Field<T>::planes;
    const int lane = threadIdx.x & 63, li = lane & 15;
    tile_acc<T> acc;
    clear<T>(acc);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        R left[P], right[P];
        load_planes<T>(D + Op::row(lane, s) * kL + li, left);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            left[p] = -left[p];
            right[p] = t[p][s];
        }
        mma_add(left, right, acc);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) C[p * kPlane + li * kL + Op::row(lane, e)] = acc[p][e];
}

// X = L^-1 for the lower triangle of S, rdiag[i] = 1 / L(i, i) (real).  The
// lower triangle of X is complete on return, with zeros above the diagonal in
// its diagonal 16 x 16 blocks; the blocks above those are not written.
template <class T>
__device__ __forceinline__ void invert_lower(const real_t<T>* S, const real_t<T>* rdiag,
                                                                   real_t<T>* X)
{
    using R = real_t<T>;
    constexpr int P = Field<T>::planes;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    auto s_at = [&](int r, int c) { return S + kW * c * kL + kW * r; };
    auto x_at = [&](int r, int c) { return X + kW * c * kL + kW * r; };
    // diagonal 16 x 16 inverses; in wavefront p, lane c < 16 owns column c of D(p)
    {
        const int o = kW * wave;
        T x[kW];
#pragma unroll
        for (int i = 0; i < kW; ++i) {
            T t = element<T>(i == lane ? R(1) : R(0), R(0));
#pragma unroll
            for (int k = 0; k < i; ++k) {
                R l[P];
                load_planes<T>(S + (o + k) * kL + o + i, l);
                t = sub_mul(t, element<T>(l[0], l[P - 1]), x[k]);
            }
            x[i] = scale(t, rdiag[o + i]);
        }
        if (lane < kW) {
#pragma unroll
            for (int i = 0; i < kW; ++i)
#pragma unroll
                for (int p = 0; p < P; ++p) X[p * kPlane + (o + lane) * kL + o + i] = plane(x[i], p);
        }
    }
    __syncthreads();
    // X(r, c) = -D(r) sum_{c <= k < r} L(r, k) X(k, c), one subdiagonal of blocks at a time
#pragma unroll
    for (int s = 1; s < 4; ++s) {
        if (wave + s < 4) {
            tile_acc<T> t;
            clear<T>(t);
            for (int k = wave; k < wave + s; ++k) tile_product<T>(s_at(wave + s, k), x_at(k, wave), t);
            left_product<T>(x_at(wave + s, wave + s), t, x_at(wave + s, wave));
        }
        __syncthreads();
    }
}

// Factorization of the lower triangle of S in place and, when it succeeds,
// X = L^-1 (its lower triangle; the 16 x 16 blocks above the diagonal are not
// written).  Returns 0 or the 1-based index of the first failed pivot (uniform
// over the workgroup).  Every thread of the workgroup must call it, and it
// ends with a barrier.  before() and after() run on every thread around the
// barrier that ends the first strip.
template <class T, class Before, class After>
__device__ __forceinline__ int factor_invert64(real_t<T>* S, real_t<T>* X, int* s_flag,
                                                                     Before before, After after)
{
    const int wave = threadIdx.x >> 6;
    auto s_at = [&](int r, int c) { return S + kW * c * kL + kW * r; };
    auto x_at = [&](int r, int c) { return X + kW * c * kL + kW * r; };
    tile_acc<T> t;  // L X product of the block of X that the wavefront forms next
    clear<T>(t);
    // strip b beside work() on the wavefronts that have no rows in it; 0 or the failed pivot
    auto pass = [&](auto strip, auto work) __attribute__((always_inline)) -> int {
        constexpr int b = decltype(strip)::value;
        real_t<T> diag[4][Field<T>::planes];
        if (wave < 4 - b) {
            const int f = factor_strip<T, b>(S, X, diag);
            if (threadIdx.x == 0) *s_flag = f;
        } else {
            work();
        }
        if (b == 0) before();
        __syncthreads();
        if (b == 0) after();
        if (wave == 0) store_diagonal<T>(diag, b, S);
        const int f = *s_flag;
        if (f != 0) __syncthreads();
        return f;
    };
    int f = pass(Const<0>(), [] {});
    if (f != 0) return f;
    if (wave < 3) update_tile<T>(S, 0, 1 + wave, 1);
    else tile_product<T>(s_at(1, 0), x_at(0, 0), t);
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
        clear<T>(t);
        if (wave == 2) {
            tile_product<T>(s_at(2, 0), x_at(0, 0), t);
            tile_product<T>(s_at(2, 1), x_at(1, 0), t);
        } else {
            update_tile<T>(S, 1, 3, 3);
            tile_product<T>(s_at(2, 1), x_at(1, 1), t);
        }
    });
    if (f != 0) return f;
    if (wave == 0) update_tile<T>(S, 2, 3, 3);
    else if (wave > 1) left_product<T>(x_at(2, 2), t, x_at(2, wave - 2));
    __syncthreads();
    f = pass(Const<3>(), [&] {
        clear<T>(t);
        for (int k = wave - 1; k < 3; ++k) tile_product<T>(s_at(3, k), x_at(k, wave - 1), t);
    });
    if (f != 0) return f;
    if (wave > 0) left_product<T>(x_at(3, 3), t, x_at(3, wave - 1));
    __syncthreads();
    return 0;
}

template <class T>
__device__ __forceinline__ int factor_invert64(real_t<T>* S, real_t<T>* X, int* s_flag)
{
    return factor_invert64<T>(S, X, s_flag, [] {}, [] {});
}

// The same as an out-of-line function, for kernels whose register budget
// cannot hold it inlined (it would spill there).
template <class T>
__device__ __attribute__((noinline)) int factor_invert64_call(real_t<T>* S, real_t<T>* X, int* s_flag)
{
    return factor_invert64<T>(S, X, s_flag);
}

// Copies the referenced triangle of the w x w diagonal block at A (uplo
// L: A[r + c * lda], r >= c; uplo U: conj(A[c + r * lda])) into the lower
// triangle of S, zeros above it and the identity beyond order w.
template <class T>
__device__ void load_block(bool upper, int w, const T* A, long long lda, real_t<T>* S)
{
    using R = real_t<T>;
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int fast = idx & (kB - 1), slow = idx >> 6;
        const int r = upper ? slow : fast, c = upper ? fast : slow;
        T v = element<T>(R(0), R(0));
        if (r < w && c < w) {
            if (r >= c) v = upper ? A[c + (long long)r * lda] : A[r + (long long)c * lda];
        } else if (r == c) {
            v = element<T>(R(1), R(0));
        }
        S[c * kL + r] = plane(v, 0);
        if (Field<T>::planes == 2) S[kPlane + c * kL + r] = upper ? -plane(v, 1) : plane(v, 1);
    }
}

// Writes the lower triangle of S (order w) back to the referenced triangle at A.
template <class T>
__device__ void store_factor(bool upper, int w, const real_t<T>* S, T* A, long long lda)
{
    constexpr int last = (Field<T>::planes - 1) * kPlane;
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int fast = idx & (kB - 1), slow = idx >> 6;
        const int r = upper ? slow : fast, c = upper ? fast : slow;
        if (r < w && c < w && r >= c) {
            if (upper) A[c + (long long)r * lda] = element<T>(S[c * kL + r], -S[last + c * kL + r]);
            else A[r + (long long)c * lda] = element<T>(S[c * kL + r], S[last + c * kL + r]);
        }
    }
}

// Stores X as a full 64 x 64 column-major block (leading dimension 64) with
// exact zeros above the diagonal.
template <class T>
__device__ void store_inverse(const real_t<T>* X, T* inv)
{
    constexpr int last = (Field<T>::planes - 1) * kPlane;
#pragma unroll 4
    for (int e = 0; e < kB * kB / 256; ++e) {
        const int idx = threadIdx.x + 256 * e;
        const int r = idx & (kB - 1), c = idx >> 6;
        inv[idx] = r >= c ? element<T>(X[c * kL + r], X[last + c * kL + r]) : element<T>(0, 0);
    }
}

} // namespace potf2_detail
} // namespace kern
} // namespace ddla
