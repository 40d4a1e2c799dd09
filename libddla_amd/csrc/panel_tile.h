// One block column (panel) of the blocked Cholesky factorization in a single
// persistent launch (device code, included by kernels.hip and zkernels.hip),
// real or complex Hermitian (^T below is ^H then).
//
// The panel is columns [k, k + kb) of the lower triangle, rows k .. n-1, cut
// into 64 x 64 blocks: P = ceil(kb / 64) <= 64 block columns and R = ceil((n -
// k) / 64) block rows.  It may be the whole rest of the matrix (P = R).  The
// work is cut into units, one workgroup each, taken in order from a ticket
// counter: the diagonal unit 0, then for c = 0, 1, .. P - 1
//   * the diagonal unit c + 1 (if c + 1 < P): blocks (c + 1, c) and (c + 1, c + 1);
//   * one unit for each other block (t, c) of the column, t < R.
// Block (t, c) is formed left-looking,
//     acc = A(t, c) - sum_{i < c} L(t, i) L(c, i)^T,    L(t, c) = acc D_c^T,
// D_c = L(c, c)^-1, as the blocks of rows t and c are published (a flag each;
// the blocks of step i + 1 in flight while step i is multiplied).  A diagonal
// unit t forms A(t, t) - sum_i L(t, i) L(t, i)^T beside that, from the same blocks, and
// factors and inverts its diagonal block in LDS (potf2_tile.h).  A unit waits
// only on units with smaller tickets, which are running or done, so the panel
// always progresses; each wait is still bounded (spin limit -> error word, and
// the panel is abandoned).  A failed pivot sets *info and a failure flag that
// releases every waiter.
//
// What bounds a panel is the chain from D_c to D_{c+1}: publish D_c, read it, one
// product with the triangular D_c (10 of 16 tiles), one rank update of the lower
// diagonal block (10 of 16 tiles), the 64 x 64 factorization; everything else is
// off it: the accumulations are done when D_c arrives, and L(c + 1, c) is
// acknowledged and flagged inside the factorization.  With one workgroup a block row, the accumulations
// of the lower rows (up to P - 1 products a block, ~5 us each with their loads)
// outlasted the chain's step: from block to block 18 us at the first, 40 us at
// the eighth (FP64).
//
// Publication: the blocks and the D_c are written with agent-scope stores, which go through the L2 to the
// coherence point; every wavefront waits until its stores are acknowledged, the
// workgroup meets at a barrier, and one thread stores the flag.  No L2
// write-back is needed (a release fence writes back every dirty line of the
// XCD's L2, the trailing update's running beside the panel among them).  Readers
// poll relaxed and read published blocks with agent-scope loads (never served
// from a stale L1 or L2 line).
#pragma once
#include <hip/hip_runtime.h>

#include "gemm_tile.h"
#include "potf2_tile.h"

namespace ddla {
namespace kern {
namespace panel_detail {

using gemm_detail::Mfma;
using potf2_detail::clear;
using potf2_detail::kB;
using potf2_detail::kL;
using potf2_detail::kPlane;
using potf2_detail::load_planes;
using potf2_detail::tile_acc;
using namespace field;

constexpr int kMaxCols = 64;  // block columns per panel (the flags of a row fit one wavefront)

// Counters of a factorization of nb block rows, per block column; a panel of P
// columns and R rows uses 2 + R P of its P times as many: [0] ticket, [1]
// failure, [2 + P t + c] block (t, c) published.
constexpr int sync_ints(int nb) { return nb + 2; }
constexpr int kPer = kB * kB / 256;

template <class T>
struct PanelArgs {
    T* A;
    long long lda;
    int n, k, kb;
    int* info;       // device info: the panel is skipped if nonzero on entry; receives k + 64 t + j (1-based),
                     // or kInfoWaitLimit when a wait gave up
    T* inv;          // the inverses D_c, 64 x 64 column-major each
    int* sync;       // this panel's counters, zero on entry
    int* error;      // set to 1 when a wait exceeds spin_limit
    int spin_limit;
    long long bstride;  // grid x = independent problems (fastest, so that their chains advance together), grid
                        // y = units: problem b's A, info, inv, sync and error sit
                        // b * bstride bytes after problem 0's
};

// Agent-scope accesses of one element (complex: its parts, or FP32 both at once).
__device__ __forceinline__ double agent_load(const double* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float agent_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ Cx<double> agent_load(const Cx<double>* p) { return {agent_load(&p->re), agent_load(&p->im)}; }
__device__ __forceinline__ Cx<float> agent_load(const Cx<float>* p)
{
    return __builtin_bit_cast(Cx<float>, agent_load(reinterpret_cast<const double*>(p)));
}
__device__ __forceinline__ void agent_store(double* p, double x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void agent_store(float* p, float x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void agent_store(Cx<double>* p, Cx<double> x)
{
    agent_store(&p->re, x.re);
    agent_store(&p->im, x.im);
}
__device__ __forceinline__ void agent_store(Cx<float>* p, Cx<float> x)
{
    agent_store(reinterpret_cast<double*>(p), __builtin_bit_cast(double, x));
}

template <class T, bool COHERENT>
__device__ __forceinline__ T ld(const T* p)
{
    if constexpr (COHERENT) return agent_load(p);
    else return *p;
}

template <class T, bool COHERENT>
__device__ __forceinline__ void st(T* p, T x)
{
    if constexpr (COHERENT) agent_store(p, x);
    else *p = x;
}

// Element e of this thread's share of a 64 x 64 block: (row, column).  The
// column is the wavefront's, in a scalar register, so that an access is a
// scalar address and the lane's one row offset.
__device__ __forceinline__ int share_row() { return threadIdx.x & (kB - 1); }
__device__ __forceinline__ int share_col(int e) { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) + 4 * e; }

// v = this thread's share of A(i0 .. i0 + rows, j0 .. j0 + cols) (rows, cols >=
// 1).  Loads beyond the block are clamped to its last row or column, so all 16
// are in flight together; put_block drops them (here, that would wait for them).
template <class T, bool COHERENT>
__device__ __forceinline__ void fetch_block(const PanelArgs<T>& a, long long i0, long long j0, int rows, int cols,
                                            T (&v)[kPer])
{
    const unsigned row = min(share_row(), rows - 1);
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const T* column = a.A + i0 + (j0 + min(share_col(e), cols - 1)) * a.lda;
        v[e] = ld<T, COHERENT>(column + row);
    }
}

// v = this thread's share of the published inverse D (column-major 64 x 64);
// the 16 x 16 blocks above its diagonal, which no product reads, are left out.
template <class T>
__device__ __forceinline__ void fetch_inverse(const T* d, T (&v)[kPer])
{
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        v[e] = element<T>(0, 0);
        if ((share_row() >> 4) >= (share_col(e) >> 4)) v[e] = ld<T, true>(d + kB * share_col(e) + (unsigned)share_row());
    }
}

// buf[c * kL + r] = the block's element (r, c), from every thread's share; zero
// from row `rows` and column `cols` on.
template <class T>
__device__ __forceinline__ void put_block(const T (&v)[kPer], int rows, int cols, real_t<T>* buf)
{
    const bool live = share_row() < rows;
#pragma unroll
    for (int e = 0; e < kPer; ++e)
#pragma unroll
        for (int p = 0; p < Field<T>::planes; ++p)
            buf[p * kPlane + share_col(e) * kL + share_row()] =
                live && share_col(e) < cols ? plane(v[e], p) : real_t<T>(0);
}

template <class T>
__device__ __forceinline__ T buffer_element(const real_t<T>* buf, int r, int c)
{
    return element<T>(buf[c * kL + r], buf[(Field<T>::planes - 1) * kPlane + c * kL + r]);
}

// A(i0 + r, j0 + c) = buf[c * kL + r] for r < rows, c < cols.
template <class T, bool COHERENT>
__device__ __forceinline__ void store_block(const PanelArgs<T>& a, long long i0, long long j0, int rows, int cols,
                                   const real_t<T>* buf)
{
    const unsigned r = share_row();
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int c = share_col(e);
        T* column = a.A + i0 + (j0 + c) * a.lda;
        if ((int)r < rows && c < cols) st<T, COHERENT>(column + r, buffer_element<T>(buf, r, c));
    }
}

// STEPS product steps whose N operands come from LDS: the operands of step s + 1
// are read before the products of step s are issued (the scheduling barrier
// keeps them there), so that a step waits for reads issued a step earlier.
// Without it each product waited for its own operands: 2.7 us for the
// triangular product of a block, whose matrix steps take 1.1 (FP64).
template <class T, int STEPS, int N, class Read, class Multiply>
__device__ __forceinline__ void product_steps(Read read, Multiply multiply)
{
    real_t<T> x[2][N][Field<T>::planes];
    read(0, x[0]);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        if (s + 1 < STEPS) read(s + 1, x[(s + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        multiply(x[s & 1]);
    }
}

// The accumulators of a 64 x 64 block: wavefront w owns rows 32 (w / 2) .. + 31
// as two 16-row tiles, and the two 16-column tiles COL(w, 0) and COL(w, 1).
// Accumulator (i, jj), element e of lane l is row 32 (w / 2) + 16 i + row(l, e),
// column 16 COL(w, jj) + l % 16.
template <class T>
struct Acc64 {
    using R = real_t<T>;
    static constexpr int P = Field<T>::planes;
    tile_acc<T> v[2][2];
    // columns 0 and 3, or 1 and 2: the same number of products with a triangular D
    __device__ __forceinline__ static int col_tile(int jj)
    {
        const int w = (threadIdx.x >> 6) & 1;
        return jj == 0 ? w : 3 - w;
    }
    __device__ __forceinline__ void zero()
    {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) clear<T>(v[i][jj]);
    }
    // visit(accumulator element, its place buf[col * kL + row])
    template <class Self, class Visit>
    __device__ __forceinline__ static void each(Self& self, R* buf, Visit visit)
    {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ro = 32 * (wave >> 1);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int pl = 0; pl < P; ++pl)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        visit(self.v[i][jj][pl], e, buf + pl * kPlane + (16 * col_tile(jj) + (lane & 15)) * kL + ro +
                                                        16 * i + Mfma<R>::row(lane, e));
    }
    __device__ __forceinline__ void load(R* buf)
    {
        each(*this, buf, [](auto& acc, int e, R* p) __attribute__((always_inline)) { acc[e] = *p; });
    }
    __device__ __forceinline__ void store(R* buf) const
    {
        each(*this, buf, [](auto& acc, int e, R* p) __attribute__((always_inline)) { *p = acc[e]; });
    }
    // -= As Bs^T (the 64 terms as one sum) with As(row, k) = As[k * kL + row], Bs(col, k) = Bs[k * kL + col]
    __device__ __forceinline__ void subtract_nt(const R* As, const R* Bs)
    {
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, at = (lane >> 4) * kL + (lane & 15);
        const R* ap = As + at + 32 * (wave >> 1);
        const R *b0p = Bs + at + 16 * col_tile(0), *b1p = Bs + at + 16 * col_tile(1);
        Acc64 sum;
        sum.zero();
        product_steps<T, kB / 4, 4>(
            [&](int s, R (&x)[4][P]) {
                load_planes<T>(ap + 4 * kL * s, x[0]);
                load_planes<T>(ap + 4 * kL * s + 16, x[1]);
                load_planes<T>(b0p + 4 * kL * s, x[2]);
                load_planes<T>(b1p + 4 * kL * s, x[3]);
            },
            [&](R (&x)[4][P]) {
                mma_add_conj(x[0], x[2], sum.v[0][0]);
                mma_add_conj(x[0], x[3], sum.v[0][1]);
                mma_add_conj(x[1], x[2], sum.v[1][0]);
                mma_add_conj(x[1], x[3], sum.v[1][1]);
            });
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int pl = 0; pl < P; ++pl) v[i][jj][pl] -= sum.v[i][jj][pl];
    }
    // = As D^T for a lower-triangular D(c, k) = Ds[k * kL + c]: column tile t takes k < 16 (t + 1)
    __device__ __forceinline__ void product_triangular(const R* As, const R* Ds)
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int lane = threadIdx.x & 63, at = (lane >> 4) * kL + (lane & 15);
        const int t0 = wave & 1, t1 = 3 - t0;  // the column tiles: t0 < t1
        const R* ap = As + at + 32 * (wave >> 1);
        const R *b0p = Ds + at + 16 * t0, *b1p = Ds + at + 16 * t1;
        zero();
        // sixteen k at a time
        for (int t = 0; t <= t0; ++t, ap += 16 * kL, b0p += 16 * kL, b1p += 16 * kL)
            product_steps<T, 4, 4>(
                [&](int s, R (&x)[4][P]) {
                    load_planes<T>(ap + 4 * kL * s, x[0]);
                    load_planes<T>(ap + 4 * kL * s + 16, x[1]);
                    load_planes<T>(b0p + 4 * kL * s, x[2]);
                    load_planes<T>(b1p + 4 * kL * s, x[3]);
                },
                [&](R (&x)[4][P]) {
                    mma_add_conj(x[0], x[2], v[0][0]);
                    mma_add_conj(x[0], x[3], v[0][1]);
                    mma_add_conj(x[1], x[2], v[1][0]);
                    mma_add_conj(x[1], x[3], v[1][1]);
                });
        for (int t = t0 + 1; t <= t1; ++t, ap += 16 * kL, b1p += 16 * kL)
            product_steps<T, 4, 3>(
                [&](int s, R (&x)[3][P]) {
                    load_planes<T>(ap + 4 * kL * s, x[0]);
                    load_planes<T>(ap + 4 * kL * s + 16, x[1]);
                    load_planes<T>(b1p + 4 * kL * s, x[2]);
                },
                [&](R (&x)[3][P]) {
                    mma_add_conj(x[0], x[2], v[0][1]);
                    mma_add_conj(x[1], x[2], v[1][1]);
                });
    }
};

// The ten 16 x 16 tiles of a diagonal block's lower triangle over the four
// wavefronts: (0,0) (1,0) (1,1) | (2,0) (2,1) (2,2) | (3,0) (3,1) | (3,2) (3,3).
template <class T>
struct AccLower {
    using R = real_t<T>;
    static constexpr int P = Field<T>::planes;
    tile_acc<T> v[3];
    __device__ __forceinline__ static int row_tile(int i)
    {
        const int w = threadIdx.x >> 6;
        return w == 0 ? (i > 0) : w == 1 ? 2 : 3;
    }
    __device__ __forceinline__ static int col_tile(int i)
    {
        const int w = threadIdx.x >> 6;
        return w == 0 ? (i > 1) : w == 3 ? 2 + i : i;
    }
    __device__ __forceinline__ static int count()
    {
        return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < 2 ? 3 : 2;
    }
    // -= S S^T (as one sum), S(row, k) = S[k * kL + row]
    __device__ __forceinline__ void subtract_square(const R* S)
    {
        const int lane = threadIdx.x & 63;
        const R* p = S + (lane >> 4) * kL + (lane & 15);
        const R *a0 = p + 16 * row_tile(0), *a1 = p + 16 * row_tile(1);
        const R *b0 = p + 16 * col_tile(0), *b1 = p + 16 * col_tile(1), *b2 = p + 16 * col_tile(2);
        tile_acc<T> sum[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) clear<T>(sum[i]);
        if (count() == 3)  // row_tile(2) == row_tile(1)
            product_steps<T, kB / 4, 5>(
                [&](int s, R (&x)[5][P]) {
                    load_planes<T>(a0 + 4 * kL * s, x[0]);
                    load_planes<T>(a1 + 4 * kL * s, x[1]);
                    load_planes<T>(b0 + 4 * kL * s, x[2]);
                    load_planes<T>(b1 + 4 * kL * s, x[3]);
                    load_planes<T>(b2 + 4 * kL * s, x[4]);
                },
                [&](R (&x)[5][P]) {
                    mma_add_conj(x[0], x[2], sum[0]);
                    mma_add_conj(x[1], x[3], sum[1]);
                    mma_add_conj(x[1], x[4], sum[2]);
                });
        else
            product_steps<T, kB / 4, 4>(
                [&](int s, R (&x)[4][P]) {
                    load_planes<T>(a0 + 4 * kL * s, x[0]);
                    load_planes<T>(a1 + 4 * kL * s, x[1]);
                    load_planes<T>(b0 + 4 * kL * s, x[2]);
                    load_planes<T>(b1 + 4 * kL * s, x[3]);
                },
                [&](R (&x)[4][P]) {
                    mma_add_conj(x[0], x[2], sum[0]);
                    mma_add_conj(x[1], x[3], sum[1]);
                });
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int pl = 0; pl < P; ++pl) v[i][pl] -= sum[i][pl];
    }
    template <class Self, class Visit>
    __device__ __forceinline__ static void each(Self& self, R* buf, Visit visit)
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (i < count()) {
                R* p = buf + (16 * col_tile(i) + (lane & 15)) * kL + 16 * row_tile(i);
#pragma unroll
                for (int pl = 0; pl < P; ++pl)
#pragma unroll
                    for (int e = 0; e < 4; ++e) visit(self.v[i][pl], e, p + pl * kPlane + Mfma<R>::row(lane, e));
            }
    }
    __device__ __forceinline__ void load(R* buf)
    {
#pragma unroll
        for (int i = 0; i < 3; ++i) clear<T>(v[i]);
        each(*this, buf, [](auto& acc, int e, R* p) __attribute__((always_inline)) { acc[e] = *p; });
    }
    __device__ __forceinline__ void store(R* buf) const
    {
        each(*this, buf, [](auto& acc, int e, R* p) __attribute__((always_inline)) { *p = acc[e]; });
    }
};

// Units of a panel of P block columns and R block rows.
__host__ __device__ inline int panel_units(int P, int R)
{
    return (P - 1) * (R - 1) - (P - 1) * (P - 2) / 2 + 1 + R - P;
}

// Workgroups per CU that the registers are sized for: 2 leaves a lane 256, so
// that two units, or one and a workgroup of the trailing update running beside
// the panel (256 registers, 74 KB of LDS), fit on a CU; FP64 complex blocks fill
// the LDS by themselves.
template <class T>
constexpr int panel_occupancy()
{
    return sizeof(T) == 16 ? 1 : 2;
}

template <class T>
__global__ __launch_bounds__(256, panel_occupancy<T>()) void panel_kernel(PanelArgs<T> a)
{
    using R = real_t<T>;
    __shared__ R S[Field<T>::planes * kPlane], X[Field<T>::planes * kPlane];
    __shared__ int s_ticket, s_flag, s_ready;
    const int tid = threadIdx.x, lane = tid & 63;
    if (gridDim.x > 1) {
        const long long off = (long long)blockIdx.x * a.bstride;
        a.A = reinterpret_cast<T*>(reinterpret_cast<char*>(a.A) + off);
        a.info = reinterpret_cast<int*>(reinterpret_cast<char*>(a.info) + off);
        a.inv = reinterpret_cast<T*>(reinterpret_cast<char*>(a.inv) + off);
        a.sync = reinterpret_cast<int*>(reinterpret_cast<char*>(a.sync) + off);
        a.error = reinterpret_cast<int*>(reinterpret_cast<char*>(a.error) + off);
    }
    int* const failed = a.sync + 1;
    int* const flags = a.sync + 2;

    const int P = (a.kb + kB - 1) / kB, rows = (a.n - a.k + kB - 1) / kB;
    auto row_of = [&](int t) { return (long long)a.k + (long long)kB * t; };
    auto rows_in = [&](int t) { return (int)min((long long)kB, (long long)a.n - row_of(t)); };

    // The leading blocks i <= c of which L(t, i) and L(c, i) are published; c + 1
    // when D_c is too; or -1 if the panel failed.  Wavefront 0, in one round trip:
    // lane i < c reads both flags, lane c that of D_c, the lanes from c on the
    // failure flag.
    auto read_flags = [&](int t, int c, int& f, int& g) __attribute__((always_inline)) {
        const int* p = flags + (long long)P * c + min(lane, c);
        const int* q = lane >= c ? failed : flags + (long long)P * t + lane;
        f = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        g = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto count_published = [&](int c, int f, int g) __attribute__((always_inline)) -> int {
        if (__ballot(lane >= c && g != 0) != 0) return -1;
        const unsigned long long missing = ~__ballot(lane <= c && f != 0 && (lane == c || g != 0));
        return missing == 0 ? 64 : (int)__builtin_ctzll(missing);
    };
    // Waits until that count is >= need and returns it (uniform), or -1: the panel
    // failed, or the spin limit (error word set).  Every call is followed by a
    // barrier before s_ready is written again.
    auto wait_published = [&](int t, int c, int need) __attribute__((always_inline)) -> int {
        if (tid < 64) {
            int ready, spins = 0;
            for (;;) {
                int f, g;
                read_flags(t, c, f, g);
                ready = count_published(c, f, g);
                if (ready < 0 || ready >= need) break;
                if (++spins > a.spin_limit) {
                    ready = -1;
                    if (tid == 0) {
                        atomicExch(a.error, 1);
                        // the factor is not valid: the device info says so too
                        // (unless a failed pivot was recorded first), and every
                        // later panel and update of this factorization is skipped
                        atomicCAS(a.info, 0, kInfoWaitLimit);
                        atomicExch(failed, 1);
                    }
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (tid == 0) s_ready = ready;
        }
        __syncthreads();
        return __builtin_amdgcn_readfirstlane(s_ready);
    };
    auto set_flag = [&](int t, int c) {
        __hip_atomic_store(flags + (long long)P * t + c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    T vs[kPer], vx[kPer];  // the blocks in flight
    AccLower<T> dacc;      // A(t, t) - sum_i L(t, i) L(t, i)^T of a diagonal unit

    // S = L(t, c), in LDS only; diag: dacc as well, which lacks L(t, c)'s part.
    // The accumulators start from A and take the 64 terms of each block as one sum:
    // the roundings shrink with the Schur complement, and its scale rounds once in
    // 64 terms.  FP64 solutions with a smooth kernel matrix of order 4096 are off by
    // 3.1e-13 so, by 1.8e-12 if A is added to one long sum (an elementwise
    // factorization: 8.8e-13); complex64 factors of order 4500 by 5.0e-8, by more than
    // 2e-7 if every term rounds at the scale of A.  False: the panel was abandoned.
    auto form_block = [&](int t, int c, bool diag) __attribute__((always_inline)) -> bool {
        const long long rt = row_of(t), rc = row_of(c);
        const int ht = rows_in(t), wc = min(kB, a.kb - kB * c);
        const T* const dc = a.inv + (long long)c * kB * kB;
        Acc64<T> acc;
        int ready = 0;
        bool have_inverse = false;
        fetch_block<T, false>(a, rt, rc, ht, wc, vs);
        if (diag) fetch_block<T, false>(a, rt, rt, ht, ht, vx);
        put_block(vs, ht, wc, S);
        if (diag) put_block(vx, ht, ht, X);
        __syncthreads();
        if (diag) dacc.load(X);
        if (c > 0) {
            acc.load(S);
            ready = wait_published(t, c, 1);  // with a barrier: S and X are read
            if (ready < 0) return false;
            fetch_block<T, true>(a, rt, a.k, ht, kB, vs);
            fetch_block<T, true>(a, rc, a.k, wc, kB, vx);
        }
        for (int i = 0; i < c; ++i) {
            const long long ci = row_of(i + 1);
            put_block(vs, ht, kB, S);
            put_block(vx, wc, kB, X);
            __syncthreads();
            const bool more = i + 1 < c, fetched = more && ready >= i + 2, look = ready <= c;
            int f = 0, g = 0;
            if (look && tid < 64) read_flags(t, c, f, g);
            if (fetched) {
                fetch_block<T, true>(a, rt, ci, ht, kB, vs);
                fetch_block<T, true>(a, rc, ci, wc, kB, vx);
            } else if (!more) {
                have_inverse = ready > c;
                if (have_inverse) fetch_inverse(dc, vx);
            }
            acc.subtract_nt(S, X);
            if (diag) dacc.subtract_square(S);
            if (look && tid < 64) {
                const int now = count_published(c, f, g);
                if (tid == 0) s_ready = now;
            }
            __syncthreads();
            if (look) ready = __builtin_amdgcn_readfirstlane(s_ready);
            if (ready < 0) return false;
            if (more && !fetched) {
                if (ready < i + 2) {
                    __syncthreads();  // s_ready has been read
                    ready = wait_published(t, c, i + 2);
                    if (ready < 0) return false;
                }
                fetch_block<T, true>(a, rt, ci, ht, kB, vs);
                fetch_block<T, true>(a, rc, ci, wc, kB, vx);
            }
        }
        if (c > 0) acc.store(S);
        if (!have_inverse) {
            if (ready <= c) {
                __syncthreads();  // s_ready has been read
                if (wait_published(t, c, c + 1) < 0) return false;
            }
            fetch_inverse(dc, vx);
        }
        put_block(vx, kB, kB, X);
        __syncthreads();
        acc.product_triangular(S, X);  // L(t, c) = acc D_c^T
        __syncthreads();
        acc.store(S);
        __syncthreads();
        return true;
    };

    if (tid == 0) {
        s_ticket = atomicAdd(a.sync, 1);
        s_flag = __hip_atomic_load(a.info, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (s_flag != 0) return;  // an earlier panel (or this one) failed
    // uniform, in scalar registers: every address below depends on it
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    // block (t, c); diag: of the diagonal unit t
    int c = 0, t = 0;
    bool diag = true;
    if (ticket > 0) {
        int u = ticket - 1;
        while (c < P - 1 && u >= rows - c - 1) {
            u -= rows - c - 1;
            ++c;
        }
        t = c + 1 + u;
        diag = u == 0 && c < P - 1;
    }
    const long long r0 = row_of(t);
    const int h = rows_in(t);
    if (t == 0) {
        fetch_block<T, false>(a, r0, r0, h, h, vs);
        put_block(vs, h, h, X);
        __syncthreads();
    } else {
        if (!form_block(t, c, diag)) return;
        store_block<T, true>(a, r0, row_of(c), h, kB, S);
        if (!diag) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (tid == 0) set_flag(t, c);
            return;
        }
        dacc.subtract_square(S);
        dacc.store(X);
        __syncthreads();
    }
    // diagonal block t (order h); the identity beyond h
    if (h < kB) {
        if (tid >= h && tid < kB) X[tid * kL + tid] = 1;
        __syncthreads();
    }
    // L(t, t - 1)'s stores are acknowledged during the first strip and flagged after it
    const int fail = potf2_detail::factor_invert64<T>(
        X, S, &s_flag, [] { __builtin_amdgcn_s_waitcnt(0); },
        [&] {
            if (t > 0 && tid == 255) set_flag(t, t - 1);
        });
    if (fail != 0) {
        potf2_detail::store_factor<T>(false, h, X, a.A + r0 + r0 * a.lda, a.lda);
        if (tid == 0) {
            atomicExch(a.info, (int)r0 + fail);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            atomicExch(failed, 1);
        }
        return;
    }
    T* const dt = a.inv + (long long)t * kB * kB;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int r = share_row(), col = share_col(e);
        if ((r >> 4) >= (col >> 4))
            st<T, true>(dt + kB * col + (unsigned)r, r >= col ? buffer_element<T>(S, r, col) : element<T>(0, 0));
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) set_flag(t, t);
    potf2_detail::store_factor<T>(false, h, X, a.A + r0 + r0 * a.lda, a.lda);
}

} // namespace panel_detail
} // namespace kern
} // namespace ddla
