// Triangular solves with a real Cholesky factor over 128-row blocks, one
// persistent launch per direction (device code, included by kernels.hip).
//
// Forward (L Y = B) and backward (L^T X = Y) substitution, 16 right-hand sides
// (a slab) at a time.  Op(t, q) below is block (t, q) of L, or (q, t) of L
// transposed, with t and q counted in sweep order (backward from the bottom),
// and G_t the inverse of Op(t, t).  Workgroup t of a slab (t from a ticket
// counter) computes
//     acc = B_t - sum_{q < t - 1} Op(t, q) X_q      as the X_q are published,
//     X_t = G_t acc - M X_{t-1},   M = G_t Op(t, t - 1),
// with M (128 x 128) formed in LDS before the loop and G_t acc before X_{t-1}
// arrives, so that the chain from block to block is one hand-over through the
// coherence point and one 128 x 128 x 16 product.  It bounds the sweep up to
// orders where reading L does.  The 64-row sweeps of solve_tile.h pay the
// hand-over (~3 us) twice as often and multiply 64 columns whatever their
// number; 512-row stages (a 512 x 512 product per hand-over, shared by eight
// workgroups that also exchange their accumulators) took 40 us a stage.
//
// The blocks of L go straight from memory into the matrix cores' left operand
// (each is read once per slab): lane l of the wavefront of rows 16 w .. holds
// row l % 16, column column_of(s, l / 16) in step s.  Where Op's rows run along
// stored columns (backward with a lower triangle) the columns of two (FP32: four)
// steps are neighbours, so that a lane reads 16 bytes at a time: one element a load
// took that sweep 1500 us (FP32, n = 16384, 64 right-hand sides; now 690, forward
// 640), FP64 554 us (n = 8192; now 420, forward 370).  A step's register takes the next block's value as soon as
// its product is issued, so a whole block is in flight.
//
// Waiting and publication are the panel kernel's (panel_tile.h): a workgroup
// waits only on smaller tickets, i.e. running workgroups, each wait is bounded
// (the error word then), blocks are written with agent-scope stores, waited
// for before the slab's counter moves, and read with agent-scope loads.
#pragma once
#include <hip/hip_runtime.h>

#include "field.h"
#include "gemm_tile.h"
#include "panel_tile.h"
#include "potf2_tile.h"

namespace ddla {
namespace kern {
namespace wide_detail {

using gemm_detail::Mfma;
using panel_detail::agent_load;
using panel_detail::agent_store;

constexpr int kWB = 128;        // rows of a block
constexpr int kWC = 16;         // right-hand sides of a slab
constexpr int kWThreads = 512;  // eight wavefronts, 16 rows of the block each
constexpr int kML = kWB + 1;    // LDS stride of M's columns
// LDS stride of a solution block's rows: with VW = 2 (FP64) or 4 (FP32), the rows
// column_of(s, 0..3) of a step fall on distinct banks (FP64: two rows a pass)
template <int VW>
constexpr int kXL = VW == 2 ? 24 : VW == 4 ? 20 : kWC + 1;
constexpr int kSteps = kWB / 4;
constexpr int kPer = kWB * kWC / kWThreads;  // elements of a solution block per thread

inline int blocks(int n) { return (n + kWB - 1) / kWB; }
inline int slabs(int nrhs) { return (nrhs + kWC - 1) / kWC; }

template <class T>
struct WideArgs {
    int n, nrhs, nblk, nslab;
    const T* L;  // the factor, L view: L(i, j) = upper ? L[j + i*ldl] : L[i + j*ldl]
    long long ldl;
    const T* E;  // inverses of the 128 x 128 diagonal blocks (wide_inverse_kernel)
    T* B;
    long long ldb;
    int vec;     // L and ldl allow 16-byte loads along a stored column
    int* sync;   // per slab: ticket counter, published blocks; zero on entry
    int* error;  // set to 1 if a wait exceeds spin_limit
    int spin_limit;
};

// acc += the 64 x 64 product A B over k in [k0(tile row, tile column), k1(..)),
// multiples of 16: A(r, k) = A[k * kL + r], B(k, c) = B[c * kL + k].  Wavefront w
// of four: rows 32 (w / 2) .., columns 32 (w % 2) .., as 2 x 2 tiles.
template <class T, class K0, class K1>
__device__ __forceinline__ void product64(const T* A, const T* B, K0 k0, K1 k1, typename Mfma<T>::acc_t (&acc)[2][2])
{
    using potf2_detail::kL;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int rt = 2 * (wave >> 1) + i, ct = 2 * (wave & 1) + j;
            acc[i][j] = typename Mfma<T>::acc_t{0, 0, 0, 0};
            for (int k = k0(rt, ct); k < k1(rt, ct); k += 16)
#pragma unroll
                for (int s = 0; s < 16; s += 4)
                    acc[i][j] = Mfma<T>::mma(A[(k + s + lk) * kL + 16 * rt + li], B[(16 * ct + li) * kL + k + s + lk],
                                             acc[i][j]);
        }
}

// E(block b) = the inverse of L's 128 x 128 diagonal block b, column-major, zeros
// above the diagonal, the identity beyond order n: the 64 x 64 inverses X1, X2
// (potf2_tile.h) and E21 = -X2 (L21 X1).
template <class T>
__global__ __launch_bounds__(256) void wide_inverse_kernel(bool upper, int n, const T* L, long long ldl, T* E)
{
    using namespace potf2_detail;
    __shared__ T S[kPlane], X1[kPlane], X2[kPlane], rdiag[kB];
    const int tid = threadIdx.x;
    const long long j0 = (long long)blockIdx.x * kWB;
    const int w1 = (int)min((long long)kB, n - j0), w2 = (int)max(0LL, min((long long)kB, n - j0 - kB));
    E += (long long)blockIdx.x * kWB * kWB;
    auto invert = [&](int w, long long at, T* X) {
        load_block<T>(upper, w, L + at + at * ldl, ldl, S);
        __syncthreads();
        if (tid < kB) rdiag[tid] = T(1) / S[tid * kL + tid];
        __syncthreads();
        invert_lower<T>(S, rdiag, X);
        __syncthreads();
    };
    invert(w1, j0, X1);
    if (w2 > 0) {
        invert(w2, j0 + kB, X2);
    } else {
        for (int i = tid; i < kB * kB; i += 256) X2[(i >> 6) * kL + (i & 63)] = (i >> 6) == (i & 63) ? T(1) : T(0);
    }
    for (int i = tid; i < kB * kB; i += 256) {
        const int fast = i & (kB - 1), slow = i >> 6, r = upper ? slow : fast, c = upper ? fast : slow;
        T v = T(0);
        if (r < w2) v = upper ? L[(j0 + c) + (j0 + kB + r) * ldl] : L[(j0 + kB + r) + (j0 + c) * ldl];
        S[c * kL + r] = v;
    }
    __syncthreads();
    typename Mfma<T>::acc_t t[2][2];
    product64<T>(S, X1, [](int, int ct) { return 16 * ct; }, [](int, int) { return kB; }, t);
    const int wave = tid >> 6, lane = tid & 63;
    auto store = [&](T* D, int ld, int r0, T sign) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    D[(16 * (2 * (wave & 1) + j) + (lane & 15)) * ld + r0 + 16 * (2 * (wave >> 1) + i) +
                      Mfma<T>::row(lane, e)] = sign * t[i][j][e];
    };
    __syncthreads();
    store(S, kL, 0, T(1));
    __syncthreads();
    product64<T>(X2, S, [](int, int) { return 0; }, [](int rt, int) { return 16 * (rt + 1); }, t);
    store(E, kWB, kB, T(-1));
    for (int i = tid; i < kB * kB; i += 256) {
        const int r = i & (kB - 1), c = i >> 6;
        E[r + c * kWB] = r >= c ? X1[c * kL + r] : T(0);
        E[kB + r + (kB + c) * kWB] = r >= c ? X2[c * kL + r] : T(0);
        E[r + (kB + c) * kWB] = T(0);
    }
}

// Grid: nslab * nblk workgroups, slabs fastest, so that all slabs advance together.
// DIRECT: Op(t, q)'s rows run along a stored column, else along a stored row
// (BACKWARD == upper; with both in one kernel FP64's forward sweep spilled with a lower
// factor too: 400 us where it takes 370, n = 8192.  With an upper one it still keeps 20
// registers in memory).
template <class T, bool BACKWARD, bool DIRECT>
__global__ __launch_bounds__(kWThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void wide_sweep_kernel(
    WideArgs<T> a)
{
    using Op = Mfma<T>;
    __shared__ T Ms[kWB * kML];  // [k][row] of M
    constexpr int VW = DIRECT ? 1 : Op::kVec, kXL = wide_detail::kXL<VW>;
    using vec_t = typename Op::vec_t;
    __shared__ T Xs[kWB * kXL];  // [k][column] of a solution block
    __shared__ int s_ticket, s_seen;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // row tile of the wavefront: the triangular products of the two wavefronts
    // of a SIMD (w and w + 4) are equally long together
    const int tile = wave < 4 ? wave : 11 - wave;
    const int slab = blockIdx.x % a.nslab, c0 = slab * kWC, nc = min(kWC, a.nrhs - c0);
    int* const done = a.sync + 2 * slab + 1;
    if (tid == 0) s_ticket = atomicAdd(a.sync + 2 * slab, 1);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_ticket);
    auto block_of = [&](int q) { return BACKWARD ? a.nblk - 1 - q : q; };
    const int bt = block_of(t);
    const long long r0 = (long long)bt * kWB;
    const int w = (int)min((long long)kWB, a.n - r0);
    constexpr bool direct = DIRECT;

    // the term that lane quarter q takes in step s; steps 4 b .. 4 b + 3 take the
    // columns 16 b .. 16 b + 15
    auto column_of = [](int s, int q) { return 4 * VW * (s / VW) + VW * q + s % VW; };
    T f[kSteps];  // left operand: (row 16 tile + li, columns column_of(s, lk)) of a block
    const long long row = r0 + min(16 * tile + li, w - 1);
    // element (row, k) of Op(t, q), k < n - q0
    auto factor = [&](long long q0, int k) {
        return direct ? a.L[row + (q0 + k) * a.ldl] : a.L[(q0 + k) + row * a.ldl];
    };
    const bool wide_loads = !direct && a.vec;
    // the lane's place in column 0; the rest of an address is uniform
    const T* const lane_at = direct ? a.L + row + (long long)(VW * lk) * a.ldl : a.L + row * a.ldl + VW * lk;
    const long long step_stride = direct ? a.ldl : 1;
    // f[s ..  s + VW) of the block at q0, whole
    auto fetch_steps = [&](bool wide, long long q0, int s) __attribute__((always_inline)) {
        const T* p = lane_at + (q0 + column_of(s, 0)) * step_stride;
        if (VW > 1 && wide) {
            const vec_t v = *reinterpret_cast<const vec_t*>(p);
#pragma unroll
            for (int i = 0; i < VW; ++i) f[s + i] = v[i];
        } else {
#pragma unroll
            for (int i = 0; i < VW; ++i) f[s + i] = p[i * step_stride];
        }
    };
    auto fetch_factor = [&](int q) {
        const long long q0 = (long long)block_of(q) * kWB;
        const int wq = (int)min((long long)kWB, a.n - q0);
        if (wq == kWB) {
#pragma unroll
            for (int s = 0; s < kSteps; s += VW) fetch_steps(false, q0, s);
        } else {
#pragma unroll
            for (int s = 0; s < kSteps; ++s) f[s] = factor(q0, min(column_of(s, lk), wq - 1));
        }
    };
    T vx[kPer];
    const int xk = tid & (kWB - 1), xc = tid >> 7;  // this thread's row and first column of a solution block
    auto fetch_solution = [&](int q) {
        const long long q0 = (long long)block_of(q) * kWB;
        const long long at = q0 + min((long long)xk, a.n - 1 - q0);
#pragma unroll
        for (int e = 0; e < kPer; ++e) vx[e] = agent_load(a.B + at + (long long)(c0 + min(xc + 4 * e, nc - 1)) * a.ldb);
    };
    auto put_solution = [&](int q) {
        const bool live = (long long)block_of(q) * kWB + xk < a.n;
#pragma unroll
        for (int e = 0; e < kPer; ++e) Xs[xk * kXL + xc + 4 * e] = live && xc + 4 * e < nc ? vx[e] : T(0);
    };
    // progress of the slab, at least `need` blocks published (uniform); false: the wait limit
    int seen = 0;
    auto wait_for = [&](int need) -> bool {
        if (seen >= need) return true;
        if (tid == 0) {
            int d, spins = 0;
            while ((d = __hip_atomic_load(done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) < need) {
                if (++spins > a.spin_limit) {
                    d = -1;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            s_seen = d;
        }
        __syncthreads();
        seen = __builtin_amdgcn_readfirstlane(s_seen);
        return seen >= 0;
    };

    // f[s .. s + VW) of G_t = E or E^T; out = G_t Xs over the columns that its
    // triangle holds, with G_t in f
    auto fetch_inverse = [&](int s) __attribute__((always_inline)) {
        const T* e = a.E + (long long)bt * kWB * kWB;
        const int r = 16 * tile + li, k = column_of(s, lk);
        if constexpr (BACKWARD && VW > 1) {
            const vec_t v = *reinterpret_cast<const vec_t*>(e + k + r * kWB);
#pragma unroll
            for (int i = 0; i < VW; ++i) f[s + i] = v[i];
        } else {
#pragma unroll
            for (int i = 0; i < VW; ++i) f[s + i] = BACKWARD ? e[k + i + r * kWB] : e[r + (k + i) * kWB];
        }
    };
    auto triangular_product = [&]() {
        typename Op::acc_t out = {0, 0, 0, 0};
#pragma unroll
        for (int b = 0; b < kWB / 16; ++b)
            if (BACKWARD ? b >= tile : b <= tile)
#pragma unroll
                for (int s = 4 * b; s < 4 * b + 4; ++s) out = Op::mma(f[s], Xs[column_of(s, lk) * kXL + li], out);
        return out;
    };
#pragma unroll
    for (int s = 0; s < kSteps; s += VW) fetch_inverse(s);
    if (t >= 1) {
        // M, sixteen columns at a time through Xs
        const long long p0 = (long long)block_of(t - 1) * kWB;
        const int wp = (int)min((long long)kWB, a.n - p0);
        auto fetch_part = [&](int part) {
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                // (k, column) of Op(t, t - 1): along a stored column or row
                const int k = direct ? (tid & (kWB - 1)) : (tid >> 4) + 32 * e;
                const int c = kWC * part + (direct ? (tid >> 7) + 4 * e : (tid & 15));
                const long long i = r0 + min(k, w - 1), j = p0 + min(c, wp - 1);
                vx[e] = direct ? a.L[i + j * a.ldl] : a.L[j + i * a.ldl];
            }
        };
        fetch_part(0);
        for (int part = 0; part < kWB / kWC; ++part) {
            __syncthreads();
#pragma unroll
            for (int e = 0; e < kPer; ++e) {
                const int k = direct ? (tid & (kWB - 1)) : (tid >> 4) + 32 * e;
                const int c = direct ? (tid >> 7) + 4 * e : (tid & 15);
                Xs[k * kXL + c] = k < w && kWC * part + c < wp ? vx[e] : T(0);
            }
            __syncthreads();
            if (part + 1 < kWB / kWC) fetch_part(part + 1);
            const typename Op::acc_t m = triangular_product();
#pragma unroll
            for (int r = 0; r < 4; ++r) Ms[(kWC * part + li) * kML + 16 * tile + Op::row(lane, r)] = m[r];
        }
        __syncthreads();
    }
    typename Op::acc_t acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * tile + Op::row(lane, r);
        acc[r] = i < w && li < nc ? a.B[(r0 + i) + (long long)(c0 + li) * a.ldb] : T(0);
    }
    bool failed = false, have_x = false;
    if (t > 1) fetch_factor(0);
    for (int q = 0; q < t - 1; ++q) {
        if (!have_x) {
            if (!wait_for(q + 1)) {
                failed = true;
                break;
            }
            fetch_solution(q);
        }
        put_solution(q);
        __syncthreads();
        have_x = q + 1 < t - 1 && seen >= q + 2;
        if (have_x) fetch_solution(q + 1);
        if (q + 1 < t - 1) {
            // block q + 1 replaces block q in f step by step (only the sweep's
            // first block can be short of 128 columns)
            const long long q0 = (long long)block_of(q + 1) * kWB;
            auto steps = [&](bool wide) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < kSteps; s += VW) {
#pragma unroll
                    for (int i = 0; i < VW; ++i)
                        acc = Op::mma(-f[s + i], Xs[column_of(s + i, lk) * kXL + li], acc);
                    fetch_steps(wide, q0, s);
                }
            };
            if (wide_loads) steps(true);
            else steps(false);
        } else {  // G_t replaces the last block
#pragma unroll
            for (int s = 0; s < kSteps; s += VW) {
#pragma unroll
                for (int i = 0; i < VW; ++i)
                    acc = Op::mma(-f[s + i], Xs[column_of(s + i, lk) * kXL + li], acc);
                fetch_inverse(s);
            }
        }
        __syncthreads();
    }
    // acc = G_t acc (rows beyond the order are zero), then minus M X_{t-1}
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * tile + Op::row(lane, r);
        Xs[i * kXL + li] = i < w ? acc[r] : T(0);
    }
    __syncthreads();
    acc = triangular_product();
    __syncthreads();
    if (t >= 1 && !failed) {
        if (!wait_for(t)) {
            failed = true;
        } else {
            fetch_solution(t - 1);
            put_solution(t - 1);
            __syncthreads();
            const T* m = Ms + 16 * tile + li;
#pragma unroll 8
            for (int s = 0; s < kSteps; ++s)
                acc = Op::mma(-m[column_of(s, lk) * kML], Xs[column_of(s, lk) * kXL + li], acc);
            __syncthreads();
        }
    }
    if (failed && tid == 0) atomicExch(a.error, 1);
    // X_t leaves through LDS, along the columns
#pragma unroll
    for (int r = 0; r < 4; ++r) Xs[(16 * tile + Op::row(lane, r)) * kXL + li] = acc[r];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int c = xc + 4 * e;
        if (xk < w && c < nc) agent_store(a.B + (r0 + xk) + (long long)(c0 + c) * a.ldb, Xs[xk * kXL + c]);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) __hip_atomic_store(done, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace wide_detail
} // namespace kern
} // namespace ddla
