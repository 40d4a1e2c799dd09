// Triangular solves with a complex Cholesky factor, one persistent launch per
// direction (device code, included by zkernels.hip).
//
// Forward (L Y = B) and backward (L^H X = Y) substitution over 64-row blocks,
// 16 right-hand sides (a slab) at a time.  Workgroup t of a slab (t from a
// ticket counter) solves block t of the sweep (from the top forward, from the
// bottom backward): it accumulates acc = B_t - sum_{q < t} L(t, q) X_q
// (backward L(q, t)^H) as the blocks X_q are published, the factor's next block
// in flight meanwhile, and ends with
//     X_t = D acc - (D L(t, t-1)) X_{t-1},
// both products with D, the inverse of its diagonal block, formed before
// X_{t-1} arrives, so that one 64 x 64 x 16 product is left on the chain from
// block to block.  That chain bounds the sweep: about one hand-over through the
// coherence point and one product per block.
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

namespace ddla {
namespace kern {
namespace zsolve_detail {

using gemm_detail::Mfma;
using panel_detail::agent_load;
using panel_detail::agent_store;
using namespace field;

constexpr int kSB = 64;        // rows of a block
constexpr int kSC = 16;        // right-hand sides of a slab
constexpr int kSThreads = 256; // four wavefronts, 16 rows of the block each
constexpr int kSL = kSB + 1;   // LDS stride of a factor block's column
constexpr int kXL = kSC + 1;   // LDS stride of a solution block's row
constexpr int kFactorPlane = kSB * kSL, kSolutionPlane = kSB * kXL;
constexpr int kFactorPer = kSB * kSB / kSThreads, kSolutionPer = kSB * kSC / kSThreads;

inline int slabs(int nrhs) { return (nrhs + kSC - 1) / kSC; }

template <class R>
struct SweepArgs {
    int n, nrhs, nblk;
    const Cx<R>* A;  // the factor, L view: L(i, j) = A[i + j lda], or conj(A[j + i lda]) when upper
    long long lda;
    int upper;
    const Cx<R>* dinv;  // inverted 64 x 64 diagonal blocks, column-major
    Cx<R>* B;
    long long ldb;
    int* sync;   // per slab: ticket counter, published blocks; zero on entry
    int* error;  // set to 1 if a wait exceeds spin_limit
    int spin_limit;
};

template <class R, bool BACKWARD>
__global__ __launch_bounds__(kSThreads) void sweep_kernel(SweepArgs<R> a)
{
    using Op = Mfma<R>;
    __shared__ R Ls[2 * kFactorPlane];    // [k][row] of a factor block or of D, by planes
    __shared__ R Ms[2 * kFactorPlane];    // [k][row] of M = D L(t, t-1)
    __shared__ R Xs[2 * kSolutionPlane];  // [k][column] of a solution block
    __shared__ int s_ticket, s_seen;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int slab = blockIdx.y, c0 = slab * kSC, nc = min(kSC, a.nrhs - c0);
    int* const done = a.sync + 2 * slab + 1;
    if (tid == 0) s_ticket = atomicAdd(a.sync + 2 * slab, 1);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_ticket);
    auto block_of = [&](int q) { return BACKWARD ? a.nblk - 1 - q : q; };
    const int bt = block_of(t);
    const long long r0 = (long long)bt * kSB;
    const int w = (int)min((long long)kSB, a.n - r0);

    // Element e of this thread's share of the block that X_q multiplies, (r, k)
    // of L(t, q) or of L(q, t)^H: along a stored column (direct) or, conjugated,
    // along a stored row.
    const bool direct = BACKWARD == (a.upper != 0);
    auto factor_place = [&](int e, int& r, int& k) {
        const int fast = tid & (kSB - 1), slow = wave + 4 * e;
        r = direct ? fast : slow;
        k = direct ? slow : fast;
    };
    Cx<R> vl[kFactorPer], vx[kSolutionPer];
    auto fetch_factor = [&](int q) {
        const long long q0 = (long long)block_of(q) * kSB;
        const int wq = (int)min((long long)kSB, a.n - q0);
#pragma unroll
        for (int e = 0; e < kFactorPer; ++e) {
            int r, k;
            factor_place(e, r, k);
            const int rc = min(r, w - 1), kc = min(k, wq - 1);
            const Cx<R> x = direct ? a.A[(r0 + rc) + (q0 + kc) * a.lda] : a.A[(q0 + kc) + (r0 + rc) * a.lda];
            const bool in = r < w && k < wq;
            vl[e] = Cx<R>{in ? x.re : R(0), in ? (direct ? x.im : -x.im) : R(0)};
        }
    };
    auto put_factor = [&]() {
#pragma unroll
        for (int e = 0; e < kFactorPer; ++e) {
            int r, k;
            factor_place(e, r, k);
            Ls[k * kSL + r] = vl[e].re;
            Ls[kFactorPlane + k * kSL + r] = vl[e].im;
        }
    };
    // Ls = D of this block, or D^H (backward)
    auto put_inverse = [&]() {
        const Cx<R>* d = a.dinv + (long long)bt * kSB * kSB;
        Cx<R> v[kFactorPer];
#pragma unroll
        for (int e = 0; e < kFactorPer; ++e) v[e] = d[tid + kSThreads * e];
#pragma unroll
        for (int e = 0; e < kFactorPer; ++e) {
            const int i = tid & (kSB - 1), j = wave + 4 * e;  // D(i, j)
            const int at = BACKWARD ? i * kSL + j : j * kSL + i;
            Ls[at] = v[e].re;
            Ls[kFactorPlane + at] = BACKWARD ? -v[e].im : v[e].im;
        }
    };
    auto fetch_solution = [&](int q) {
        const long long q0 = (long long)block_of(q) * kSB;
        const int k = tid & (kSB - 1), kc = (int)min((long long)k, a.n - q0 - 1);
#pragma unroll
        for (int e = 0; e < kSolutionPer; ++e) {
            const int c = wave + 4 * e;
            const Cx<R> x = agent_load(a.B + (q0 + kc) + (long long)(c0 + min(c, nc - 1)) * a.ldb);
            const bool in = k == kc && c < nc;
            vx[e] = Cx<R>{in ? x.re : R(0), in ? x.im : R(0)};
        }
    };
    auto put_solution = [&]() {
        const int k = tid & (kSB - 1);
#pragma unroll
        for (int e = 0; e < kSolutionPer; ++e) {
            Xs[k * kXL + wave + 4 * e] = vx[e].re;
            Xs[kSolutionPlane + k * kXL + wave + 4 * e] = vx[e].im;
        }
    };
    // out += sign F Xs for the wavefront's 16 rows, F(row, k) = Fs[k][row], the 64
    // terms as one sum (out's scale rounds once)
    typename Op::acc_t acc[2];
    auto product = [&](const R* Fs, R sign, typename Op::acc_t (&out)[2]) {
        const R* fp = Fs + 16 * wave + li;
        typename Op::acc_t sum[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll 4
        for (int ks = 0; ks < kSB; ks += 4) {
            const R f[2] = {fp[(ks + lk) * kSL], fp[kFactorPlane + (ks + lk) * kSL]};
            const R x[2] = {Xs[(ks + lk) * kXL + li], Xs[kSolutionPlane + (ks + lk) * kXL + li]};
            mma_add(f, x, sum);
        }
        out[0] += sign * sum[0];
        out[1] += sign * sum[1];
    };
    // progress of the slab, at least `need` blocks published (uniform), or -1: the wait limit
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

    // M(row, c) = sum_k D(row, k) L(t, t-1)(k, c), sixteen columns c at a time
    // through Xs
    bool failed = false;
    if (t >= 1) {
        put_inverse();
        fetch_factor(t - 1);
        for (int part = 0; part < kSB / kSC; ++part) {
            __syncthreads();
#pragma unroll
            for (int e = 0; e < kFactorPer; ++e) {
                int r, k;
                factor_place(e, r, k);
                if (k / kSC == part) {
                    Xs[r * kXL + k % kSC] = vl[e].re;
                    Xs[kSolutionPlane + r * kXL + k % kSC] = vl[e].im;
                }
            }
            __syncthreads();
            typename Op::acc_t m[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
            product(Ls, R(1), m);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int at = (kSC * part + li) * kSL + 16 * wave + Op::row(lane, r);
                Ms[at] = m[0][r];
                Ms[kFactorPlane + at] = m[1][r];
            }
        }
        __syncthreads();
    }
    // acc = B_t - sum_{q < t - 1} L(t, q) X_q
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * wave + Op::row(lane, r);
        const bool in = row < w && li < nc;
        const Cx<R> x = in ? a.B[(r0 + row) + (long long)(c0 + li) * a.ldb] : Cx<R>{R(0), R(0)};
        acc[0][r] = x.re;
        acc[1][r] = x.im;
    }
    if (t > 1) fetch_factor(0);
    bool have_x = false;
    for (int q = 0; q < t - 1; ++q) {
        if (!have_x) {
            if (!wait_for(q + 1)) {
                failed = true;
                break;
            }
            fetch_solution(q);
        }
        put_factor();
        put_solution();
        __syncthreads();
        have_x = q + 1 < t - 1 && seen >= q + 2;
        if (q + 1 < t - 1) fetch_factor(q + 1);
        if (have_x) fetch_solution(q + 1);
        product(Ls, R(-1), acc);
        __syncthreads();
    }
    // acc = D acc, then minus M X_{t-1}
    put_inverse();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * wave + Op::row(lane, r);
        Xs[row * kXL + li] = acc[0][r];
        Xs[kSolutionPlane + row * kXL + li] = acc[1][r];
    }
    __syncthreads();
    acc[0] = acc[1] = typename Op::acc_t{0, 0, 0, 0};
    product(Ls, R(1), acc);
    __syncthreads();
    if (t >= 1 && !failed) {
        if (!wait_for(t)) {
            failed = true;
        } else {
            fetch_solution(t - 1);
            put_solution();
            __syncthreads();
            product(Ms, R(-1), acc);
        }
    }
    if (failed && tid == 0) atomicExch(a.error, 1);
    // X_t leaves through LDS, along the columns
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int row = 16 * wave + Op::row(lane, r);
        Xs[row * kXL + li] = acc[0][r];
        Xs[kSolutionPlane + row * kXL + li] = acc[1][r];
    }
    __syncthreads();
    {
        const int row = tid & (kSB - 1);
#pragma unroll
        for (int e = 0; e < kSolutionPer; ++e) {
            const int c = wave + 4 * e, at = row * kXL + c;
            if (row < w && c < nc)
                agent_store(a.B + (r0 + row) + (long long)(c0 + c) * a.ldb, Cx<R>{Xs[at], Xs[kSolutionPlane + at]});
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) __hip_atomic_store(done, t + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace zsolve_detail
} // namespace kern
} // namespace ddla
