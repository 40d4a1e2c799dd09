// Complex kernels of the Hermitian Cholesky path (declarations and contracts
// in zkernels.h).  There is no counterpart kernel in the reference, which calls
// vendor routines (hipSOLVER zpotrf / hipBLAS ztrsm, OpenBLAS on the CPU) for
// the complex types; the semantics followed are those of LAPACK ?potrf /
// ?potrs and of the reference's gemmVbatched and diag_logdet
// (src/vbatched/gemm_template_kernel_vbatched.hpp:46-105,
// src/diag_logdet_impl.h:50-113).
//
// Complex products run on the matrix cores as products of real and imaginary
// planes, four 16x16x4 steps for one of complex tiles (field.h); the planes are
// parted when a slab is staged in LDS.  (On the vector ALUs, at the same peak
// rates, every product also paid for its operands' LDS reads: 23 us for the
// average trailing update of an FP64 order-2000 factorization, 64 columns deep.)
#include "zkernels.h"
#include "gemm_tile.h"
#include "internal.h"
#include "kernels.h"
#include "panel_host.h"
#include "panel_tile.h"
#include "potf2_tile.h"
#include "zsolve_tile.h"

#include <cfloat>
#include <climits>
#include <cstdint>
#include <stdexcept>
#include <string>

namespace ddla {
namespace kern {

namespace {

inline void zcheck_launch(const char* what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

template <class R>
__device__ __forceinline__ Cx<R> cmul(Cx<R> a, Cx<R> b)
{
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <class R>
__device__ __forceinline__ void cfma(Cx<R>& c, Cx<R> a, Cx<R> b)  // c += a b
{
    c.re = fma(a.re, b.re, c.re);
    c.re = fma(-a.im, b.im, c.re);
    c.im = fma(a.re, b.im, c.im);
    c.im = fma(a.im, b.re, c.im);
}
template <class R>
__device__ __forceinline__ Cx<R> conj(Cx<R> a)
{
    return {a.re, -a.im};
}

// ---------------------------------------------------------------------------
// GEMM tile: 64 x 64 of C per 256-thread workgroup, four wavefronts (2 x 2) of
// 32 x 32, slabs of 16 columns of op(A) and rows of op(B) in LDS by
// planes, the next slab's loads in flight while one is multiplied.
// ---------------------------------------------------------------------------
using gemm_detail::kPad;
using gemm_detail::map_tile;
using gemm_detail::Mfma;
using gemm_detail::spread;
using gemm_detail::TileOrder;

constexpr int kT = 64;   // rows and columns of a tile
constexpr int kK = 16;   // slab depth
constexpr int kTh = 256;

template <class R>
struct ZProblem {
    int m, n, k;
    Cx<R> alpha, beta;
    const void* A;
    long long lda;
    int opa;
    const void* B;
    long long ldb;
    int opb;
    Cx<R>* C;
    long long ldc;
    int tri;
    long long diag;
};

// LDS elements of a tile's slabs (op(A)'s planes, then op(B)'s).
template <bool ACPX, bool BCPX>
constexpr int zslab_elems()
{
    return kK * (kT + kPad) * ((ACPX ? 2 : 1) + (BCPX ? 2 : 1));
}

// One operand's slabs: kT consecutive indices (rows of op(A) or columns of
// op(B)) by kK of the inner dimension, for the tile at origin o of `extent`.
// along: the stored contiguous dimension is that of the indices.  Loads of a slab that
// reaches beyond the operand are clamped and dropped.
template <class R, bool CPX>
struct ZOperand {
    static constexpr int PER = kT * kK / kTh, LD = kT + kPad;
    using E = std::conditional_t<CPX, Cx<R>, R>;
    const E* P;
    long long ld;
    int o, extent, k;
    bool along, conjugate;
    E v[PER];
    __device__ int index(int e) const { const int i = threadIdx.x + kTh * e; return along ? i % kT : i / kK; }
    __device__ int inner(int e) const { const int i = threadIdx.x + kTh * e; return along ? i / kT : i % kK; }
    __device__ void load(int k0)
    {
        if (o + kT <= extent && k0 + kK <= k) {
            const E* base = P + (along ? o + k0 * ld : k0 + o * ld);
#pragma unroll
            for (int e = 0; e < PER; ++e) v[e] = base[along ? index(e) + inner(e) * ld : inner(e) + index(e) * ld];
        } else {
#pragma unroll
            for (int e = 0; e < PER; ++e) {
                const int i = o + index(e), kk = k0 + inner(e);
                const long long ci = min(i, extent - 1), ck = min(kk, k - 1);
                const E x = P[along ? ci + ck * ld : ck + ci * ld];
                v[e] = i < extent && kk < k ? x : E{};
            }
        }
    }
    // element (k, i) at column i ^ place(k) of row k: the lanes that store along k fall on
    // distinct banks (gemm_detail::spread).  'T' 'N' products of complex128, batches of
    // 4000 of order 16: 131 -> 107 us, 16 of order 512: 496 -> 356 us, together with the
    // wavefronts that have no element of C and multiply nothing.
    __device__ int place(int k) const { return along ? 0 : spread<R, kT>(k); }
    __device__ void store(R* S) const
    {
#pragma unroll
        for (int e = 0; e < PER; ++e) {
            R* p = S + inner(e) * LD + (index(e) ^ place(inner(e)));
            if constexpr (CPX) {
                p[0] = v[e].re;
                p[kK * LD] = conjugate ? -v[e].im : v[e].im;
            } else {
                p[0] = v[e];
            }
        }
    }
};

template <class R, bool ACPX, bool BCPX>
__device__ void ztile(const ZProblem<R>& p, int ti, int tj, R* smem)
{
    using Op = Mfma<R>;
    constexpr int TM = kT / 32, TN = kT / 32;
    const int m0 = ti * kT, n0 = tj * kT;
    if (m0 >= p.m || n0 >= p.n) return;
    if (p.tri == 1 && (long long)(m0 + kT - 1) + p.diag < n0) return;  // wholly above the written lower part
    if (p.tri == 2 && (long long)m0 + p.diag > n0 + kT - 1) return;    // wholly below the written upper part
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = (wave & 1) * (kT / 2), wn = (wave >> 1) * (kT / 2);
    const int pair = sizeof(R) == 8 ? 4 * (lk >> 1) : 0;
    const bool any = m0 + wm < p.m && n0 + wn < p.n;  // the wavefront has elements of C
    // D^T = op(B)^T op(A)^T: lane l % 16 of an accumulator runs along i, C's contiguous dimension
    // The terms add up 64 at a time (acc, then into sum): C's scale rounds once in
    // 64 terms, as in a factorization by block columns of 64.
    typename Op::acc_t acc[TM][TN][2], sum[TM][TN][2];
#pragma unroll
    for (int x = 0; x < TM; ++x)
#pragma unroll
        for (int y = 0; y < TN; ++y)
#pragma unroll
            for (int c = 0; c < 2; ++c) acc[x][y][c] = sum[x][y][c] = typename Op::acc_t{0, 0, 0, 0};
    if (p.k > 0 && (p.alpha.re != R(0) || p.alpha.im != R(0))) {
        using OpA = ZOperand<R, ACPX>;
        using OpB = ZOperand<R, BCPX>;
        OpA a{static_cast<const typename OpA::E*>(p.A), p.lda, m0, p.m, p.k, p.opa == 0, p.opa == 2, {}};
        OpB b{static_cast<const typename OpB::E*>(p.B), p.ldb, n0, p.n, p.k, p.opb != 0, p.opb == 2, {}};
        R* const As = smem;
        R* const Bs = smem + (ACPX ? 2 : 1) * kK * OpA::LD;
        a.load(0);
        b.load(0);
        for (int k0 = 0; k0 < p.k; k0 += kK) {
            a.store(As);
            b.store(Bs);
            __syncthreads();
            if (k0 + kK < p.k) {
                a.load(k0 + kK);
                b.load(k0 + kK);
            }
            if (any) {
#pragma unroll
                for (int kk = 0; kk < kK; kk += 4) {
                    // place(kk + lk): place(kk), and in FP64 the pair of rows by bit 2
                    const int pa = a.place(kk), pb = b.place(kk);
                    const R* ap = As + (kk + lk) * OpA::LD + wm + (li ^ (pa & 15) ^ (a.along ? 0 : pair));
                    const R* bp = Bs + (kk + lk) * OpB::LD + wn + (li ^ (pb & 15) ^ (b.along ? 0 : pair));
                    R ar[TM], ai[TM], br[TN], bi[TN];
#pragma unroll
                    for (int x = 0; x < TM; ++x) {
                        ar[x] = ap[16 * (x ^ (pa >> 4))];
                        if (ACPX) ai[x] = ap[kK * OpA::LD + 16 * (x ^ (pa >> 4))];
                    }
#pragma unroll
                    for (int y = 0; y < TN; ++y) {
                        br[y] = bp[16 * (y ^ (pb >> 4))];
                        if (BCPX) bi[y] = bp[kK * OpB::LD + 16 * (y ^ (pb >> 4))];
                    }
#pragma unroll
                    for (int x = 0; x < TM; ++x)
#pragma unroll
                        for (int y = 0; y < TN; ++y) {
                            acc[x][y][0] = Op::mma(br[y], ar[x], acc[x][y][0]);
                            if (ACPX) acc[x][y][1] = Op::mma(br[y], ai[x], acc[x][y][1]);
                            if (ACPX && BCPX) acc[x][y][0] = Op::mma(bi[y], -ai[x], acc[x][y][0]);
                            if (BCPX) acc[x][y][1] = Op::mma(bi[y], ar[x], acc[x][y][1]);
                        }
                }
            }
            if ((k0 + kK) % 64 == 0 || k0 + kK >= p.k)
#pragma unroll
                for (int x = 0; x < TM; ++x)
#pragma unroll
                    for (int y = 0; y < TN; ++y)
#pragma unroll
                        for (int c = 0; c < 2; ++c) {
                            sum[x][y][c] += acc[x][y][c];
                            acc[x][y][c] = typename Op::acc_t{0, 0, 0, 0};
                        }
            __syncthreads();
        }
    }
    if (!any) return;
    // Accumulator (x, y, r) of lane l: i = 16 x + l % 16, j = 16 y + row(l, r)
    // within the wavefront's block.  A row of blocks of C is read before it is
    // written, so that its reads are in flight together.
    const bool beta_zero = p.beta.re == R(0) && p.beta.im == R(0);
#pragma unroll
    for (int x = 0; x < TM; ++x) {
        const int i = m0 + wm + 16 * x + li;
        Cx<R> cv[TN][4];
        bool live[TN][4];
#pragma unroll
        for (int y = 0; y < TN; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = n0 + wn + 16 * y + Op::row(lane, r);
                live[y][r] = i < p.m && j < p.n && (p.tri != 1 || (long long)i + p.diag >= j) &&
                             (p.tri != 2 || (long long)i + p.diag <= j);
                cv[y][r] = Cx<R>{R(0), R(0)};
                if (!beta_zero && live[y][r]) cv[y][r] = p.C[i + (long long)j * p.ldc];
            }
#pragma unroll
        for (int y = 0; y < TN; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = n0 + wn + 16 * y + Op::row(lane, r);
                Cx<R> v = cmul(p.alpha, Cx<R>{sum[x][y][0][r], sum[x][y][1][r]});
                if (!beta_zero) cfma(v, p.beta, cv[y][r]);
                if (live[y][r]) p.C[i + (long long)j * p.ldc] = v;
            }
    }
}

template <class R, bool ACPX, bool BCPX>
__global__ __launch_bounds__(kTh, 2) void zgemm_kernel(ZProblem<R> p, TileOrder o, const int* abort)
{
    __shared__ R smem[zslab_elems<ACPX, BCPX>()];
    if (abort != nullptr && *abort != 0) return;
    int ti, tj;
    if (!map_tile(o, blockIdx.x, ti, tj)) return;
    ztile<R, ACPX, BCPX>(p, ti, tj, smem);
}

template <class R>
struct ZBatch {
    const int *m, *n, *k, *lda, *ldb, *ldc;
    const void* const* A;
    const void* const* B;
    Cx<R>* const* C;
    Cx<R> alpha, beta;
    int opa, opb, batch, z0;
};

template <class R, bool ACPX, bool BCPX>
__global__ __launch_bounds__(kTh, 2) void zgemm_vbatched_kernel(ZBatch<R> v)
{
    __shared__ R smem[zslab_elems<ACPX, BCPX>()];
    const int b = v.z0 + blockIdx.z;
    if (b >= v.batch) return;
    ZProblem<R> p;
    p.m = v.m[b];
    p.n = v.n[b];
    p.k = v.k[b];
    if (p.m <= 0 || p.n <= 0) return;
    p.alpha = v.alpha;
    p.beta = v.beta;
    p.A = v.A[b];
    p.lda = v.lda[b];
    p.opa = v.opa;
    p.B = v.B[b];
    p.ldb = v.ldb[b];
    p.opb = v.opb;
    p.C = v.C[b];
    p.ldc = v.ldc[b];
    p.tri = 0;
    p.diag = 0;
    ztile<R, ACPX, BCPX>(p, blockIdx.x, blockIdx.y, smem);
}

// inv(block b) = L(b, b)^-1 for every 64 x 64 diagonal block of a factor.
template <class R>
__global__ __launch_bounds__(256) void ztrtri_kernel(bool upper, int n, const Cx<R>* A, long long lda, Cx<R>* inv)
{
    using namespace potf2_detail;
    __shared__ R S[2 * kPlane], X[2 * kPlane], rdiag[kB];
    const long long j0 = (long long)blockIdx.x * kB;
    load_block<Cx<R>>(upper, (int)min((long long)kB, n - j0), A + j0 + j0 * lda, lda, S);
    __syncthreads();
    if (threadIdx.x < kB) rdiag[threadIdx.x] = R(1) / S[threadIdx.x * kL + threadIdx.x];
    __syncthreads();
    invert_lower<Cx<R>>(S, rdiag, X);
    store_inverse<Cx<R>>(X, inv + (long long)blockIdx.x * kB * kB);
}

// ---------------------------------------------------------------------------
// Transposes and the Hermitian triangle swap, 32 x 32 tiles through LDS.
// ---------------------------------------------------------------------------
template <class R>
__global__ __launch_bounds__(256) void zconj_transpose_kernel(int m, int n, const Cx<R>* in, long long ldi, Cx<R>* out,
                                                              long long ldo)
{
    __shared__ Cx<R> t[32][33];
    const int i0 = blockIdx.x * 32, j0 = blockIdx.y * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + tx, j = j0 + r;
        if (i < m && j < n) t[r][tx] = in[i + (long long)j * ldi];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int j = j0 + tx, i = i0 + r;  // out(j, i) = conj(in(i, j))
        if (i < m && j < n) out[j + (long long)i * ldo] = conj(t[tx][r]);
    }
}

// Tile pair (bi, bj), bi >= bj, of the 32 x 32 tiling: lower tile (bi, bj)
// and upper tile (bj, bi) exchange with conjugation (diagonal tiles: their
// strict triangles).
template <class R>
__global__ __launch_bounds__(256) void zswap_triangles_kernel(int n, Cx<R>* A, long long lda)
{
    __shared__ Cx<R> lo[32][33], up[32][33];
    // blockIdx.x enumerates the lower triangle of tiles
    const int t = blockIdx.x;
    int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) / 2.0);
    while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
    while (bi * (bi + 1) / 2 > t) --bi;
    const int bj = t - bi * (bi + 1) / 2;
    const int i0 = bi * 32, j0 = bj * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int i = i0 + tx, j = j0 + r;  // lower tile element (i, j)
        if (i < n && j < n) lo[tx][r] = A[i + (long long)j * lda];
        const int ui = j0 + tx, uj = i0 + r;  // upper tile element (ui, uj)
        if (ui < n && uj < n) up[tx][r] = A[ui + (long long)uj * lda];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        // lower (i, j) <- conj(upper (j, i)); upper (ui, uj) <- conj(lower (uj, ui))
        const int i = i0 + tx, j = j0 + r;
        if (i < n && j < n && i > j) A[i + (long long)j * lda] = conj(up[r][tx]);
        const int ui = j0 + tx, uj = i0 + r;
        if (ui < n && uj < n && uj > ui) A[ui + (long long)uj * lda] = conj(lo[r][tx]);
    }
}

// ---------------------------------------------------------------------------
// log-determinant of the diagonal: deterministic two-pass reduction
// ---------------------------------------------------------------------------
constexpr int kZParts = 64;

template <class R>
__global__ __launch_bounds__(256) void zlogdet_partial_kernel(int n, const Cx<R>* A, long long lda, double* pmag,
                                                              double* pphase, int* pflags)
{
    __shared__ double sm[256], sp[256];
    __shared__ int sf[256];
    double mag = 0, ph = 0;
    int f = 0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const Cx<R> z = A[(long long)i * (lda + 1)];
        const double x = (double)z.re, y = (double)z.im;
        if (!(x <= DBL_MAX && x >= -DBL_MAX && y <= DBL_MAX && y >= -DBL_MAX)) {
            f |= 1;
            continue;
        }
        const double ax = fabs(x), ay = fabs(y);
        const double hi = ax > ay ? ax : ay, lo = ax > ay ? ay : ax;
        if (hi == 0) {
            f |= 2;
            continue;
        }
        const double ratio = lo / hi;
        mag += log(hi) + 0.5 * log1p(ratio * ratio);  // log |z| without overflowing |z|
        if (y == 0) {
            if (x < 0) f ^= 4;
        } else {
            ph += atan2(y, x);
        }
    }
    sm[threadIdx.x] = mag;
    sp[threadIdx.x] = ph;
    sf[threadIdx.x] = f;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sm[threadIdx.x] += sm[threadIdx.x + s];
            sp[threadIdx.x] += sp[threadIdx.x + s];
            const int a = sf[threadIdx.x], b = sf[threadIdx.x + s];
            sf[threadIdx.x] = ((a | b) & 3) | ((a ^ b) & 4);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        pmag[blockIdx.x] = sm[0];
        pphase[blockIdx.x] = sp[0];
        pflags[blockIdx.x] = sf[0];
    }
}

__global__ void zlogdet_final_kernel(const double* pmag, const double* pphase, const int* pflags, double* out)
{
    if (threadIdx.x != 0) return;
    double m = 0, ph = 0;
    int f = 0;
    for (int b = 0; b < kZParts; ++b) {
        m += pmag[b];
        ph += pphase[b];
        f = ((f | pflags[b]) & 3) | ((f ^ pflags[b]) & 4);
    }
    out[0] = m;
    out[1] = ph;
    *reinterpret_cast<int*>(out + 2) = f;
}

template <class R>
void launch_zgemm(hipStream_t s, bool ac, bool bc, const ZProblem<R>& p, const int* abort)
{
    TileOrder o;
    o.ntm = (p.m + kT - 1) / kT;
    o.ntn = (p.n + kT - 1) / kT;
    o.lower_enum = (p.tri == 1 && p.diag == 0 && p.m == p.n) ? 1 : 0;
    const long long total = o.lower_enum ? (long long)o.ntm * (o.ntm + 1) / 2 : (long long)o.ntm * o.ntn;
    if (total > (long long)INT_MAX / 2) throw std::invalid_argument("zgemm: problem too large for one launch");
    o.total = (int)total;
    o.group = 8;
    o.per_xcd = (o.total + 7) / 8;
    const unsigned grid = (unsigned)(o.per_xcd * 8);
    if (ac && bc) zgemm_kernel<R, true, true><<<grid, kTh, 0, s>>>(p, o, abort);
    else if (ac) zgemm_kernel<R, true, false><<<grid, kTh, 0, s>>>(p, o, abort);
    else if (bc) zgemm_kernel<R, false, true><<<grid, kTh, 0, s>>>(p, o, abort);
    else throw std::invalid_argument("zgemm: at least one complex operand");
    zcheck_launch("zgemm");
}

} // namespace

int op_code(char op)
{
    switch (op) {
    case 'N': case 'n': return 0;
    case 'T': case 't': return 1;
    case 'C': case 'c': return 2;
    default: throw std::invalid_argument("invalid transpose operation");
    }
}

template <class R>
void zgemm(hipStream_t s, bool a_complex, bool b_complex, char ta, char tb, int m, int n, int k,
           std::complex<R> alpha, const void* A, long long lda, const void* B, long long ldb, std::complex<R> beta,
           std::complex<R>* C, long long ldc, int tri, long long diag, const int* abort)
{
    if (m <= 0 || n <= 0) return;
    ZProblem<R> p;
    p.m = m;
    p.n = n;
    p.k = k < 0 ? 0 : k;
    p.alpha = {alpha.real(), alpha.imag()};
    p.beta = {beta.real(), beta.imag()};
    p.A = A;
    p.lda = lda;
    p.opa = op_code(ta);
    p.B = B;
    p.ldb = ldb;
    p.opb = op_code(tb);
    p.C = reinterpret_cast<Cx<R>*>(C);
    p.ldc = ldc;
    p.tri = tri;
    p.diag = diag;
    launch_zgemm<R>(s, a_complex, b_complex, p, abort);
}

template <class R>
void zgemm_vbatched(hipStream_t s, bool a_complex, bool b_complex, char ta, char tb, const int* m, const int* n,
                    const int* k, std::complex<R> alpha, const void* const* A, const int* lda, const void* const* B,
                    const int* ldb, std::complex<R> beta, std::complex<R>* const* C, const int* ldc, int batch,
                    int max_m, int max_n)
{
    if (batch <= 0 || max_m <= 0 || max_n <= 0) return;
    ZBatch<R> v;
    v.m = m;
    v.n = n;
    v.k = k;
    v.lda = lda;
    v.ldb = ldb;
    v.ldc = ldc;
    v.A = A;
    v.B = B;
    v.C = reinterpret_cast<Cx<R>* const*>(C);
    v.alpha = {alpha.real(), alpha.imag()};
    v.beta = {beta.real(), beta.imag()};
    v.opa = op_code(ta);
    v.opb = op_code(tb);
    v.batch = batch;
    const unsigned gx = (unsigned)((max_m + kT - 1) / kT), gy = (unsigned)((max_n + kT - 1) / kT);
    if (gy > 65535) throw std::invalid_argument("zgemm_vbatched: too many column tiles");
    for (int z0 = 0; z0 < batch; z0 += 65535) {
        v.z0 = z0;
        const dim3 grid(gx, gy, (unsigned)std::min(65535, batch - z0));
        if (a_complex && b_complex) zgemm_vbatched_kernel<R, true, true><<<grid, kTh, 0, s>>>(v);
        else if (a_complex) zgemm_vbatched_kernel<R, true, false><<<grid, kTh, 0, s>>>(v);
        else if (b_complex) zgemm_vbatched_kernel<R, false, true><<<grid, kTh, 0, s>>>(v);
        else throw std::invalid_argument("zgemm_vbatched: at least one complex operand");
        zcheck_launch("zgemm_vbatched");
    }
}

template <class R>
void ztrtri_diag_blocks(hipStream_t s, bool upper, int n, const std::complex<R>* A, long long lda,
                        std::complex<R>* inv)
{
    if (n <= 0) return;
    ztrtri_kernel<R><<<(n + 63) / 64, 256, 0, s>>>(upper, n, reinterpret_cast<const Cx<R>*>(A), lda,
                                                   reinterpret_cast<Cx<R>*>(inv));
    zcheck_launch("ztrtri_diag_blocks");
}

std::size_t zsolve_sync_bytes(int nrhs)
{
    return ((std::size_t)zsolve_detail::slabs(nrhs) * 4 * sizeof(int) + 255) / 256 * 256;
}

// The sweeps are bound by the chain of blocks while their workgroups (64-row blocks
// times 16-column slabs) are a few waves of the chip, and by reading the factor once a
// slab beyond; products of 64-row steps read it once for all columns.  A solve by
// products / by sweeps, us: complex128 n = 1500 with 768 columns (1152 workgroups)
// 2174 / 2033, n = 600 with 2048 (1280) 906 / 960, n = 4000 with 1024 (4032) 8036 /
// 17394; complex64 n = 1000 with 2048 (2048) 1011 / 1005, n = 600 with 4096 (2560)
// 658 / 808, n = 4000 with 1024 (4032) 4699 / 7753.
template <class R>
bool zsolve_sweeps(int n, int nrhs)
{
    return (long long)((n + 63) / 64) * zsolve_detail::slabs(nrhs) <= (sizeof(R) == 8 ? 1200 : 2048);
}

template <class R>
void zpotrs_sweeps(hipStream_t s, bool upper, int n, int nrhs, const std::complex<R>* A, long long lda,
                   const std::complex<R>* dinv, std::complex<R>* B, long long ldb, void* sync, int* error)
{
    using namespace zsolve_detail;
    if (n <= 0 || nrhs <= 0) return;
    const int ns = slabs(nrhs);
    SweepArgs<R> a{n, nrhs, (n + kSB - 1) / kSB, reinterpret_cast<const Cx<R>*>(A), lda, upper ? 1 : 0,
                   reinterpret_cast<const Cx<R>*>(dinv), reinterpret_cast<Cx<R>*>(B), ldb, static_cast<int*>(sync),
                   error, wait_limit()};
    zero_counters(s, a.sync, 4 * ns);
    const dim3 grid((unsigned)a.nblk, (unsigned)ns);
    sweep_kernel<R, false><<<grid, kSThreads, 0, s>>>(a);
    a.sync += 2 * ns;
    sweep_kernel<R, true><<<grid, kSThreads, 0, s>>>(a);
    zcheck_launch("zpotrs_sweeps");
}

template <class R>
void zconj_transpose(hipStream_t s, int m, int n, const std::complex<R>* in, long long ldi, std::complex<R>* out,
                     long long ldo)
{
    if (m <= 0 || n <= 0) return;
    const dim3 grid((unsigned)((m + 31) / 32), (unsigned)((n + 31) / 32));
    if (grid.y > 65535) throw std::invalid_argument("zconj_transpose: too many columns");
    zconj_transpose_kernel<R><<<grid, 256, 0, s>>>(m, n, reinterpret_cast<const Cx<R>*>(in), ldi,
                                                   reinterpret_cast<Cx<R>*>(out), ldo);
    zcheck_launch("zconj_transpose");
}

template <class R>
void zswap_triangles(hipStream_t s, int n, std::complex<R>* A, long long lda)
{
    if (n <= 1) return;
    const long long nt = (n + 31) / 32, tiles = nt * (nt + 1) / 2;
    if (tiles > 0x7fffffffLL) throw std::invalid_argument("zswap_triangles: order too large");
    zswap_triangles_kernel<R><<<(unsigned)tiles, 256, 0, s>>>(n, reinterpret_cast<Cx<R>*>(A), lda);
    zcheck_launch("zswap_triangles");
}

std::size_t zlogdet_work_bytes() { return (std::size_t)kZParts * (2 * sizeof(double) + sizeof(int)); }

template <class R>
void zdiag_logdet(hipStream_t s, int n, const std::complex<R>* A, long long lda, void* work, double* out)
{
    double* pmag = static_cast<double*>(work);
    double* pphase = pmag + kZParts;
    int* pflags = reinterpret_cast<int*>(pphase + kZParts);
    zlogdet_partial_kernel<R><<<kZParts, 256, 0, s>>>(n, reinterpret_cast<const Cx<R>*>(A), lda, pmag, pphase,
                                                       pflags);
    zcheck_launch("zdiag_logdet");
    zlogdet_final_kernel<<<1, 64, 0, s>>>(pmag, pphase, pflags, out);
    zcheck_launch("zdiag_logdet");
}

#define DDLA_ZINSTANTIATE(R)                                                                                      \
    template void zgemm<R>(hipStream_t, bool, bool, char, char, int, int, int, std::complex<R>, const void*,     \
                           long long, const void*, long long, std::complex<R>, std::complex<R>*, long long, int,  \
                           long long, const int*);                                                               \
    template void zgemm_vbatched<R>(hipStream_t, bool, bool, char, char, const int*, const int*, const int*,     \
                                    std::complex<R>, const void* const*, const int*, const void* const*,         \
                                    const int*, std::complex<R>, std::complex<R>* const*, const int*, int, int,  \
                                    int);                                                                        \
    template bool zsolve_sweeps<R>(int, int);                                                                    \
    template void zpotrs_sweeps<R>(hipStream_t, bool, int, int, const std::complex<R>*, long long,               \
                                   const std::complex<R>*, std::complex<R>*, long long, void*, int*);            \
    template size_t panel_work_bytes<std::complex<R>>(int);                                                      \
    template void panel_reset<std::complex<R>>(hipStream_t, int, void*, const Batch&);                           \
    template int* panel_error_word<std::complex<R>>(int, void*);                                                 \
    template void panel_factor<std::complex<R>>(hipStream_t, int, std::complex<R>*, long long, int, int, int*,   \
                                                void*, const Batch&);                                            \
    template void ztrtri_diag_blocks<R>(hipStream_t, bool, int, const std::complex<R>*, long long,              \
                                        std::complex<R>*);                                                       \
    template void zconj_transpose<R>(hipStream_t, int, int, const std::complex<R>*, long long, std::complex<R>*, \
                                     long long);                                                                 \
    template void zswap_triangles<R>(hipStream_t, int, std::complex<R>*, long long);                             \
    template void zdiag_logdet<R>(hipStream_t, int, const std::complex<R>*, long long, void*, double*);
DDLA_ZINSTANTIATE(float)
DDLA_ZINSTANTIATE(double)
#undef DDLA_ZINSTANTIATE

} // namespace kern
} // namespace ddla
