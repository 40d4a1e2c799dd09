// Hermitian Cholesky path for std::complex<float> / std::complex<double> on one
// GPU: the blocked factorization, the two triangular solves and the
// log-determinant behind ppotrf / ppotrs / pposv / potrf / diag_logdet, and
// the complex and mixed real/complex gemmVbatched(2s).
//
// Reference behaviour followed (1 x 1 grid), as for the real types:
//   ppotrf   src/Cholesky/ppotrf.cpp:21-54 (A = L L^H for uplo 'L', U^H U for 'U')
//   ppotrs   src/Cholesky/ppotrs.cpp:38-61 (side 'L' applies L then L^H; side 'R'
//            the reverse; trans 'N' and 'C' solve the same Hermitian system)
//   logdet   src/diag_logdet_impl.h:50-113 (principal phase in (-pi, pi])
//   vbatched include/ddla/ddla.h:1878-1960 (mixed overloads: 'C' on a real operand is 'T')
// The arithmetic is this project's: the real types' blocked factorization with
// its two-panel look-ahead (potrf_blocked) on complex panels and the complex
// GEMM tile, and one persistent launch per solve sweep (zsolve_tile.h), or for
// many columns products of 64-row steps (solve_by_products).
#include "internal.h"
#include "kernels.h"
#include "zkernels.h"

#include <cmath>
#include <cstring>
#include <limits>
#include <stdexcept>

namespace ddla {

template <class T>
void potrf_blocked_dispatch(DdlaStream* h, bool upper, int n, T* A, long long lda, int* info, void* work);

namespace complex_impl {

namespace {

constexpr int kZB = 64;

std::size_t zdiag_inverse_elems(int n) { return (std::size_t)((n + kZB - 1) / kZB) * kZB * kZB; }

} // namespace

// Solves A X = B in place (B n x nrhs) with A = L L^H given by its L view
// (lower: L = A's lower triangle; upper: L = U^H of A's upper triangle) and the
// inverses D_t of its 64 x 64 diagonal blocks: forward L Y = B, then backward
// L^H X = Y, 64 rows a step (X_t = D_t B_t, then one product for all rows left).
template <class R>
void solve_by_products(DdlaStream* h, bool upper, int n, int nrhs, const std::complex<R>* A, long long lda,
                       const std::complex<R>* dinv, std::complex<R>* B, long long ldb)
{
    using C = std::complex<R>;
    const int nb = (n + kZB - 1) / kZB;
    // B(rows) -= op(block (r0, c0) of the L view, m x k or k x m) B(at)
    auto subtract = [&](int r0, int c0, char op, int m, int k, int rows, int at) {
        if (m <= 0) return;
        // upper: L(r, c) = conj(A(c, r)), so the block is stored conjugate transposed
        const C* p = upper ? A + c0 + r0 * lda : A + r0 + c0 * lda;
        const char stored = upper ? (op == 'N' ? 'C' : 'N') : op;
        kern::zgemm<R>(h->stream, true, true, stored, 'N', m, nrhs, k, C(-1), p, lda, B + at, ldb, C(1), B + rows, ldb);
    };
    // B_t := D_t B_t, or D_t^H B_t: one row of tiles, each of which reads its columns before it writes them
    auto multiply = [&](int t, char op) {
        const int w = std::min(kZB, n - t * kZB);
        C* bt = B + t * kZB;
        kern::zgemm<R>(h->stream, true, true, op, 'N', w, nrhs, w, C(1), dinv + (long long)t * kZB * kZB, kZB, bt, ldb,
                       C(0), bt, ldb);
    };
    for (int t = 0; t < nb; ++t) {
        const int r0 = t * kZB, r1 = std::min(n, r0 + kZB);
        multiply(t, 'N');
        subtract(r1, r0, 'N', n - r1, r1 - r0, r1, r0);
    }
    for (int t = nb - 1; t >= 0; --t) {
        const int r0 = t * kZB, r1 = std::min(n, r0 + kZB);
        multiply(t, 'C');
        subtract(r0, 0, 'C', r0, r1 - r0, 0, r0);
    }
}

template <class R>
std::size_t ppotrs_bytes(char side, int n, int nrhs)
{
    if (n == 0 || nrhs == 0) return 0;
    // [ inverses of the 64 x 64 diagonal blocks | sweep counters | error word | B^H (side 'R') ]
    std::size_t b = detail::padded_bytes<std::complex<R>>(zdiag_inverse_elems(n)) + kern::zsolve_sync_bytes(nrhs) +
                    detail::padded_bytes<int>(1);
    if (side == 'R') b += detail::padded_bytes<std::complex<R>>((std::size_t)n * nrhs);
    return b;
}

template <class R>
std::size_t ppotrf_bytes(int n)
{
    if (n <= 0) return 0;
    return detail::padded_bytes<int>(1) + detail::padded_bytes<char>(kern::panel_work_bytes<std::complex<R>>(n));
}

template <class R>
void ppotrf_run(const DdlaHandle_t& h, char uplo, int n, std::complex<R>* A, const int* d, int& info,
                void* work, std::size_t bytes)
{
    if (n == 0) {
        info = 0;
        return;
    }
    if (bytes < ppotrf_bytes<R>(n) || work == nullptr)
        throw std::invalid_argument("ppotrf: backend workspace smaller than the workspace query");
    char* w = static_cast<char*>(work);
    int* d_info = detail::take<int>(w, 1);
    fill_int(h->stream, d_info, 0);
    potrf_blocked_dispatch<std::complex<R>>(h, uplo == 'U', n, A, d[DDLA_LLD_], d_info, w);
    int error = 0;
    DDLA_HIP(hipMemcpyAsync(&info, d_info, sizeof(int), hipMemcpyDeviceToHost, h->stream));
    DDLA_HIP(hipMemcpyAsync(&error, kern::panel_error_word<std::complex<R>>(n, w), sizeof(int), hipMemcpyDeviceToHost,
                            h->stream));
    DDLA_HIP(hipStreamSynchronize(h->stream));
    if (error != 0) throw std::runtime_error("ppotrf: a panel factorization wait exceeded its limit");
}

template <class R>
void ppotrs_run(const DdlaHandle_t& h, char side, char uplo, int n, int nrhs, const std::complex<R>* A,
                const int* da, std::complex<R>* B, const int* db, void* work, std::size_t bytes)
{
    using C = std::complex<R>;
    if (n == 0 || nrhs == 0) return;
    if (bytes < ppotrs_bytes<R>(side, n, nrhs) || work == nullptr)
        throw std::invalid_argument("ppotrs: backend workspace smaller than the workspace query");
    const bool upper = uplo == 'U';
    const long long lda = da[DDLA_LLD_], ldb = db[DDLA_LLD_];
    char* w = static_cast<char*>(work);
    C* dinv = detail::take<C>(w, zdiag_inverse_elems(n));
    void* sync = w;
    w += kern::zsolve_sync_bytes(nrhs);
    int* error = detail::take<int>(w, 1);
    fill_int(h->stream, error, 0);
    auto sweeps = [&](C* b, long long ld) {
        LaunchTimer timer(h, kClassSolve, 8.0 * n * (double)n * nrhs, 2.0 * n * n * sizeof(R));
        if (kern::zsolve_sweeps<R>(n, nrhs))
            kern::zpotrs_sweeps<R>(h->stream, upper, n, nrhs, A, lda, dinv, b, ld, sync, error);
        else
            solve_by_products<R>(h, upper, n, nrhs, A, lda, dinv, b, ld);
    };
    {
        LaunchTimer timer(h, kClassTrtri, 4.0 * n * kZB * kZB / 3.0);
        kern::ztrtri_diag_blocks<R>(h->stream, upper, n, A, lda, dinv);
    }
    if (side == 'L') {
        sweeps(B, ldb);
    } else {
        // X A = B (B nrhs x n) with Hermitian A: A X^H = B^H
        C* bt = detail::take<C>(w, (std::size_t)n * nrhs);
        kern::zconj_transpose<R>(h->stream, nrhs, n, B, ldb, bt, n);
        sweeps(bt, n);
        kern::zconj_transpose<R>(h->stream, n, nrhs, bt, n, B, ldb);
    }
    int host_error = 0;
    DDLA_HIP(hipMemcpyAsync(&host_error, error, sizeof(int), hipMemcpyDeviceToHost, h->stream));
    DDLA_HIP(hipStreamSynchronize(h->stream));
    if (host_error != 0) throw std::runtime_error("ppotrs: a triangular-solve sweep exceeded its wait limit");
}

template <class R>
void potrf(const DdlaHandle_t& h, bool upper, int n, std::complex<R>* A, int lda, int* info)
{
    void* work = h->ensure_scratch(kern::panel_work_bytes<std::complex<R>>(n));
    fill_int(h->stream, info, 0);
    potrf_blocked_dispatch<std::complex<R>>(h, upper, n, A, lda, info, work);
}

// sum of log |d_i| and the principal phase, src/diag_logdet_impl.h:50-113
template <class R>
void diag_logdet(const DdlaHandle_t& h, int n, const std::complex<R>* a, int lda, std::complex<R>& result)
{
    if (n == 0) {
        result = {R(0), R(0)};
        return;
    }
    const std::size_t part = detail::padded_bytes<char>(kern::zlogdet_work_bytes());
    char* w = static_cast<char*>(h->ensure_scratch(part + detail::padded_bytes<double>(3)));
    double* out = reinterpret_cast<double*>(w + part);
    kern::zdiag_logdet<R>(h->stream, n, a, lda, w, out);
    double host[3];
    DDLA_HIP(hipMemcpyAsync(host, out, sizeof(host), hipMemcpyDeviceToHost, h->stream));
    DDLA_HIP(hipStreamSynchronize(h->stream));
    int flags;
    std::memcpy(&flags, &host[2], sizeof(int));
    if (flags & 1) throw std::domain_error("diag_logdet: nonfinite diagonal entry");
    if (flags & 2) {
        result = {-std::numeric_limits<R>::infinity(), R(0)};
        return;
    }
    const double pi = std::acos(-1.0);
    double phase = std::remainder(host[1] + ((flags >> 2) & 1) * pi, 2 * pi);
    if (phase <= -pi) phase = pi;
    result = {static_cast<R>(host[0]), static_cast<R>(phase)};
}

#define DDLA_CINSTANTIATE(R)                                                                                      \
    template std::size_t ppotrs_bytes<R>(char, int, int);                                                        \
    template std::size_t ppotrf_bytes<R>(int);                                                                   \
    template void ppotrf_run<R>(const DdlaHandle_t&, char, int, std::complex<R>*, const int*, int&, void*,       \
                                std::size_t);                                                                    \
    template void ppotrs_run<R>(const DdlaHandle_t&, char, char, int, int, const std::complex<R>*, const int*,   \
                                std::complex<R>*, const int*, void*, std::size_t);                               \
    template void potrf<R>(const DdlaHandle_t&, bool, int, std::complex<R>*, int, int*);                         \
    template void diag_logdet<R>(const DdlaHandle_t&, int, const std::complex<R>*, int, std::complex<R>&);
DDLA_CINSTANTIATE(float)
DDLA_CINSTANTIATE(double)
#undef DDLA_CINSTANTIATE

} // namespace complex_impl
} // namespace ddla
