// Host side of the panel factorization (kernels.h), for the element types that
// the including file instantiates.
#pragma once
#include "kernels.h"
#include "panel_tile.h"

#include <algorithm>
#include <complex>
#include <stdexcept>
#include <string>

namespace ddla {
namespace kern {

// The device element of a matrix of T.
template <class T>
struct PanelElement {
    using type = T;
};
template <class R>
struct PanelElement<std::complex<R>> {
    using type = Cx<R>;
};

inline void panel_check(const char* what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// panel work: [ inverses of a panel's diagonal blocks | sync_ints counters per 64-column block | error word ]
inline size_t panel_blocks(int n) { return (size_t)(n + panel_detail::kB - 1) / panel_detail::kB; }
inline size_t panel_counters(int n) { return panel_blocks(n) * panel_detail::sync_ints((int)panel_blocks(n)); }

template <class T>
inline size_t panel_inverse_bytes(int n)
{
    using namespace panel_detail;
    return (std::min(panel_blocks(n), (size_t)kMaxCols) * kB * kB * sizeof(T) + 255) / 256 * 256;
}

template <class T>
size_t panel_work_bytes(int n)
{
    using namespace panel_detail;
    return panel_inverse_bytes<T>(n) + ((panel_counters(n) + 1) * sizeof(int) + 255) / 256 * 256;
}

template <class T>
inline int* panel_sync(int n, void* work)
{
    return reinterpret_cast<int*>(static_cast<char*>(work) + panel_inverse_bytes<T>(n));
}

template <class T>
int* panel_error_word(int n, void* work)
{
    return panel_sync<T>(n, work) + panel_counters(n);
}

// p[0, count) := 0 for each problem y (problem y's words stride bytes after problem 0's)
static __global__ void zero_ints_kernel(int* p, int count, long long stride)
{
    int* q = reinterpret_cast<int*>(reinterpret_cast<char*>(p) + blockIdx.y * stride);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) q[i] = 0;
}

// The counters of a launch that waits inside, or a work queue: p[0, count) := 0.
inline void zero_counters(hipStream_t s, int* p, int count)
{
    zero_ints_kernel<<<1, 256, 0, s>>>(p, count, 0);
}

template <class T>
void panel_reset(hipStream_t s, int n, void* work, const Batch& batch)
{
    if (batch.count <= 0) return;
    const int count = (int)panel_counters(n) + 1;
    const dim3 grid((unsigned)((count + 255) / 256), (unsigned)batch.count);
    zero_ints_kernel<<<grid, 256, 0, s>>>(panel_sync<T>(n, work), count, batch.stride);
    panel_check("panel_reset");
}

template <class T>
void panel_factor(hipStream_t s, int n, T* A, long long lda, int k, int kb, int* info, void* work,
                  const Batch& batch)
{
    using namespace panel_detail;
    using E = typename PanelElement<T>::type;
    if (kb <= 0 || k < 0 || k + kb > n) return;
    if (kb > kMaxCols * kB) throw std::invalid_argument("panel_factor: panel wider than 4096 columns");
    if (k % kB != 0 || (kb % kB != 0 && k + kb < n))
        throw std::invalid_argument("panel_factor: panel must start and, before the last column, end on a 64-column boundary");
    if (batch.count <= 0) return;
    PanelArgs<E> a{reinterpret_cast<E*>(A), lda, n, k, kb, info, static_cast<E*>(work),
                   panel_sync<T>(n, work) + (size_t)(k / kB) * sync_ints((int)panel_blocks(n)),
                   panel_error_word<T>(n, work), wait_limit(), batch.stride};
    const int P = (kb + kB - 1) / kB, R = (n - k + kB - 1) / kB;
    const int units = panel_units(P, R);
    if (units > 65535) throw std::invalid_argument("panel_factor: too many blocks for one launch");
    panel_kernel<E><<<dim3((unsigned)batch.count, (unsigned)units), 256, 0, s>>>(a);
    panel_check("panel_factor");
}

} // namespace kern
} // namespace ddla
