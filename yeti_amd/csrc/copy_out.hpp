// copy_out.hpp -- stores of an element's COO range by a workgroup.
//
// An element's range starts at any entry, so 16-byte stores by position in the range cross 16-byte
// and cache-line borders: 3321-entry ranges (p = 2) are written at 4.4 TB/s that way and at 5.7 TB/s
// with the stores aligned by address (a head of up to 127 bytes, then 16 bytes per lane). Ranges that
// share a cache line should be written by the same XCD (its L2 then completes the line):
// xcd_element gives each of the 8 XCDs, to which workgroups are dealt in turn, one run of elements
// (300-entry ranges, p = 1: 3.3 -> 6.2 TB/s; 3321: 3.5 -> 5.7 TB/s together with the alignment).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace yeti {

constexpr int XCDS = 8;

// grid of a one-element-per-workgroup kernel and the element of workgroup b (>= n: none)
__host__ __device__ inline int64_t xcd_per(int64_t n) { return (n + XCDS - 1) / XCDS; }
inline unsigned xcd_grid(int64_t n) { return (unsigned)(xcd_per(n) * XCDS); }
__device__ __forceinline__ int64_t xcd_element(int64_t b, int64_t n) { return b % XCDS * xcd_per(n) + b / XCDS; }

// dst[x] = get(x), x < n, by threads t of NTH
template <int NTH, typename T, typename F>
__device__ __forceinline__ void store_run(T *__restrict__ dst, int n, int t, F &&get) {
    constexpr int V = 16 / sizeof(T), LINE = 128 / sizeof(T);
    typedef T vec __attribute__((ext_vector_type(V)));
    static_assert(NTH >= LINE, "the head by one thread each");
    const int head = min(n, (int)((0 - reinterpret_cast<uintptr_t>(dst)) / sizeof(T) % LINE));
    const int end = head + (n - head) / V * V;
    if (t < head) dst[t] = get(t);
#pragma unroll 4
    for (int x = head + V * t; x < end; x += V * NTH) {
        vec v;
#pragma unroll
        for (int u = 0; u < V; ++u) v[u] = get(x + u);
        *reinterpret_cast<vec *>(dst + x) = v;
    }
    if (t < n - end) dst[end + t] = get(end + t);
}

}  // namespace yeti
