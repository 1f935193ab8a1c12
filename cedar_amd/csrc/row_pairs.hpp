// Two neighbouring points of a row per thread: the loads and the exchange shared by the
// Gauss-Seidel kernels that relax both colours of a row in one launch (gs_rows2d.hip,
// gs_rows3d.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace cdr {

// Two adjacent values moved by one access.  Global accesses of 8 and 16 bytes need only 4-byte
// alignment on this GPU, so a pair may start at any element (rows of odd length included).
template <typename T>
struct __attribute__((aligned(alignof(T)))) row_pair {
    T a, b;
};
template <typename T>
__device__ inline row_pair<T> load2(const T *p) {
    row_pair<T> v;
    __builtin_memcpy(&v, p, sizeof(v));
    return v;
}
template <typename T>
__device__ inline void store2(T *p, T a, T b) {
    const row_pair<T> v{a, b};
    __builtin_memcpy(p, &v, sizeof(v));
}
// (p[1], p[2]); the row's last pair may lack its second point (has1 false): then p[2] may lie
// past the array, is not needed, and (p[0], p[1]) is read instead
template <typename T>
__device__ inline row_pair<T> load2_next(const T *p, bool has1) {
    row_pair<T> v = load2(p + (has1 ? 1 : 0));
    if (!has1) v.a = v.b;
    return v;
}

}  // namespace cdr
