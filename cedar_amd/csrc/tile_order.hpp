// Workgroup order of launches over batches of 2D problems.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace cdr {
namespace k2 {

// Problems that share an operator come in groups of rep right-hand sides (problem b uses
// operator b / rep).  Such launches renumber their workgroups so that the rep workgroups of one
// tile of one operator run one after another on one XCD (workgroups are dealt round-robin over
// the 8 XCDs in launch order): the operator's tile comes from HBM once and from that XCD's L2
// for the other right-hand sides.  t (the workgroup's tile, tiles per problem) and b (its
// problem) are replaced by the logical pair; the map is a permutation of the launch, so every
// tile of every problem is still done once.  Launches whose tiles per problem are not a
// multiple of 8 keep the launch order.  Measured on 29 operators of 2049^2 with 4 right-hand
// sides each (mixed V(1,1) line-xy solve): 688 against 720 ms.
__device__ inline void shared_op_order(int tiles, int rep, int &t, int &b) {
    if (__builtin_expect(rep <= 1, 1) || tiles % 8 != 0) return;
    const int op = b / rep;
    const int off = (b - op * rep) * tiles + t;  // position in the operator's range, which
    const int k = off / 8;                       // starts on an XCD-0 workgroup
    t = (k / rep) * 8 + off % 8;
    b = op * rep + k % rep;
}

// The operator of problem b.  Problems fit 32 bits and most launches have one right-hand side per
// operator: as a 64-bit quotient this was a hundred instructions before a kernel's first load
// (1023^2 mixed solve 4.60 -> 4.37 ms, 4095^2 29.1 -> 28.5).
__device__ inline std::size_t operator_of(std::size_t b, int rep) {
    if (__builtin_expect(rep <= 1, 1)) return b;
    return (unsigned)b / (unsigned)rep;
}

// logical tile (x, y) and problem z of a tiled launch (problem index in blockIdx.z)
struct wg_pos {
    int x, y;
    std::size_t z;
};
__device__ inline wg_pos tiled_wg(int rep) {
    if (__builtin_expect(rep <= 1, 1))
        return {(int)blockIdx.x, (int)blockIdx.y, (std::size_t)blockIdx.z};
    int t = (int)(blockIdx.y * gridDim.x + blockIdx.x), b = (int)blockIdx.z;
    shared_op_order((int)(gridDim.x * gridDim.y), rep, t, b);
    return {t % (int)gridDim.x, t / (int)gridDim.x, (std::size_t)b};
}

}  // namespace k2
}  // namespace cdr
