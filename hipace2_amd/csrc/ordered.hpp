// What the ordered depositions of the plasma (ordered.hip) and of the beam (gather.hip) share:
// where a stencil starts, the tile of a start cell, and the part of a stencil inside a block.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace hpq {

// start cell = floor(xmid + 0.5 * BASE) + DELTA, for the order-O shape factor and for the
// type-T derivative shape factor (ShapeFactors.H: compute_single_shape_factor,
// single_derivative_shape_factor)
template <int O> constexpr int shape_base() { return (O == 0 || O == 2) ? 1 : 0; }
template <int O> constexpr int shape_delta() { return O >= 2 ? -1 : 0; }
template <int T, int O> constexpr int dshape_base() {
    return T == 0 ? shape_base<O>() : (T == 1 ? ((O == 1 || O == 3) ? 1 : 0) : ((O == 0 || O == 2) ? 1 : 0));
}
template <int T, int O> constexpr int dshape_delta() {
    return T == 0 ? shape_delta<O>() : (T == 1 ? (O == 0 ? 0 : (O == 3 ? -2 : -1)) : (O >= 2 ? -2 : -1));
}

// the tile of start cell s along one direction (C division truncates toward zero, as the
// reference's (cell - lo) / tile does; clamped to the tile grid)
__device__ __forceinline__ int dep_tile(int s, int ng, int T, int nt) { return min(max((s + ng) / T, 0), nt - 1); }

// bits [first, last) of a stencil's S, S < 32. Both ends may lie on either side of it: a stencil
// that starts beyond the last cell of its block (a particle outside the plane) has last < 0.
__host__ __device__ __forceinline__ uint32_t stencil_bits(int first, int last, int S) {
    const int a = first < 0 ? 0 : first < S ? first : S, b = last < 0 ? 0 : last < S ? last : S;
    return a < b ? (1u << b) - (1u << a) : 0u;
}

}  // namespace hpq
