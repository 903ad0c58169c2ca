// Grid cell and offset of an ion on the mesh of the smooth PME sum
// (get_scaled_fractionals and the cell of fill_charge_grid, pme_kernel.f90).
//
// Several kernels form the cell of the same ion: the sort that puts it into a
// brick, and the passes that add or read its points relative to that brick,
// in LDS, where another cell would be another brick's.  The roundings are
// therefore written out: fused where fma is called and nowhere else, whatever
// the loop around it is compiled to.
#pragma once
#include "agpu_internal.hpp"

namespace agpu {

struct PmeGrid {
    int K[3], nb[3];     // points and bricks per axis
};

__host__ __device__ __forceinline__ int wrapi(int x, int K) { return ((x % K) + K) % K; }

// scaled fractional of one axis, fr = K (w - anint(w) + 1/2): wrapped grid
// cell ib and the offset in it
__host__ __device__ __forceinline__ double pme_cell(const CellArg &B, const PmeGrid &g, int e, double x, double y,
                                                    double z, int &ib)
{
#pragma clang fp contract(off)
    // w = x recip(1,e) + y recip(2,e) + z recip(3,e)
    const double w = fma(z, B.A[2 + 3 * e], fma(x, B.A[0 + 3 * e], y * B.A[1 + 3 * e]));
    const double t = w - round(w) + 0.5, K = g.K[e];
    const int i = (int)(t * K);
    ib = wrapi(i, g.K[e]);
    return fma(t, K, -(double)i);
}

}  // namespace agpu
