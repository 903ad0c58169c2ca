// The batch handle: many small periodic structures of uneven size,
// concatenated (atoms of structure s are off[s] .. off[s+1]-1), shared by the
// batched Tersoff (batch.hip) and batched Ewald (ewald_batch.hip) paths.
#pragma once
#include <cstdint>
#include <vector>

#include "agpu_internal.hpp"

struct agpu_batch {
    int nstruct = 0;
    int ntot = 0;
    std::vector<int> h_off;        // atom offsets (nstruct + 1)
    std::vector<double> h_cell;    // 9 per structure: cell[9*s + 3*k + x]
    agpu::DevBuf off, sof, cell, rec, r, u, counts, offsets, nbr, scan_tmp, eatom,
        partial, gacc, flags;
    // per list entry: bond i -> j as {unit vector, length} in FP64 and FP32,
    // the index of the reverse entry j -> i (-1 if absent) and the owner i
    agpu::DevBuf bnd64, bnd32, rev, own;
    // per list entry: {fc, dfc}, {dE/dzeta, dE/dr}, the bond energy and the
    // force the owner's energy puts on the neighbour; per atom: its own force
    agpu::DevBuf fcd, pp, ebond, fslot, fown;
    // first atom of each chunk of whole rows with at most 256 list entries
    // (nchunk = 0 when some row is longer: the unfused path)
    agpu::DevBuf chunk;
    int nchunk = 0;
    // per list entry, backward: fc, dfc/dr and their R and S derivatives
    agpu::DevBuf cut;
    agpu::HostStats stats;
    double nl_cut = -1.0;          // cutoff of the current list (the requested one + skin)
    uint64_t pos_rev = 0, nl_rev = ~0ull;
    uint64_t struct_rev = 0;       // bumped by every set_structures
    int64_t total = 0;
    // batched Ewald state (k-vector runs per structure), owned
    void *ewb = nullptr;
    void (*ewb_free)(void *) = nullptr;
    ~agpu_batch()
    {
        if (ewb && ewb_free) ewb_free(ewb);
    }
};

namespace agpu {
// Fractional coordinates per atom into b->u, in units of 2^-32 of a lattice
// vector: the difference of two, taken modulo 2^32 as a signed number, is the
// difference to the nearest image along each axis.
int batch_fractions(agpu_batch *b);

// the wrapped difference of two of them as fractions of the lattice vectors
__device__ __forceinline__ void batch_diff(const int4 &a, const int4 &b, int (&d)[3])
{
    d[0] = (int)((unsigned)a.x - (unsigned)b.x);
    d[1] = (int)((unsigned)a.y - (unsigned)b.y);
    d[2] = (int)((unsigned)a.z - (unsigned)b.z);
}

constexpr double BATCH_TURN = 2.3283064365386963e-10;    // 2^-32

// Images around the nearest one that come within rc of an atom of a cell with
// reciprocal vectors b (m per axis), and the screening radius in FP32: a
// difference vector formed there is off by a few 2^-24 of its summands.
__device__ __forceinline__ float batch_reach(const double *A, const double *b, double rc, int (&m)[3])
{
    float reach = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double t = rc * sqrt(b[3 * k] * b[3 * k] + b[3 * k + 1] * b[3 * k + 1] + b[3 * k + 2] * b[3 * k + 2]);
        m[k] = max(0, (int)ceil(t - 0.5 + 1e-6));
        const float len = (float)sqrt(A[3 * k] * A[3 * k] + A[3 * k + 1] * A[3 * k + 1] + A[3 * k + 2] * A[3 * k + 2]);
        reach += (0.5f + m[k]) * len;
    }
    return (float)rc * 1.000001f + 1e-6f * reach;
}
}  // namespace agpu
