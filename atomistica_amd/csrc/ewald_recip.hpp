// Direct reciprocal Ewald sums over one or many periodic structures
// (ewald_recip.hip), used by the Ewald class (ewald.hip) and by the batched
// Ewald path (ewald_batch.hip).
#pragma once
#include <vector>

#include "agpu_internal.hpp"

namespace agpu {

// A patch of 4 x 4 columns (n1 .. n1 + 3, n2 .. n2 + 3) with the n3 = n3c +- m,
// m = mb .. mb + 4 ks - 1, of one structure.
struct EwrItem {
    int n1, n2, n3c, mb;
    int nt, ks;          // 8-wide tiles of m (S(k)), 4-wide steps of m (forces)
    int s;               // structure
    int tile;            // first tile of T (128 entries each)
    int stile, sstride;  // first tile of the first split of S, tiles per split
    int nsplit, pad;
};

// S(k): one workgroup: items [item, item + nitem) (one structure, one mb),
// their tiles t0 .. t0 + nt - 1, ions [a0, a1)
struct EwrSBlock {
    int item, nitem, a0, a1, split, t0, nt, pad;
};

// forces: one workgroup: ions [a0, a1) of one structure, items [i0, i1); ion
// j's partial sums go to record rec + j
struct EwrFBlock {
    int a0, a1, i0, i1;
    long long rec, pad;
};

// where the partial sums of a structure's forces are: those of ion j and split
// k < nsplit are record rec + k n + j
struct EwrFRec {
    long long rec;
    int n, nsplit;
};

struct EwrState {
    int ntile = 0;       // tiles of T (and records)
    long long nfrec = 0; // partial force records, each structure's ions times its splits
    std::vector<EwrItem> items;
    std::vector<EwrSBlock> sblk;
    std::vector<EwrFBlock> fblk;
    std::vector<int> tile0;   // first tile of each structure (nstruct + 1)
    DevBuf d_items, d_sblk, d_fblk, d_frec, d_map, d_geo, d_tile0, S, T, s4, fpart;
};

// Patches, tiles and work blocks for structures with cells[9 s + 3 k + x] =
// component x of lattice vector k of structure s and atoms off[s] ..
// off[s + 1] - 1, |k| <= kmax.
int ewr_plan(EwrState &st, int ns, const double *cells, const int *off, double kmax);

// Records (10 doubles {e, W column-major} per tile, st.ntile of them; none
// without ions) into rec; f += forces,
// phi += potentials (either may be NULL); r, q, f, phi and sof (structure of
// each ion, NULL for one structure) are device arrays.
int ewr_run(EwrState &st, int nat, const double *r, const double *q, const int *sof, double kmax, double beta,
            double *rec, double *f, double *phi);

}  // namespace agpu
