// Ewald Coulomb sum (e^2/Angstrom) on gfx950.
//
// Real space and self term follow pme_energy_and_forces / pme_potential
// (src/potentials/coulomb/pme.f90:215-321, 386-437, 467-472): erfc(beta r)/r
// over every neighbour image inside the cutoff, charges with |q| <= 1e-10
// skipped, self energy -beta/sqrt(pi) sum q^2.  Here each atom owns its full
// row (16 lanes per atom), so the reference's i<j scatter becomes a
// gather with the 1/2 of the directed double count -- no atomics.
//
// Reciprocal space (Ewald class): the direct structure-factor sum over the half
// space of k = 2 pi Bbox^T n with |k| <= kmax (the reference's PME class uses
// smooth PME, pme_kernel.f90:251-752, built in pme.hip), in ewald_recip.hip.
// The PME class (agpu_pme_create) shares the real space and self term and
// takes its reciprocal sum from pme.hip.
#include <cmath>
#include <cstring>
#include <vector>

#include "agpu_internal.hpp"
#include "ewald_pair.hpp"
#include "ewald_recip.hpp"
#include "profile.hpp"

namespace agpu {

struct EwaldState {
    double cutoff = 10.0, beta = 0.0, kmax = 0.0;
    double beta_req = 0.0, kmax_req = 0.0;
    double cell_key[9];
    int nat_key = -1;
    bool have_k = false;
    EwrState recip;
    DevBuf partial, phi_tmp, q4;
    // smooth PME reciprocal sum instead of the direct S(k) sum (PME class)
    PmeState *pme = nullptr;
    ~EwaldState()
    {
        if (pme) pme_state_free(pme);
    }
};

static void ewald_free(void *p) { delete static_cast<EwaldState *>(p); }

// ---------------------------------------------------------------------------
// real space
// ---------------------------------------------------------------------------
// {x, y, z, q} per slot of the list's bin order (caller atom order[p])
__global__ void k_ewald_pack(int nat, const SortedAtom *__restrict__ atoms, const int *__restrict__ order,
                             const double *__restrict__ q, double4 *__restrict__ q4)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nat) return;
    const SortedAtom a = atoms[p];
    q4[p] = make_double4(a.x, a.y, a.z, q[order[p]]);
}

constexpr int EW_NOSHIFT = (512 << 20) | (512 << 10) | 512;   // dc_pack(0, 0, 0)

// EWG lanes per ion.  16 (four ions per wavefront) when the ions fill the
// chip: with a wavefront per ion the ten sums over the lanes cost as much as
// one of the three trips that 190 neighbours take.  216 000 ions: 560 -> 332 us
// with 16 lanes and the shared exp of ewp_pair, 299 with the next neighbour's
// record fetched ahead; 1200 ions: 9 us with 64 lanes, 17 with 16.
template <typename R, int EWG>
__global__ void __launch_bounds__(256)
k_ewald_real(int nat, const int *__restrict__ order, const double4 *__restrict__ q4, CellArg C, NlRows L,
             double cutoff_sq, double beta, double sqrt_alpha_pi, double *__restrict__ f, double *__restrict__ phi,
             double *__restrict__ partial)
{
    __shared__ double s_red[4][7];
    const int lane = threadIdx.x & (EWG - 1), wave = threadIdx.x >> 6;
    const int ai = xcd_block() * (256 / EWG) + threadIdx.x / EWG;
    double e = 0.0, acc[3] = {0, 0, 0}, ph = 0.0;
    double w[6] = {0, 0, 0, 0, 0, 0};
    int i = -1;
    double qi = 0.0;
    if (ai < nat) {
        i = order[ai];
        const double4 hi = q4[ai];
        qi = hi.w;
        if (fabs(qi) > 1e-10) {
            const double ri[3] = {hi.x, hi.y, hi.z};
            int n;
            const int2 *row = nl_row(L, ai, n);
            if (n > 0) {
            const R b = (R)beta, sap = (R)sqrt_alpha_pi;
            auto pair = [&](const int2 en, const double4 qa) {
                const double qj = qa.w;
                if (!(fabs(qj) > 1e-10)) return;
                double d[3] = {ri[0] - qa.x, ri[1] - qa.y, ri[2] - qa.z};
                if (en.y != EW_NOSHIFT) {
                    int a, bb, c;
                    dc_unpack(en.y, a, bb, c);
#pragma unroll
                    for (int x = 0; x < 3; ++x) d[x] += image_x(C, x, a, bb, c);
                }
                const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
                if (!(r2 < cutoff_sq)) return;
                double hlp1, fr;
                ewp_pair(r2, b, sap, hlp1, fr);
                ph += qj * hlp1;
                const double fs = qj * fr;
                const double h[3] = {fs * d[0], fs * d[1], fs * d[2]};
                acc[0] += h[0];
                acc[1] += h[1];
                acc[2] += h[2];
                w[0] += d[0] * h[0];
                w[1] += d[1] * h[1];
                w[2] += d[2] * h[2];
                w[3] += d[1] * h[2];
                w[4] += d[0] * h[2];
                w[5] += d[0] * h[1];
            };
            // the next entry's record is on its way while a pair is evaluated
            // (past the row's end: its last entry again, not used)
            int2 en = row[min(lane, n - 1)];
            double4 qa = q4[en.x];
            for (int s = lane; s < n; s += EWG) {
                const int2 en1 = row[min(s + EWG, n - 1)];
                const double4 qa1 = q4[en1.x];
                pair(en, qa);
                en = en1;
                qa = qa1;
            }
            }
        }
    }
    ph = group_sum<EWG>(ph);
    for (int x = 0; x < 3; ++x) acc[x] = group_sum<EWG>(acc[x]);
    if (i >= 0 && lane == 0) {
        e = 0.5 * qi * ph;
        // self term (pme.f90:467-472; phi: pme.f90:256)
        if (fabs(qi) > 1e-10) ph -= 2.0 * qi * sqrt_alpha_pi;
        e -= qi * qi * sqrt_alpha_pi;
        if (f) {
            f[3 * (size_t)i] += qi * acc[0];
            f[3 * (size_t)i + 1] += qi * acc[1];
            f[3 * (size_t)i + 2] += qi * acc[2];
        }
        if (phi) phi[i] += ph;
    }
    // the wavefront's sums of the energy and of -1/2 q_i d x h over its ions
    double v[7] = {e, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 6; ++k) v[1 + k] = -0.5 * qi * w[k];
#pragma unroll
    for (int k = 0; k < 7; ++k) v[k] = group_sum<64>(v[k]);
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 7; ++k) s_red[wave][k] = v[k];
    __syncthreads();
    if (threadIdx.x < 7) {
        int qn = threadIdx.x;
        double v = ((s_red[0][qn] + s_red[1][qn]) + s_red[2][qn]) + s_red[3][qn];
        double *rec = partial + (size_t)blockIdx.x * 10;
        if (qn == 0) rec[0] = v;
        else if (qn == 1) rec[1] = v;
        else if (qn == 2) rec[5] = v;
        else if (qn == 3) rec[9] = v;
        else if (qn == 4) { rec[6] = v; rec[8] = v; }
        else if (qn == 5) { rec[3] = v; rec[7] = v; }
        else { rec[2] = v; rec[4] = v; }
    }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
int ewald_bind(agpu_potential *pot)
{
    EwaldState *st = static_cast<EwaldState *>(pot->impl);
    agpu_particles *p = pot->p;
    if (!(p->cell.pbc[0] && p->cell.pbc[1] && p->cell.pbc[2]))
        return set_error(AGPU_ERR_PBC, "Ewald summation only works for 3d periodic systems.");
    // beta <= 0: the reference's rule alpha = ln(10)*12/cutoff^2, beta = sqrt(alpha)
    st->beta = st->beta_req > 0.0 ? st->beta_req : std::sqrt(std::log(10.0) * 12.0 / (st->cutoff * st->cutoff));
    st->kmax = st->kmax_req > 0.0 ? st->kmax_req : 2.0 * st->beta * std::sqrt(-std::log(1e-13));
    AGPU_CHECK(agpu_neighbors_request_interaction_range(pot->nl, st->cutoff));
    st->have_k = false;
    return AGPU_OK;
}

static int ewald_run(agpu_potential *pot, const double *q, double *epot, double *f, double *wpot,
                     double *phi)
{
    EwaldState *st = static_cast<EwaldState *>(pot->impl);
    agpu_particles *p = pot->p;
    agpu_neighbors *nl = pot->nl;
    AGPU_CHECK(nl_update(nl, p, 0, false));
    const int nat = p->nat;
    if (!st->pme &&
        (!st->have_k || st->nat_key != nat || std::memcmp(st->cell_key, p->cell.A, sizeof st->cell_key) != 0)) {
        const int off[2] = {0, nat};
        st->have_k = false;
        AGPU_CHECK(ewr_plan(st->recip, 1, p->cell.A, off, st->kmax));
        std::memcpy(st->cell_key, p->cell.A, sizeof st->cell_key);
        st->nat_key = nat;
        st->have_k = true;
    }
    hipStream_t s = stream();
    if (epot) AGPU_HIP(hipMemsetAsync(epot, 0, sizeof(double), s));
    if (nat == 0) return AGPU_OK;
    CellArg C;
    std::memcpy(C.A, p->cell.A, sizeof C.A);
    const double sap = std::sqrt(st->beta * st->beta / M_PI);
    const bool few = nat < 16384;       // fewer than four wavefronts per SIMD with 16 lanes each
    const int ipb = few ? 4 : 16, nblk_r = (nat + ipb - 1) / ipb;
    const int nrec_k = st->pme ? 0 : st->recip.ntile;
    AGPU_CHECK(st->partial.reserve(sizeof(double) * 10 * (size_t)(nblk_r + nrec_k + 1)));
    double *part = st->partial.as<double>();
    const int *order = nl->idx_sorted.as<int>();
    const NlRows L = nl_rows(nl);
    AGPU_CHECK(st->q4.reserve(sizeof(double4) * (size_t)(nat + 1)));
    double4 *q4 = st->q4.as<double4>();
    AGPU_LAUNCH("ewald_pack", k_ewald_pack, dim3((nat + 255) / 256), dim3(256), 0, s, nat, L.atoms, order, q, q4);
    if (pot->precision == AGPU_PREC_MIXED)
        AGPU_LAUNCH("ewald_real_mixed", (few ? k_ewald_real<float, 64> : k_ewald_real<float, 16>), dim3(nblk_r),
                    dim3(256), 0, s, nat, order, q4, C, L, st->cutoff * st->cutoff, st->beta, sap, f, phi, part);
    else
        AGPU_LAUNCH("ewald_real_fp64", (few ? k_ewald_real<double, 64> : k_ewald_real<double, 16>), dim3(nblk_r),
                    dim3(256), 0, s, nat, order, q4, C, L, st->cutoff * st->cutoff, st->beta, sap, f, phi, part);
    if (st->pme) {
        // reciprocal record after the real-space block records
        AGPU_CHECK(pme_recip(st->pme, p, q, st->beta, part + 10 * (size_t)nblk_r, f, phi));
        AGPU_CHECK(reduce_ev(part, nblk_r + 1, 10, epot, wpot, nullptr));
        AGPU_HIP(hipStreamSynchronize(s));
        return AGPU_OK;
    }
    AGPU_CHECK(ewr_run(st->recip, nat, p->d_r, q, nullptr, st->kmax, st->beta, part + 10 * (size_t)nblk_r, f, phi));
    AGPU_CHECK(reduce_ev(part, nblk_r + nrec_k, 10, epot, wpot, nullptr));
    AGPU_HIP(hipStreamSynchronize(s));
    return AGPU_OK;
}

int ewald_compute(agpu_potential *pot, const agpu_eval_args *a)
{
    if (a->mask || a->epot_per_at || a->wpot_per_at)
        return set_error(AGPU_ERR_UNSUPPORTED, "Ewald: mask and per-atom properties are not supported");
    return ewald_run(pot, a->q, a->epot, a->f, a->wpot, nullptr);
}

int ewald_potential(agpu_potential *pot, const double *q, double *phi, int)
{
    EwaldState *st = static_cast<EwaldState *>(pot->impl);
    AGPU_CHECK(st->phi_tmp.reserve(sizeof(double) * 16));
    double *tmp = st->phi_tmp.as<double>();   // [0] epot, [1..9] wpot scratch
    AGPU_HIP(hipMemsetAsync(tmp, 0, sizeof(double) * 16, stream()));
    return ewald_run(pot, q, tmp, nullptr, tmp + 1, phi);
}

}  // namespace agpu

using namespace agpu;

extern "C" int agpu_ewald_create(agpu_potential **pot, double cutoff, double beta, double kmax)
{
    if (!pot || !(cutoff > 0.0)) return set_error(AGPU_ERR_ARG, "ewald_create: bad arguments");
    EwaldState *st = new EwaldState();
    st->cutoff = cutoff;
    st->beta_req = beta;
    st->kmax_req = kmax;
    agpu_potential *p = new agpu_potential();
    p->kind = AGPU_KIND_EWALD;
    p->cutoff = cutoff;
    p->impl = st;
    p->free_impl = ewald_free;
    *pot = p;
    return AGPU_OK;
}

extern "C" int agpu_pme_create(agpu_potential **pot, double cutoff, int order, const int *grid)
{
    if (!pot) return set_error(AGPU_ERR_ARG, "pme_create: pot is NULL");
    // pme_t defaults (pme.f90:36-46): cutoff 10, grid 64^3, order 8
    if (!(cutoff > 0.0)) cutoff = 10.0;
    if (order <= 0) order = 8;
    int K[3] = {64, 64, 64};
    if (grid)
        for (int d = 0; d < 3; ++d) K[d] = grid[d];
    if (order < 3 || order > 12) return set_error(AGPU_ERR_ARG, "PME: order must be 3 .. 12");
    for (int d = 0; d < 3; ++d)
        if (K[d] < order || K[d] > 1000)
            return set_error(AGPU_ERR_ARG, "PME: every grid dimension must be >= order and <= 1000");
    if ((long long)K[0] * K[1] * K[2] > (1ll << 30)) return set_error(AGPU_ERR_ARG, "PME: grid too large");
    EwaldState *st = new EwaldState();
    st->cutoff = cutoff;
    st->pme = pme_state_new(order, K);
    agpu_potential *p = new agpu_potential();
    p->kind = AGPU_KIND_PME;
    p->cutoff = cutoff;
    p->impl = st;
    p->free_impl = ewald_free;
    *pot = p;
    return AGPU_OK;
}
