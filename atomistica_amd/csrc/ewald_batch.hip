// Batched Ewald Coulomb sum (e^2/Angstrom) over many small periodic cells of
// uneven size, one launch per pass for the whole batch.
//
// Per structure, the same sums as the single-structure Ewald path (ewald.hip;
// real space and self term of pme.f90:215-321, 386-437, 467-472; reciprocal
// space as the direct structure-factor sum over the half space of
// k = 2 pi Bbox^T n, |k| <= kmax, in ewald_recip.hip):
//   k_ewb_real<R>  one wavefront per tile of <= 64 ions of one structure:
//                  every ion of the structure is staged through LDS and every
//                  periodic image within the cut-off is summed (the image
//                  range per axis comes from the reciprocal vectors), so no
//                  neighbour list is stored.  erfc/exp in R (double, or float
//                  with FP64 distances and FP64 accumulation).
//   k_ewb_sum      one wavefront per structure: energy and virial from the
//                  per-ion records and those of the reciprocal sum in a
//                  fixed order.
// There is no counterpart of batching in the reference, which evaluates one
// structure per call.  No atomics anywhere: every output has one writer.
#include <cmath>
#include <cstring>
#include <vector>

#include "agpu_internal.hpp"
#include "batch_internal.hpp"
#include "ewald_recip.hpp"
#include "profile.hpp"

namespace agpu {

constexpr int EWB_T = 64;      // ions per wavefront tile

struct EwbTile {
    int s, b, e, pad;      // structure, [b, e): ions
};

struct EwbState {
    double kmax = 0.0;
    uint64_t struct_rev = ~0ull;
    std::vector<EwbTile> itiles;
    EwrState recip;
    DevBuf d_itiles, d_ionrec, d_krec, d_q;
};

static void ewb_free(void *p) { delete static_cast<EwbState *>(p); }

// record layout (7 doubles): e, w_xx, w_yy, w_zz, w_yz, w_xz, w_xy
constexpr int EWB_REC = 7;

template <typename R> __device__ __forceinline__ R ewb_erfc(R x);
template <> __device__ __forceinline__ double ewb_erfc<double>(double x) { return erfc(x); }
template <> __device__ __forceinline__ float ewb_erfc<float>(float x) { return erfcf(x); }
template <typename R> __device__ __forceinline__ R ewb_exp(R x);
template <> __device__ __forceinline__ double ewb_exp<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float ewb_exp<float>(float x) { return expf(x); }

struct EwbGeom {
    const int *off;        // atom offsets per structure
    const double *cell;    // 9 per structure, cell[3k+x] = a_k[x]
    const double *rec;     // 9 per structure, rec[3k+x] = b_k[x], a_k . b_l = delta_kl
};

template <typename R>
__global__ void __launch_bounds__(EWB_T)
k_ewb_real(const EwbTile *__restrict__ tiles, EwbGeom G, const double *__restrict__ r,
           const double *__restrict__ q, double cutoff, double beta, double *__restrict__ f,
           double *__restrict__ phi, double *__restrict__ ionrec)
{
    __shared__ double sh_r[EWB_T][3];
    __shared__ double sh_q[EWB_T];
    const EwbTile T = tiles[blockIdx.x];
    const int lane = threadIdx.x;
    const int i = T.b + lane;
    const bool act = i < T.e;
    double A[9], b[9], t[3];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        A[k] = G.cell[9 * (size_t)T.s + k];
        b[k] = G.rec[9 * (size_t)T.s + k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
        t[k] = cutoff * sqrt(b[3 * k] * b[3 * k] + b[3 * k + 1] * b[3 * k + 1] + b[3 * k + 2] * b[3 * k + 2]);
    const double rc2 = cutoff * cutoff;
    const double sap = beta / sqrt(M_PI);
    const R bR = (R)beta, sapR = (R)sap, alR = (R)(beta * beta);
    double ri[3] = {0.0, 0.0, 0.0}, qi = 0.0;
    if (act) {
        ri[0] = r[3 * (size_t)i];
        ri[1] = r[3 * (size_t)i + 1];
        ri[2] = r[3 * (size_t)i + 2];
        qi = q[i];
    }
    const bool live = act && fabs(qi) > 1e-10;
    double e = 0.0, ph = 0.0, acc[3] = {0.0, 0.0, 0.0}, w[6] = {0, 0, 0, 0, 0, 0};
    const int a0 = G.off[T.s], a1 = G.off[T.s + 1];
    for (int base = a0; base < a1; base += EWB_T) {
        const int jj = base + lane;
        __syncthreads();
        if (jj < a1) {
            sh_r[lane][0] = r[3 * (size_t)jj];
            sh_r[lane][1] = r[3 * (size_t)jj + 1];
            sh_r[lane][2] = r[3 * (size_t)jj + 2];
            sh_q[lane] = q[jj];
        }
        __syncthreads();
        if (!live) continue;
        const int m = min(EWB_T, a1 - base);
        for (int tt = 0; tt < m; ++tt) {
            const double qj = sh_q[tt];
            if (!(fabs(qj) > 1e-10)) continue;
            const int j = base + tt;
            const double d0[3] = {ri[0] - sh_r[tt][0], ri[1] - sh_r[tt][1], ri[2] - sh_r[tt][2]};
            int lo[3], hi[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double ds = b[3 * k] * d0[0] + b[3 * k + 1] * d0[1] + b[3 * k + 2] * d0[2];
                lo[k] = (int)ceil(-ds - t[k] - 1e-9);
                hi[k] = (int)floor(-ds + t[k] + 1e-9);
            }
            for (int n0 = lo[0]; n0 <= hi[0]; ++n0)
                for (int n1 = lo[1]; n1 <= hi[1]; ++n1)
                    for (int n2 = lo[2]; n2 <= hi[2]; ++n2) {
                        if (j == i && n0 == 0 && n1 == 0 && n2 == 0) continue;
                        double d[3];
#pragma unroll
                        for (int x = 0; x < 3; ++x)
                            d[x] = d0[x] + (A[x] * n0 + A[3 + x] * n1 + A[6 + x] * n2);
                        const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
                        if (!(r2 < rc2)) continue;
                        const double ar = sqrt(r2);
                        const R arr = (R)ar;
                        const R ec = ewb_erfc<R>(bR * arr);
                        const R rinv = (R)1 / arr;
                        const R hlp = ec * rinv;
                        const R fr = rinv * rinv * rinv * (ec + (R)2 * sapR * arr * ewb_exp<R>(-alR * (R)r2));
                        const double qq = qi * qj;
                        e += 0.5 * qq * (double)hlp;
                        ph += qj * (double)hlp;
                        const double fs = qq * (double)fr;
                        const double h[3] = {fs * d[0], fs * d[1], fs * d[2]};
                        acc[0] += h[0];
                        acc[1] += h[1];
                        acc[2] += h[2];
                        w[0] -= 0.5 * d[0] * h[0];
                        w[1] -= 0.5 * d[1] * h[1];
                        w[2] -= 0.5 * d[2] * h[2];
                        w[3] -= 0.5 * d[1] * h[2];
                        w[4] -= 0.5 * d[0] * h[2];
                        w[5] -= 0.5 * d[0] * h[1];
                    }
        }
    }
    if (!act) return;
    // self term (pme.f90:467-472; phi: pme.f90:256)
    if (live) ph -= 2.0 * qi * sap;
    e -= qi * qi * sap;
    if (f) {
        f[3 * (size_t)i] += acc[0];
        f[3 * (size_t)i + 1] += acc[1];
        f[3 * (size_t)i + 2] += acc[2];
    }
    if (phi) phi[i] += ph;
    double *rec = ionrec + EWB_REC * (size_t)i;
    rec[0] = e;
#pragma unroll
    for (int k = 0; k < 6; ++k) rec[1 + k] = w[k];
}

// energy and virial per structure: one wavefront per structure, lane-strided
// partial sums of the ion records and of the records of the structure's tiles
// of k (10 wide), then a fixed butterfly
__global__ void __launch_bounds__(256)
k_ewb_sum(int nstruct, const int *__restrict__ off, const int *__restrict__ tile0,
          const double *__restrict__ ionrec, const double *__restrict__ krec, double *__restrict__ es,
          double *__restrict__ ws)
{
    const int s = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (s >= nstruct) return;
    double v[EWB_REC];
#pragma unroll
    for (int c = 0; c < EWB_REC; ++c) v[c] = 0.0;
    for (int a = off[s] + lane; a < off[s + 1]; a += 64)
#pragma unroll
        for (int c = 0; c < EWB_REC; ++c) v[c] += ionrec[EWB_REC * (size_t)a + c];
    for (int k = tile0[s] + lane; k < tile0[s + 1]; k += 64) {
        const double *o = krec + 10 * (size_t)k;
        v[0] += o[0];
        v[1] += o[1];
        v[2] += o[5];
        v[3] += o[9];
        v[4] += o[6];
        v[5] += o[3];
        v[6] += o[2];
    }
#pragma unroll
    for (int c = 0; c < EWB_REC; ++c) v[c] = group_sum<64>(v[c]);
    if (lane != 0) return;
    es[s] = v[0];
    if (ws) {
        double *w = ws + 9 * (size_t)s;
        w[0] = v[1];
        w[4] = v[2];
        w[8] = v[3];
        w[5] = w[7] = v[4];
        w[2] = w[6] = v[5];
        w[1] = w[3] = v[6];
    }
}

static int ewb_ion_tiles(agpu_batch *b, EwbState &st)
{
    st.itiles.clear();
    for (int s = 0; s < b->nstruct; ++s)
        for (int a = b->h_off[s]; a < b->h_off[s + 1]; a += EWB_T)
            st.itiles.push_back(EwbTile{s, a, std::min(a + EWB_T, b->h_off[s + 1]), 0});
    AGPU_CHECK(st.d_itiles.reserve(sizeof(EwbTile) * (st.itiles.size() + 1)));
    hipStream_t hs = stream();
    if (!st.itiles.empty())
        AGPU_HIP(hipMemcpyAsync(st.d_itiles.ptr, st.itiles.data(), sizeof(EwbTile) * st.itiles.size(),
                                hipMemcpyHostToDevice, hs));
    AGPU_HIP(hipStreamSynchronize(hs));
    return AGPU_OK;
}

}  // namespace agpu

using namespace agpu;

extern "C" int agpu_ewald_batch_compute(agpu_batch *b, const double *q, double cutoff, double beta, double kmax,
                                        int precision, double *e_struct, double *f, double *wpot_struct,
                                        double *phi, int flags)
{
    if (!b || !q || !e_struct) return set_error(AGPU_ERR_ARG, "ewald_batch_compute: bad arguments");
    if (!(cutoff > 0.0) || !(beta > 0.0) || !(kmax > 0.0))
        return set_error(AGPU_ERR_ARG, "ewald_batch_compute: need cutoff, beta, kmax > 0");
    if (precision != AGPU_PREC_FP64 && precision != AGPU_PREC_MIXED)
        return set_error(AGPU_ERR_ARG, "ewald_batch_compute: unknown precision");
    const int n = b->ntot, ns = b->nstruct;
    if (ns == 0) return AGPU_OK;
    if (!b->ewb) {
        b->ewb = new EwbState();
        b->ewb_free = ewb_free;
    }
    EwbState &st = *static_cast<EwbState *>(b->ewb);
    // the k-vectors' tiles follow the cells and atom counts (set_structures)
    if (st.struct_rev != b->struct_rev || st.kmax != kmax) {
        st.struct_rev = ~0ull;
        st.kmax = kmax;
        AGPU_CHECK(ewr_plan(st.recip, ns, b->h_cell.data(), b->h_off.data(), kmax));
        AGPU_CHECK(ewb_ion_tiles(b, st));
        st.struct_rev = b->struct_rev;
    }
    hipStream_t s = stream();
    const bool host = flags & AGPU_HOST;
    // device staging for host arrays: [q (n) | f (3n) | phi (n) | e (ns) | w (9 ns)]
    AGPU_CHECK(st.d_q.reserve(sizeof(double) * ((size_t)5 * n + 10 * (size_t)ns + 8)));
    double *dq = st.d_q.as<double>(), *df = dq + n, *dphi = df + 3 * (size_t)n, *de = dphi + n, *dw = de + ns;
    const double *qv = q;
    double *fv = f, *pv = phi, *ev = e_struct, *wv = wpot_struct;
    if (host) {
        if (n) AGPU_HIP(hipMemcpyAsync(dq, q, sizeof(double) * n, hipMemcpyHostToDevice, s));
        if (f && n) AGPU_HIP(hipMemcpyAsync(df, f, sizeof(double) * 3 * n, hipMemcpyHostToDevice, s));
        if (phi && n) AGPU_HIP(hipMemcpyAsync(dphi, phi, sizeof(double) * n, hipMemcpyHostToDevice, s));
        qv = dq;
        fv = f ? df : nullptr;
        pv = phi ? dphi : nullptr;
        ev = de;
        wv = wpot_struct ? dw : nullptr;
    }
    AGPU_CHECK(st.d_ionrec.reserve(sizeof(double) * EWB_REC * ((size_t)n + 1)));
    AGPU_CHECK(st.d_krec.reserve(sizeof(double) * 10 * ((size_t)st.recip.ntile + 1)));
    EwbGeom G{b->off.as<int>(), b->cell.as<double>(), b->rec.as<double>()};
    const int nit = (int)st.itiles.size();
    if (nit > 0) {
        if (precision == AGPU_PREC_MIXED)
            AGPU_LAUNCH("ewald_batch_real_mixed", k_ewb_real<float>, dim3(nit), dim3(EWB_T), 0, s,
                        st.d_itiles.as<EwbTile>(), G, b->r.as<double>(), qv, cutoff, beta, fv, pv,
                        st.d_ionrec.as<double>());
        else
            AGPU_LAUNCH("ewald_batch_real_fp64", k_ewb_real<double>, dim3(nit), dim3(EWB_T), 0, s,
                        st.d_itiles.as<EwbTile>(), G, b->r.as<double>(), qv, cutoff, beta, fv, pv,
                        st.d_ionrec.as<double>());
    }
    AGPU_CHECK(ewr_run(st.recip, n, b->r.as<double>(), qv, b->sof.as<int>(), kmax, beta, st.d_krec.as<double>(), fv,
                       pv));
    AGPU_LAUNCH("ewald_batch_sum", k_ewb_sum, dim3((ns + 3) / 4), dim3(256), 0, s, ns, b->off.as<int>(),
                st.recip.d_tile0.as<int>(), st.d_ionrec.as<double>(), st.d_krec.as<double>(), ev, wv);
    if (host) {
        if (f && n) AGPU_HIP(hipMemcpyAsync(f, df, sizeof(double) * 3 * n, hipMemcpyDeviceToHost, s));
        if (phi && n) AGPU_HIP(hipMemcpyAsync(phi, dphi, sizeof(double) * n, hipMemcpyDeviceToHost, s));
        AGPU_HIP(hipMemcpyAsync(e_struct, de, sizeof(double) * ns, hipMemcpyDeviceToHost, s));
        if (wpot_struct) AGPU_HIP(hipMemcpyAsync(wpot_struct, dw, sizeof(double) * 9 * ns, hipMemcpyDeviceToHost, s));
    }
    AGPU_HIP(hipStreamSynchronize(s));
    return AGPU_OK;
}
