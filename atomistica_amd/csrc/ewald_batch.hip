// Batched Ewald Coulomb sum (e^2/Angstrom) over many small periodic cells of
// uneven size, one launch per pass for the whole batch.
//
// Per structure, the same sums as the single-structure Ewald path (ewald.hip;
// real space and self term of pme.f90:215-321, 386-437, 467-472; reciprocal
// space as the direct structure-factor sum over the half space of
// k = 2 pi Bbox^T n, |k| <= kmax, in ewald_recip.hip):
//   k_ewb_real<R>  one wavefront per ion: every ion of the structure and its
//                  images are screened in FP32, those within r_c collected
//                  in LDS and summed, so no neighbour list is stored.  erfc
//                  and exp in R (double, or float with FP64 distances and
//                  FP64 accumulation).
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
#include "ewald_pair.hpp"
#include "ewald_recip.hpp"
#include "profile.hpp"

namespace agpu {

struct EwbState {
    double kmax = 0.0;
    uint64_t struct_rev = ~0ull;
    int nsmall = 0;      // ions in cells of up to EWB_SMALL
    EwrState recip;
    DevBuf d_ionrec, d_krec, d_q;
};

static void ewb_free(void *p) { delete static_cast<EwbState *>(p); }

// record layout (7 doubles): e, w_xx, w_yy, w_zz, w_yz, w_xz, w_xy
constexpr int EWB_REC = 7;

struct EwbGeom {
    const int *off;        // atom offsets per structure
    const double *cell;    // 9 per structure, cell[3k+x] = a_k[x]
    const double *rec;     // 9 per structure, rec[3k+x] = b_k[x], a_k . b_l = delta_kl
};

// A wavefront per ion.  The lanes screen 64 ions of the structure at a time
// in FP32 (with slack for the rounding), for the nearest image and, in cells
// below twice the cut-off, the images around it; those that pass are
// collected in LDS and evaluated 64 at a time.  A lane per ion that walked
// all candidates by itself ran the pair evaluation for nearly every
// candidate, since one of 64 ions nearly always had it inside the cut-off.
//
// SMALL: cells of up to EWB_SMALL ions.  They leave lanes and most of EWB_C
// candidates without an ion but have many images: the ions stay on the lanes,
// one or two per lane (an ion on several lanes if they are fewer), and the
// lanes take EWB_C images at a time.  Real space of 20 000 cells of 8 ions 3.5 ->
// 0.61 ms, 1024 of 64 443 -> 304 us, of 96 691 -> 639 us; at 144 ions both are
// equal.
constexpr int EWB_W = 4;            // wavefronts per workgroup
constexpr int EWB_C = 4;            // candidates per lane loaded together, or images
constexpr int EWB_SMALL = 128;
constexpr int EWB_NCOMB = 4096;     // images up to which FP32 tells their index apart

template <typename R, bool SMALL>
__global__ void __launch_bounds__(64 * EWB_W)
k_ewb_real(int n, const int *__restrict__ sof, EwbGeom G, const double *__restrict__ r, const int4 *__restrict__ u,
           const double *__restrict__ q, double cutoff, double beta, double *__restrict__ f,
           double *__restrict__ phi, double *__restrict__ ionrec, int size0, int size1)
{
    __shared__ int2 queue[EWB_W][64 * (EWB_C + 1)];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = blockIdx.x * EWB_W + wave;
    if (i >= n) return;
    const int st = sof[i];
    const int a0 = G.off[st], a1 = G.off[st + 1];
    if (a1 - a0 < size0 || a1 - a0 > size1) return;     // the other launch's
    int2 *Q = queue[wave];
    double A[9], b[9];
    int m[3];
    float Af[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        A[k] = G.cell[9 * (size_t)st + k];
        b[k] = G.rec[9 * (size_t)st + k];
        Af[k] = (float)A[k];
    }
    const float rs = batch_reach(A, b, cutoff, m), rs2 = rs * rs;
    const double rc2 = cutoff * cutoff;
    const double sap = beta / sqrt(M_PI);
    const double ri[3] = {r[3 * (size_t)i], r[3 * (size_t)i + 1], r[3 * (size_t)i + 2]};
    const double qi = q[i];
    const int4 ui = u[i];
    double ph = 0.0, acc[3] = {0.0, 0.0, 0.0}, w[6] = {0, 0, 0, 0, 0, 0};

    // evaluates the collected candidates from .. from + cnt - 1, one per lane
    auto evaluate = [&](int from, int cnt) {
        if (lane >= cnt) return;
        const int2 c = Q[from + lane];
        const int j = c.x;
        const double qj = q[j];
        if (!(fabs(qj) > 1e-10)) return;
        const int4 uj = u[j];
        const double d0[3] = {ri[0] - r[3 * (size_t)j], ri[1] - r[3 * (size_t)j + 1], ri[2] - r[3 * (size_t)j + 2]};
        int du[3];
        batch_diff(ui, uj, du);
        double nk[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            // the whole turns between the difference and its wrapped form
            const double ds = b[3 * k] * d0[0] + b[3 * k + 1] * d0[1] + b[3 * k + 2] * d0[2];
            nk[k] = rint((double)du[k] * BATCH_TURN - ds) + (double)(((c.y >> (10 * k)) & 1023) - 512);
        }
        if (j == i && nk[0] == 0.0 && nk[1] == 0.0 && nk[2] == 0.0) return;
        double d[3];
#pragma unroll
        for (int x = 0; x < 3; ++x) d[x] = d0[x] + (A[x] * nk[0] + A[3 + x] * nk[1] + A[6 + x] * nk[2]);
        const double r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        if (!(r2 < rc2)) return;
        double hlp, fr;
        ewp_pair(r2, (R)beta, (R)sap, hlp, fr);
        ph += qj * hlp;
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

    if (fabs(qi) > 1e-10) {
        const int w0 = 2 * m[0] + 1, w1 = 2 * m[1] + 1, w2 = 2 * m[2] + 1, ncomb = w0 * w1 * w2;
        int nq = 0;
        // image (n0, n1, n2) around the nearest one of ion j, whose wrapped
        // difference in fractional coordinates is v: collected if it may be near
        auto screen = [&](bool ok, int j, float v0, float v1, float v2, int n0, int n1, int n2) {
            v0 += (float)n0;
            v1 += (float)n1;
            v2 += (float)n2;
            const float x = Af[0] * v0 + Af[3] * v1 + Af[6] * v2;
            const float y = Af[1] * v0 + Af[4] * v1 + Af[7] * v2;
            const float z = Af[2] * v0 + Af[5] * v1 + Af[8] * v2;
            const bool in = ok && x * x + y * y + z * z < rs2;
            const unsigned long long mk = __ballot(in);
            if (in)
                Q[nq + __builtin_amdgcn_mbcnt_hi((unsigned)(mk >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mk, 0))] =
                    make_int2(j, (n0 + 512) | ((n1 + 512) << 10) | ((n2 + 512) << 20));
            nq += __popcll(mk);
        };
        // the last ones collected go first: nothing is moved
        auto drain = [&](bool last) {
            while (nq >= 64 || (last && nq > 0)) {
                const int cnt = min(nq, 64);
                wave_sync();
                evaluate(nq - cnt, cnt);
                wave_sync();
                nq -= cnt;
            }
        };
        if (SMALL) {
            const int ns = a1 - a0;
            const float r12 = 1.0f / (float)(w1 * w2), r2 = 1.0f / (float)w2;
            // lane groups W wide hold the ions, and 64 / W images go together;
            // more than 64 ions are taken in turn, as ions lane and 64 + lane
            const int W = ns > 64 ? 64 : 1 << (32 - __clz(ns - 1)), jl = lane & (W - 1), P = 64 / W;
            float f[2][3];
            auto difference = [&](int h) {
                int d[3];
                batch_diff(ui, u[a0 + min(jl + 64 * h, ns - 1)], d);
#pragma unroll
                for (int k = 0; k < 3; ++k) f[h][k] = (float)d[k] * (float)BATCH_TURN;
            };
            difference(0);
            auto image = [&](int h, int o) {
                const int n0 = ncomb <= EWB_NCOMB ? (int)(((float)o + 0.5f) * r12) : o / (w1 * w2);
                const int o1 = o - n0 * (w1 * w2);
                const int n1 = ncomb <= EWB_NCOMB ? (int)(((float)o1 + 0.5f) * r2) : o1 / w2, n2 = o1 - n1 * w2;
                screen(jl + 64 * h < ns && o < ncomb, a0 + jl + 64 * h, f[h][0], f[h][1], f[h][2], n0 - m[0],
                       n1 - m[1], n2 - m[2]);
            };
            if (ns > 64) {
                difference(1);
                for (int o = 0; o < ncomb; o += EWB_C / 2) {
#pragma unroll
                    for (int c = 0; c < EWB_C; ++c) image(c & 1, o + c / 2);
                    drain(o + EWB_C / 2 >= ncomb);
                }
            } else {
                for (int o = 0; o < ncomb; o += P * EWB_C) {
#pragma unroll
                    for (int c = 0; c < EWB_C; ++c) image(0, o + P * c + lane / W);
                    drain(o + P * EWB_C >= ncomb);
                }
            }
        } else {
            for (int base = a0; base < a1; base += 64 * EWB_C) {
                float du[EWB_C][3];
                int4 uj[EWB_C];
#pragma unroll
                for (int c = 0; c < EWB_C; ++c) uj[c] = u[min(base + 64 * c + lane, a1 - 1)];
#pragma unroll
                for (int c = 0; c < EWB_C; ++c) {
                    int d[3];
                    batch_diff(ui, uj[c], d);
#pragma unroll
                    for (int k = 0; k < 3; ++k) du[c][k] = (float)d[k] * (float)BATCH_TURN;
                }
                for (int o = 0; o < ncomb; ++o) {
                    const int n0 = o / (w1 * w2) - m[0], n1 = (o / w2) % w1 - m[1], n2 = o % w2 - m[2];
#pragma unroll
                    for (int c = 0; c < EWB_C; ++c) {
                        const int j = base + 64 * c + lane;
                        screen(j < a1, j, du[c][0], du[c][1], du[c][2], n0, n1, n2);
                    }
                    drain(base + 64 * EWB_C >= a1 && o == ncomb - 1);
                }
            }
        }
    }
    ph = group_sum<64>(ph);
#pragma unroll
    for (int x = 0; x < 3; ++x) acc[x] = group_sum<64>(acc[x]);
#pragma unroll
    for (int k = 0; k < 6; ++k) w[k] = group_sum<64>(w[k]);
    if (lane != 0) return;
    double *o = ionrec + EWB_REC * (size_t)i;
    // self term (pme.f90:467-472; phi: pme.f90:256)
    o[0] = 0.5 * qi * ph - qi * qi * sap;
#pragma unroll
    for (int k = 0; k < 6; ++k) o[1 + k] = -0.5 * qi * w[k];
    if (f) {
        f[3 * (size_t)i] += qi * acc[0];
        f[3 * (size_t)i + 1] += qi * acc[1];
        f[3 * (size_t)i + 2] += qi * acc[2];
    }
    if (phi) phi[i] += fabs(qi) > 1e-10 ? ph - 2.0 * qi * sap : ph;
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
        st.nsmall = 0;
        for (int k = 0; k < ns; ++k) {
            const int size = b->h_off[k + 1] - b->h_off[k];
            if (size <= EWB_SMALL) st.nsmall += size;
        }
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
    if (n > 0) {
        AGPU_CHECK(batch_fractions(b));
        const int4 *u = b->u.as<int4>();
        const dim3 g((n + EWB_W - 1) / EWB_W), t(64 * EWB_W);
        const bool mixed = precision == AGPU_PREC_MIXED;
        const char *name = mixed ? "ewald_batch_real_mixed" : "ewald_batch_real_fp64";
        // A launch for the small cells when they hold an eighth of the ions or
        // more.  With fewer the general kernel takes them too: each launch has a
        // wavefront for every ion, and these are the small part of its work.
        // 9200 cells of 8 and 1000 of 512 ions, just beyond the line, one launch
        // 3.16 ms, two 1.87 ms.
        const bool small = st.nsmall > 0 && 8ll * st.nsmall >= n;
        if (small)
            AGPU_LAUNCH(name, (mixed ? k_ewb_real<float, true> : k_ewb_real<double, true>), g, t, 0, s, n,
                        b->sof.as<int>(), G, b->r.as<double>(), u, qv, cutoff, beta, fv, pv,
                        st.d_ionrec.as<double>(), 0, EWB_SMALL);
        if (!small || st.nsmall < n)
            AGPU_LAUNCH(name, (mixed ? k_ewb_real<float, false> : k_ewb_real<double, false>), g, t, 0, s, n,
                        b->sof.as<int>(), G, b->r.as<double>(), u, qv, cutoff, beta, fv, pv,
                        st.d_ionrec.as<double>(), small ? EWB_SMALL + 1 : 0, 0x7fffffff);
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
