// Smooth particle-mesh Ewald reciprocal sum on gfx950: the reciprocal part of
// the reference's PME class (pme.f90:443-478 calling the Darden routines of
// pme_kernel.f90:251-752).  Real space and self term are the Ewald class's
// kernels (ewald.hip); this file replaces its direct structure-factor sum.
//
//   k_pme_key      thread per ion: scaled fractionals fr = K (w - anint(w) +
//                  1/2) with w from the columns of Bbox (as the reference
//                  passes it), the brick of 8^3 grid cells of int(fr)
//   (counting sort of the ions by brick, each brick's ions then put into index
//   order; a radix sort when bricks hold many ions)
//   k_pme_spread   wavefront per brick: B-spline weights of order p
//                  (fill_bspline) and the charges of the brick's ions added
//                  into its (8 + p - 1)^3 points in LDS
//   k_pme_merge    thread per grid point: the sum of the bricks that cover it
//                  (fixed order throughout, no atomics between wavefronts)
//   hipFFT D2Z, then
//   k_pme_energy   thread per point of the half spectrum:
//                  exp(-pi^2 m^2/beta^2)/(B(m) m^2), energy and virial
//                  records, Q *= eterm (m = 0 untouched)
//   hipFFT Z2D, then
//   k_pme_gather   wavefront per brick: the brick's points in LDS, 8 lanes per
//                  ion: potential and field; f += q E, phi += phi_rec.
// The charges are real, so the reference's complex transforms (backward, then
// forward, of which the real part is used) are a real transform and its
// inverse with eterm averaged over m and -m, which differ only where a
// component of m is at the Nyquist index of a sheared cell.
// Grid layout: index g1 + K1 (g2 + K2 g3), the memory order of the
// reference's Q(nfft1, nfft2, nfft3).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include <hipfft/hipfft.h>
#include <rocprim/device/device_radix_sort.hpp>

#include "agpu_internal.hpp"
#include "pme_cell.hpp"
#include "profile.hpp"

namespace agpu {

constexpr int PME_MAXORD = 12;
constexpr int PME_B = 8;            // grid cells per brick edge
// Bytes of the bricks' points that are kept at once.  A brick has p - 1 more
// points per axis than cells, so all of them take 6.6 times the grid at order 8
// and 13.4 times at order 12, up to 115 GB: beyond this the layers of bricks go
// through in parts, at least one at a time (1000 x 1000 points of order 12 have
// 0.86 GB in one).  Parts cost a little: 400^3 points of order 8, 3.4 GB, 1.95 ms
// in one and 2.16 ms in four.
constexpr size_t PME_BRICKS = (size_t)4 << 30;

struct PmeState {
    int order = 8;
    int K[3] = {64, 64, 64};
    bool have_plan = false;
    hipfftHandle plan, plan_inv;
    hipStream_t plan_stream = nullptr;
    int cnt_zero = -1;      // bricks whose counters are zero (k_pme_scan clears what it read)
    DevBuf bsp, key, key_s, idx, idx_s, cnt, start, sort_tmp, brick, grid, spec, partial;
    void drop_plans()
    {
        if (!have_plan) return;
        (void)hipfftDestroy(plan);
        (void)hipfftDestroy(plan_inv);
        have_plan = false;
    }
    ~PmeState() { drop_plans(); }
};

PmeState *pme_state_new(int order, const int *grid)
{
    PmeState *pm = new PmeState();
    pm->order = order;
    for (int d = 0; d < 3; ++d) pm->K[d] = grid[d];
    return pm;
}

void pme_state_free(PmeState *pm) { delete pm; }

// bsp_one_pass (pme_kernel.f90), 0-based
__host__ __device__ __forceinline__ void bsp_one_pass(double *c, double x, int k)
{
    const double div = 1.0 / (k - 1);
    c[k - 1] = div * x * c[k - 2];
    for (int j = 1; j <= k - 2; ++j) c[k - j - 1] = div * ((x + j) * c[k - j - 2] + (k - j - x) * c[k - j - 1]);
    c[0] = div * (1 - x) * c[0];
}

// fill_bspline (pme_kernel.f90): weights c and derivatives d at offset w
__host__ __device__ __forceinline__ void fill_bspline(double w, int order, double *c, double *d)
{
    c[order - 1] = 0.0;
    c[1] = w;
    c[0] = 1.0 - w;
    for (int k = 3; k <= order - 1; ++k) bsp_one_pass(c, w, k);
    d[0] = -c[0];
    for (int j = 1; j < order; ++j) d[j] = c[j - 1] - c[j];
    bsp_one_pass(c, w, order);
}

// cnt (counting sort): the ion's provisional place in its brick; else its
// index, for the radix sort
__global__ void k_pme_key(int nat, const double *__restrict__ r, CellArg B, PmeGrid g, int *__restrict__ key,
                          int *__restrict__ idx, int *__restrict__ cnt)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= nat) return;
    const double x = r[3 * (size_t)n], y = r[3 * (size_t)n + 1], z = r[3 * (size_t)n + 2];
    int ib[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) pme_cell(B, g, e, x, y, z, ib[e]);
    const int b = ib[0] / PME_B + g.nb[0] * (ib[1] / PME_B + g.nb[1] * (ib[2] / PME_B));
    key[n] = b;
    idx[n] = cnt ? atomicAdd(&cnt[b], 1) : n;
}

// exclusive scan of the brick counts, one workgroup (small grids), which
// clears them for the next call
__global__ void __launch_bounds__(1024) k_pme_scan(int n, int *__restrict__ cnt, int *__restrict__ start)
{
    __shared__ int sm[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int total = 0;
    for (int base = 0; base < n; base += 4096) {
        int v[4], sum = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = base + 4 * (int)threadIdx.x + k;
            v[k] = i < n ? cnt[i] : 0;
            if (i < n) cnt[i] = 0;
            sum += v[k];
        }
        int incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        __syncthreads();
        if (lane == 63) sm[wave] = incl;
        __syncthreads();
        int before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            before += w < wave ? sm[w] : 0;
            all += sm[w];
        }
        int at = total + before + incl - sum;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = base + 4 * (int)threadIdx.x + k;
            if (i < n) start[i] = at;
            at += v[k];
        }
        total += all;
    }
    if (threadIdx.x == 0) start[n] = total;
}

__global__ void k_pme_fill(int nat, const int *__restrict__ key, const int *__restrict__ sub,
                           const int *__restrict__ start, int *__restrict__ out)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n < nat) out[start[key[n]] + sub[n]] = n;
}

// A wavefront per brick: its ions into index order.  An ion's place is the
// number of smaller indices: n^2 / 64 comparisons with one lane's value for
// the n ions of a brick.  A brick that holds many of the ions (a cluster in
// vacuum) is gathered from the keys of all ions instead, which are in index
// order, PME_WALK x 64 of them a trip.
constexpr int PME_WALK = 8;

// Comparing takes about 1.9 cycles per n^2 (2000 ions in one brick 3.1 ms, 300
// 79 us), the walk 4.2 per ion of the system (20 040 ions 35 us), so the walk
// is taken from n^2 = 2 nat.  20 000 ions in one brick 306 -> 0.035 ms; 39 304
// of a cluster in a few bricks 20.6 -> 0.056 ms.
__device__ __forceinline__ bool pme_walk(int n, int nat) { return (long long)n * n > 2ll * nat; }

__global__ void __launch_bounds__(256)
k_pme_order(int nat, int nbrick, const int *__restrict__ start, const int *__restrict__ key,
            const int *__restrict__ in, int *__restrict__ out)
{
    const int b = blockIdx.x * 4 + threadIdx.x / 64, lane = threadIdx.x & 63;
    if (b >= nbrick) return;
    const int a0 = start[b], n = start[b + 1] - a0;
    if (n > 64 && pme_walk(n, nat)) {
        int at = a0;
        for (int base = 0; base < nat; base += 64 * PME_WALK) {
            int k[PME_WALK];
#pragma unroll
            for (int c = 0; c < PME_WALK; ++c) {
                const int i = base + 64 * c + lane;
                k[c] = i < nat ? key[i] : -1;
            }
#pragma unroll
            for (int c = 0; c < PME_WALK; ++c) {
                const unsigned long long m = __ballot(k[c] == b);
                if (k[c] == b)
                    out[at + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                       __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                        base + 64 * c + lane;
                at += __popcll(m);
            }
        }
        return;
    }
    for (int c = 0; c < n; c += 64) {
        const int v = c + lane < n ? in[a0 + c + lane] : 0x7fffffff;
        int rank = 0;
        for (int d = 0; d < n; d += 64) {
            const int u = d + lane < n ? in[a0 + d + lane] : 0x7fffffff;
            for (int k = 0; k < min(64, n - d); ++k) rank += __builtin_amdgcn_readlane(u, k) < v;
        }
        if (c + lane < n) out[a0 + rank] = v;
    }
}

// Plane stride of a brick's points in LDS, E^2 and a pad: the fewest bank
// conflicts (32 banks of 8 bytes per half wavefront) of the p^2 rows that the
// lanes add at once.
constexpr int pme_conflicts(int p, int e, int plane)
{
    int sum = 0;
    for (int base = 0; base < p * p; base += 32) {
        int hit[32] = {}, top = 0;
        for (int l = base; l < base + 32 && l < p * p; ++l) {
            const int k = ((l % p) * e + (l / p) * plane) % 32;
            if (++hit[k] > top) top = hit[k];
        }
        sum += top;
    }
    return sum;
}

constexpr int pme_plane(int p)
{
    const int e = PME_B + p - 1;
    int best = e * e;
    for (int pad = 1; pad < 32; ++pad)
        if (pme_conflicts(p, e, e * e + pad) < pme_conflicts(p, e, best)) best = e * e + pad;
    return best;
}

// first sorted ion of every brick (start[nbrick] = nat)
__global__ void k_pme_start(int nat, int nbrick, const int *__restrict__ key_s, int *__restrict__ start)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p > nat) return;
    const int kprev = p == 0 ? -1 : key_s[p - 1], kcur = p == nat ? nbrick : key_s[p];
    for (int c = kprev + 1; c <= kcur; ++c) start[c] = p;
}

// a brick's edges: its first cell per axis
__device__ __forceinline__ void pme_brick(const PmeGrid &g, int b, int (&o)[3])
{
    o[0] = PME_B * (b % g.nb[0]);
    o[1] = PME_B * ((b / g.nb[0]) % g.nb[1]);
    o[2] = PME_B * (b / (g.nb[0] * g.nb[1]));
}

// Q(g) = sum over the ions n of q_n theta1(t1) theta2(t2) theta3(t3) at
// g = cell - (p - 1) + t (fill_charge_grid).  One wavefront per brick: its
// ions' stencils lie inside the brick and p - 1 points before it, which are
// kept in LDS.  An ion's p^2 (t2, t3) rows go to the lanes, which add their p
// points along x; the points of one instruction differ, and one wavefront's
// LDS operations are carried out in order, so the sums have a fixed order.
// Bound by the LDS adds (512 of 8 bytes per ion at order 8).  216 000 ions,
// order 8, 160^3 points: 106 us and 56 us for the merge (814 us as a gather by
// grid point, which looked up 64 ranges of ions for 27 ions that reach it).
template <int ORD>
__global__ void __launch_bounds__(64)
k_pme_spread(PmeGrid g, CellArg B, int first, const int *__restrict__ start, const int *__restrict__ idx,
             const double *__restrict__ r, const double *__restrict__ q, double *__restrict__ brick)
{
    constexpr int E = PME_B + ORD - 1, P = pme_plane(ORD), NI = 16;
    __shared__ double box[E * P];
    __shared__ double th[NI][3][ORD];
    __shared__ int at[NI];
    __shared__ double qs[NI];
    const int lane = threadIdx.x, b = first + blockIdx.x;
    int o[3];
    pme_brick(g, b, o);
    for (int t = lane; t < E * P; t += 64) box[t] = 0.0;
    const int a0 = start[b], a1 = start[b + 1];
    for (int base = a0; base < a1; base += NI) {
        const int m = min(NI, a1 - base);
        wave_sync();
        // weights: a lane per ion and axis
        if (lane < 4 * NI) {
            const int k = lane >> 2, e = lane & 3;
            int off = 0;
            if (k < m && e < 3) {
                const int n = idx[base + k];
                int ib;
                const double x =
                    pme_cell(B, g, e, r[3 * (size_t)n], r[3 * (size_t)n + 1], r[3 * (size_t)n + 2], ib);
                double c[ORD], d[ORD];
                fill_bspline(x, ORD, c, d);
#pragma unroll
                for (int t = 0; t < ORD; ++t) th[k][e][t] = c[t];
                off = (ib - o[e]) * (e == 0 ? 1 : e == 1 ? E : P);
                if (e == 0) qs[k] = q[n];
            }
            off += __shfl_xor(off, 1, 64);
            off += __shfl_xor(off, 2, 64);
            if (e == 0) at[k] = off;
        }
        wave_sync();
        for (int k = 0; k < m; ++k) {
            const int p0 = at[k];
            const double qk = qs[k];
            for (int pr = lane; pr < ORD * ORD; pr += 64) {
                const int t2 = pr % ORD, t3 = pr / ORD;
                const double w = th[k][1][t2] * th[k][2][t3] * qk;
                double *p = box + p0 + t2 * E + t3 * P;
#pragma unroll
                for (int t1 = 0; t1 < ORD; ++t1)
                    __hip_atomic_fetch_add(p + t1, th[k][0][t1] * w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
    }
    wave_sync();
    double *out = brick + (size_t)blockIdx.x * (E * E * E);
    for (int t = lane; t < E * E * E; t += 64) out[t] = box[t / (E * E) * P + t % (E * E)];
}

// Grid point g is in the bricks whose cells start at most p - 1 after it and
// end no earlier than it; before the first cell the grid wraps.  PART: only the
// bricks of layers l0 .. l1 - 1 are there, and are added to the points of the
// nz planes that they reach.
template <int ORD, bool PART>
__global__ void __launch_bounds__(256)
k_pme_merge(PmeGrid g, int l0, int l1, int nz, const double *__restrict__ brick, double *__restrict__ grid)
{
    constexpr int E = PME_B + ORD - 1;
    long long ind = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (ind >= (long long)g.K[0] * g.K[1] * nz) return;
    if (PART) {
        const long long plane = (long long)g.K[0] * g.K[1];
        ind = wrapi(PME_B * l0 - (ORD - 1) + (int)(ind / plane), g.K[2]) * plane + ind % plane;
    }
    const int p[3] = {(int)(ind % g.K[0]), (int)((ind / g.K[0]) % g.K[1]),
                      (int)(ind / ((long long)g.K[0] * g.K[1]))};
    // per axis: bricks b0 .. b1 with the point itself, then 0 .. c1 with the
    // point one period down
    int b0[3], nb[3], nt[3];
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        b0[e] = p[e] / PME_B;
        nb[e] = min(g.nb[e] - 1, (p[e] + ORD - 1) / PME_B) - b0[e] + 1;
        const int d = p[e] - g.K[e] + ORD - 1;
        nt[e] = nb[e] + (d >= 0 ? min(g.nb[e] - 1, d / PME_B) + 1 : 0);
    }
    double sum = 0.0;
    for (int z = 0; z < nt[2]; ++z) {
        const int bz = z < nb[2] ? b0[2] + z : z - nb[2];
        if (PART && (bz < l0 || bz >= l1)) continue;
        const int lz = (z < nb[2] ? p[2] : p[2] - g.K[2]) - PME_B * bz + ORD - 1;
        for (int y = 0; y < nt[1]; ++y) {
            const int by = y < nb[1] ? b0[1] + y : y - nb[1];
            const int ly = (y < nb[1] ? p[1] : p[1] - g.K[1]) - PME_B * by + ORD - 1;
            for (int x = 0; x < nt[0]; ++x) {
                const int bx = x < nb[0] ? b0[0] + x : x - nb[0];
                const int lx = (x < nb[0] ? p[0] : p[0] - g.K[0]) - PME_B * bx + ORD - 1;
                const size_t b = bx + (size_t)g.nb[0] * (by + (size_t)g.nb[1] * (PART ? bz - l0 : bz));
                sum += brick[b * (E * E * E) + (lz * E + ly) * E + lx];
            }
        }
    }
    grid[ind] = PART ? grid[ind] + sum : sum;
}

// energy_and_virial_sum (pme_kernel.f90): records [e, W column-major] of
// the already scaled (1 / (2 pi V)) terms; Q(m) *= eterm except m = 0.  Thread
// = point of the half spectrum k1 <= K1 / 2; inside, it stands for -k as well.
__global__ void __launch_bounds__(256)
k_pme_energy(PmeGrid g, CellArg B, const double *__restrict__ bsp, double fac, double pre,
             double2 *__restrict__ spec, double *__restrict__ partial)
{
    __shared__ double s_red[4][7];
    const int K1 = g.K[0], K2 = g.K[1], K3 = g.K[2], H = K1 / 2 + 1;
    const long long ind = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    double v[7] = {0, 0, 0, 0, 0, 0, 0};
    if (ind > 0 && ind < (long long)H * K2 * K3) {
        const int k1 = (int)(ind % H), k2 = (int)((ind / H) % K2), k3 = (int)(ind / ((long long)H * K2));
        const double2 Q = spec[ind];
        const double q2 = (Q.x * Q.x + Q.y * Q.y) * pre;
        const double bm = bsp[k1] * bsp[K1 + k2] * bsp[K1 + K2 + k3];
        // one term of the full spectrum at index (c1, c2, c3); its modulus
        // factors are even in the index
        auto term = [&](int c1, int c2, int c3, double weight) {
            const double m1 = c1 < (K1 + 1) / 2 ? c1 : c1 - K1, m2 = c2 < (K2 + 1) / 2 ? c2 : c2 - K2,
                         m3 = c3 < (K3 + 1) / 2 ? c3 : c3 - K3;
            // mhat = recip . m
            const double mh1 = B.A[0] * m1 + B.A[3] * m2 + B.A[6] * m3;
            const double mh2 = B.A[1] * m1 + B.A[4] * m2 + B.A[7] * m3;
            const double mh3 = B.A[2] * m1 + B.A[5] * m2 + B.A[8] * m3;
            const double msq = mh1 * mh1 + mh2 * mh2 + mh3 * mh3;
            const double eterm = exp(-fac * msq) / (bm * msq);
            const double vterm = 2.0 * (fac * msq + 1.0) / msq;
            const double es = eterm * q2 * weight;
            v[0] += es;
            v[1] += es * (vterm * mh1 * mh1 - 1.0);
            v[2] += es * (vterm * mh2 * mh2 - 1.0);
            v[3] += es * (vterm * mh3 * mh3 - 1.0);
            v[4] += es * (vterm * mh1 * mh2);
            v[5] += es * (vterm * mh1 * mh3);
            v[6] += es * (vterm * mh2 * mh3);
            return eterm;
        };
        const bool inside = k1 > 0 && 2 * k1 < K1;     // -k is not in the half spectrum
        const bool nyq = 2 * k1 == K1 || 2 * k2 == K2 || 2 * k3 == K3;
        double e = term(k1, k2, k3, inside && !nyq ? 2.0 : 1.0);
        if (nyq) {
            const int c1 = k1 ? K1 - k1 : 0, c2 = k2 ? K2 - k2 : 0, c3 = k3 ? K3 - k3 : 0;
            e = 0.5 * (e + term(c1, c2, c3, inside ? 1.0 : 0.0));
        }
        spec[ind] = make_double2(e * Q.x, e * Q.y);
    }
#pragma unroll
    for (int q = 0; q < 7; ++q) v[q] = group_sum<64>(v[q]);
    const int wave = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0)
        for (int q = 0; q < 7; ++q) s_red[wave][q] = v[q];
    __syncthreads();
    if (threadIdx.x < 7) {
        const int q = threadIdx.x;
        const double t = ((s_red[0][q] + s_red[1][q]) + s_red[2][q]) + s_red[3][q];
        double *rec = partial + (size_t)blockIdx.x * 10;
        if (q == 0) rec[0] = t;
        else if (q == 1) rec[1 + 0] = t;
        else if (q == 2) rec[1 + 4] = t;
        else if (q == 3) rec[1 + 8] = t;
        else if (q == 4) { rec[1 + 1] = t; rec[1 + 3] = t; }
        else if (q == 5) { rec[1 + 2] = t; rec[1 + 6] = t; }
        else { rec[1 + 5] = t; rec[1 + 7] = t; }
    }
}

// potential_and_field_sum (pme_kernel.f90): f += q E, phi += phi_rec.  One
// workgroup per brick, its points in LDS; a wavefront takes 8 ions at a time,
// 8 lanes per ion, which share its p planes of p^2 points.  216 000 ions at
// order 8: 98 us (352 us with a thread per ion reading the grid and stored
// weights; 286 us with one wavefront per brick, four of which fit a CU).
template <int ORD>
__global__ void __launch_bounds__(256)
k_pme_gather(PmeGrid g, CellArg B, const int *__restrict__ start, const int *__restrict__ idx,
             const double *__restrict__ r, const double *__restrict__ q, const double *__restrict__ grid, double fac,
             double *__restrict__ f, double *__restrict__ phi)
{
    constexpr int E = PME_B + ORD - 1, E3 = E * E * E, NI = 8;
    __shared__ double box[E3];
    __shared__ double thw[4][NI][6][ORD];
    __shared__ int atw[4][NI];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, b = blockIdx.x;
    const int a0 = start[b], a1 = start[b + 1];
    if (a0 == a1) return;
    int o[3];
    pme_brick(g, b, o);
    for (int t = threadIdx.x; t < E3; t += 256) {
        // points before the first cell wrap (p <= K); no ion's stencil takes
        // those past the last one
        int x = o[0] - (ORD - 1) + t % E, y = o[1] - (ORD - 1) + (t / E) % E, z = o[2] - (ORD - 1) + t / (E * E);
        x = x < 0 ? x + g.K[0] : min(x, g.K[0] - 1);
        y = y < 0 ? y + g.K[1] : min(y, g.K[1] - 1);
        z = z < 0 ? z + g.K[2] : min(z, g.K[2] - 1);
        box[t] = grid[x + (size_t)g.K[0] * (y + (size_t)g.K[1] * z)];
    }
    __syncthreads();
    double (&th)[NI][6][ORD] = thw[wave];
    int (&at)[NI] = atw[wave];
    for (int base = a0 + NI * wave; base < a1; base += 4 * NI) {
        const int m = min(NI, a1 - base);
        wave_sync();
        if (lane < 4 * NI) {
            const int k = lane >> 2, e = lane & 3;
            int off = 0;
            if (k < m && e < 3) {
                const int n = idx[base + k];
                int ib;
                const double x =
                    pme_cell(B, g, e, r[3 * (size_t)n], r[3 * (size_t)n + 1], r[3 * (size_t)n + 2], ib);
                double c[ORD], d[ORD];
                fill_bspline(x, ORD, c, d);
#pragma unroll
                for (int t = 0; t < ORD; ++t) {
                    th[k][e][t] = c[t];
                    th[k][3 + e][t] = d[t];
                }
                off = (ib - o[e]) * (e == 0 ? 1 : e == 1 ? E : E * E);
            }
            off += __shfl_xor(off, 1, 64);
            off += __shfl_xor(off, 2, 64);
            if (e == 0) at[k] = off;
        }
        wave_sync();
        const int sub = lane & 7;
        {
            const int k = lane >> 3;
            double f0 = 0.0, f1 = 0.0, f2 = 0.0, f3 = 0.0;
            if (k < m) {
                double t1[ORD], d1[ORD];
#pragma unroll
                for (int t = 0; t < ORD; ++t) {
                    t1[t] = th[k][0][t];
                    d1[t] = th[k][3][t];
                }
                const double *p0 = box + at[k];
                for (int t3 = sub; t3 < ORD; t3 += 8) {
                    double g0 = 0.0, g1 = 0.0, g2 = 0.0;
#pragma unroll
                    for (int t2 = 0; t2 < ORD; ++t2) {
                        const double *p = p0 + t2 * E + t3 * E * E;
                        double s = 0.0, d = 0.0;
#pragma unroll
                        for (int t = 0; t < ORD; ++t) {
                            s = fma(p[t], t1[t], s);
                            d = fma(p[t], d1[t], d);
                        }
                        const double w = th[k][1][t2];
                        g0 = fma(s, w, g0);
                        g1 = fma(d, w, g1);
                        g2 = fma(s, th[k][4][t2], g2);
                    }
                    const double w = th[k][2][t3];
                    f0 = fma(g0, w, f0);
                    f1 = fma(g1, w, f1);
                    f2 = fma(g2, w, f2);
                    f3 = fma(g0, th[k][5][t3], f3);
                }
            }
            f0 = group_sum<8>(f0);
            f1 = group_sum<8>(f1);
            f2 = group_sum<8>(f2);
            f3 = group_sum<8>(f3);
            if (k < m && sub == 0) {
                const int n = idx[base + k];
                f1 *= -g.K[0];
                f2 *= -g.K[1];
                f3 *= -g.K[2];
                if (phi) phi[n] += fac * f0;
                if (f) {
                    const double qn = q[n];
                    f[3 * (size_t)n + 0] += qn * (fac * (B.A[0] * f1 + B.A[3] * f2 + B.A[6] * f3));
                    f[3 * (size_t)n + 1] += qn * (fac * (B.A[1] * f1 + B.A[4] * f2 + B.A[7] * f3));
                    f[3 * (size_t)n + 2] += qn * (fac * (B.A[2] * f1 + B.A[5] * f2 + B.A[8] * f3));
                }
            }
        }
    }
}

// layers of bricks whose points are kept at once
static int pme_layers(const PmeGrid &g, int order)
{
    const size_t e = PME_B + order - 1, layer = sizeof(double) * e * e * e * g.nb[0] * g.nb[1];
    return (int)std::min<size_t>(g.nb[2], std::max<size_t>(1, PME_BRICKS / layer));
}

template <int ORD>
static int pme_spread_gather(bool gather, const PmeGrid &g, const PmeState *pm, const double *r, const double *q,
                             const CellArg &B, double fac, double *f, double *phi, hipStream_t s)
{
    const unsigned layer = (unsigned)g.nb[0] * g.nb[1], nbrick = layer * g.nb[2];
    if (!gather) {
        const int nl = pme_layers(g, ORD);
        if (nl < g.nb[2]) AGPU_CHECK(zero_dev(pm->grid.ptr, sizeof(double) * (size_t)g.K[0] * g.K[1] * g.K[2]));
        for (int l0 = 0; l0 < g.nb[2]; l0 += nl) {
            const int l1 = std::min(l0 + nl, g.nb[2]);
            const int nz = nl < g.nb[2] ? std::min(PME_B * (l1 - l0) + ORD - 1, g.K[2]) : g.K[2];
            const dim3 gm((unsigned)(((long long)g.K[0] * g.K[1] * nz + 255) / 256));
            AGPU_LAUNCH("pme_spread", k_pme_spread<ORD>, dim3(layer * (l1 - l0)), dim3(64), 0, s, g, B, layer * l0,
                        pm->start.as<int>(), pm->idx_s.as<int>(), r, q, pm->brick.as<double>());
            AGPU_LAUNCH("pme_merge", (nl < g.nb[2] ? k_pme_merge<ORD, true> : k_pme_merge<ORD, false>), gm, dim3(256),
                        0, s, g, l0, l1, nz, pm->brick.as<double>(), pm->grid.as<double>());
        }
    } else
        AGPU_LAUNCH("pme_gather", k_pme_gather<ORD>, dim3(nbrick), dim3(256), 0, s, g, B, pm->start.as<int>(),
                    pm->idx_s.as<int>(), r, q, pm->grid.as<double>(), fac, f, phi);
    return AGPU_OK;
}

static int pme_order_dispatch(int order, bool gather, const PmeGrid &g, const PmeState *pm, const double *r,
                              const double *q, const CellArg &B, double fac, double *f, double *phi, hipStream_t s)
{
    switch (order) {
    case 3: return pme_spread_gather<3>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 4: return pme_spread_gather<4>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 5: return pme_spread_gather<5>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 6: return pme_spread_gather<6>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 7: return pme_spread_gather<7>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 8: return pme_spread_gather<8>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 9: return pme_spread_gather<9>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 10: return pme_spread_gather<10>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 11: return pme_spread_gather<11>(gather, g, pm, r, q, B, fac, f, phi, s);
    case 12: return pme_spread_gather<12>(gather, g, pm, r, q, B, fac, f, phi, s);
    default: return set_error(AGPU_ERR_ARG, "PME: order must be 3 .. 12");
    }
}

// load_bsp_moduli / dftmod (pme_kernel.f90) on the host
static void bsp_moduli(int K, int order, std::vector<double> &mod)
{
    double arr[PME_MAXORD], darr[PME_MAXORD];
    fill_bspline(0.0, order, arr, darr);
    std::vector<double> bsp(K, 0.0);
    for (int i = 1; i <= order && i < K; ++i) bsp[i] = arr[i - 1];
    mod.assign(K, 0.0);
    const double twopi = 2.0 * M_PI;
    for (int k = 0; k < K; ++k) {
        double s1 = 0.0, s2 = 0.0;
        for (int j = 0; j < K; ++j) {
            const double arg = twopi * k * j / K;
            s1 = s1 + bsp[j] * std::cos(arg);
            s2 = s2 + bsp[j] * std::sin(arg);
        }
        mod[k] = s1 * s1 + s2 * s2;
    }
    for (int k = 0; k < K; ++k)
        if (mod[k] < 1e-7) mod[k] = 0.5 * (mod[(k + K - 1) % K] + mod[(k + 1) % K]);
}

int pme_recip(PmeState *pm, const agpu_particles *p, const double *q, double beta, double *rec10, double *f,
              double *phi)
{
    const int nat = p->nat;
    const int K1 = pm->K[0], K2 = pm->K[1], K3 = pm->K[2], order = pm->order;
    const long long ng = (long long)K1 * K2 * K3, nh = (long long)(K1 / 2 + 1) * K2 * K3;
    hipStream_t s = stream();
    if (!pm->have_plan || pm->plan_stream != s) {
        pm->drop_plans();
        if (hipfftPlan3d(&pm->plan, K3, K2, K1, HIPFFT_D2Z) != HIPFFT_SUCCESS)
            return set_error(AGPU_ERR_HIP, "PME: hipfftPlan3d failed");
        if (hipfftPlan3d(&pm->plan_inv, K3, K2, K1, HIPFFT_Z2D) != HIPFFT_SUCCESS) {
            (void)hipfftDestroy(pm->plan);
            return set_error(AGPU_ERR_HIP, "PME: hipfftPlan3d failed");
        }
        pm->have_plan = true;
        if (hipfftSetStream(pm->plan, s) != HIPFFT_SUCCESS || hipfftSetStream(pm->plan_inv, s) != HIPFFT_SUCCESS) {
            pm->drop_plans();
            return set_error(AGPU_ERR_HIP, "PME: hipfftSetStream failed");
        }
        pm->plan_stream = s;
        std::vector<double> all, m;
        for (int d = 0; d < 3; ++d) {
            bsp_moduli(pm->K[d], order, m);
            all.insert(all.end(), m.begin(), m.end());
        }
        AGPU_CHECK(pm->bsp.reserve(sizeof(double) * all.size()));
        AGPU_HIP(hipMemcpyAsync(pm->bsp.ptr, all.data(), sizeof(double) * all.size(), hipMemcpyHostToDevice, s));
    }
    PmeGrid g;
    for (int d = 0; d < 3; ++d) {
        g.K[d] = pm->K[d];
        g.nb[d] = (pm->K[d] + PME_B - 1) / PME_B;
    }
    const int nbrick = g.nb[0] * g.nb[1] * g.nb[2];
    const size_t edge = PME_B + order - 1;
    AGPU_CHECK(pm->grid.reserve(sizeof(double) * (size_t)ng));
    AGPU_CHECK(pm->spec.reserve(sizeof(double2) * (size_t)nh));
    const int nblk_g = (int)((nh + 255) / 256);
    AGPU_CHECK(pm->partial.reserve(sizeof(double) * 10 * (size_t)nblk_g));
    CellArg B;
    std::memcpy(B.A, p->cell.B, sizeof B.A);
    const double *A = p->cell.A;
    const double V = std::fabs(A[0] * (A[4] * A[8] - A[5] * A[7]) - A[1] * (A[3] * A[8] - A[5] * A[6]) +
                               A[2] * (A[3] * A[7] - A[4] * A[6]));
    AGPU_CHECK(zero_dev(rec10, sizeof(double) * 10));
    if (nat > 0) {
        AGPU_CHECK(pm->key.reserve(sizeof(int) * (size_t)nat));
        AGPU_CHECK(pm->key_s.reserve(sizeof(int) * (size_t)nat));
        AGPU_CHECK(pm->idx.reserve(sizeof(int) * (size_t)nat));
        AGPU_CHECK(pm->idx_s.reserve(sizeof(int) * (size_t)nat));
        AGPU_CHECK(pm->start.reserve(sizeof(int) * (size_t)(nbrick + 1)));
        AGPU_CHECK(pm->brick.reserve(sizeof(double) * edge * edge * edge * g.nb[0] * g.nb[1] * pme_layers(g, order)));
        const dim3 ga((nat + 255) / 256);
        // The counting sort takes 4 launches (216 000 ions in 8000 bricks:
        // 25 us; the radix sort, 16 launches, 92 us).  Its scan is one
        // workgroup's and its ordering quadratic in an ordinary brick's ions:
        // large grids and bricks that are full on the average keep the radix
        // sort.
        if (nbrick <= 32768 && nat <= 96ll * nbrick) {
            if (pm->cnt_zero != nbrick) {
                AGPU_CHECK(pm->cnt.reserve(sizeof(int) * (size_t)nbrick));
                AGPU_CHECK(zero_dev(pm->cnt.ptr, sizeof(int) * (size_t)nbrick));
            }
            pm->cnt_zero = -1;
            AGPU_LAUNCH("pme_key", k_pme_key, ga, dim3(256), 0, s, nat, p->d_r, B, g, pm->key.as<int>(),
                        pm->idx.as<int>(), pm->cnt.as<int>());
            AGPU_LAUNCH("pme_scan", k_pme_scan, dim3(1), dim3(1024), 0, s, nbrick, pm->cnt.as<int>(),
                        pm->start.as<int>());
            pm->cnt_zero = nbrick;
            AGPU_LAUNCH("pme_fill", k_pme_fill, ga, dim3(256), 0, s, nat, pm->key.as<int>(), pm->idx.as<int>(),
                        pm->start.as<int>(), pm->key_s.as<int>());
            AGPU_LAUNCH("pme_order", k_pme_order, dim3((nbrick + 3) / 4), dim3(256), 0, s, nat, nbrick,
                        pm->start.as<int>(), pm->key.as<int>(), pm->key_s.as<int>(), pm->idx_s.as<int>());
        } else {
            AGPU_LAUNCH("pme_key", k_pme_key, ga, dim3(256), 0, s, nat, p->d_r, B, g, pm->key.as<int>(),
                        pm->idx.as<int>(), (int *)nullptr);
            int bits = 1;
            while ((1ll << bits) < nbrick) ++bits;
            size_t tmp = 0;
            AGPU_HIP(rocprim::radix_sort_pairs(nullptr, tmp, pm->key.as<int>(), pm->key_s.as<int>(),
                                               pm->idx.as<int>(), pm->idx_s.as<int>(), (size_t)nat, 0, bits, s));
            AGPU_CHECK(pm->sort_tmp.reserve(tmp + 16));
            AGPU_HIP(rocprim::radix_sort_pairs(pm->sort_tmp.ptr, tmp, pm->key.as<int>(), pm->key_s.as<int>(),
                                               pm->idx.as<int>(), pm->idx_s.as<int>(), (size_t)nat, 0, bits, s));
            AGPU_LAUNCH("pme_start", k_pme_start, dim3((nat + 256) / 256), dim3(256), 0, s, nat, nbrick,
                        pm->key_s.as<int>(), pm->start.as<int>());
        }
        AGPU_CHECK(pme_order_dispatch(order, false, g, pm, p->d_r, q, B, 0.0, nullptr, nullptr, s));
    } else {
        AGPU_CHECK(zero_dev(pm->grid.ptr, sizeof(double) * (size_t)ng));
    }
    if (hipfftExecD2Z(pm->plan, pm->grid.as<double>(), pm->spec.as<hipfftDoubleComplex>()) != HIPFFT_SUCCESS)
        return set_error(AGPU_ERR_HIP, "PME: forward FFT failed");
    AGPU_LAUNCH("pme_energy", k_pme_energy, dim3(nblk_g), dim3(256), 0, s, g, B, pm->bsp.as<double>(),
                M_PI * M_PI / (beta * beta), 1.0 / (2.0 * M_PI * V), pm->spec.as<double2>(),
                pm->partial.as<double>());
    if (nat > 0 && (f || phi)) {
        if (hipfftExecZ2D(pm->plan_inv, pm->spec.as<hipfftDoubleComplex>(), pm->grid.as<double>()) != HIPFFT_SUCCESS)
            return set_error(AGPU_ERR_HIP, "PME: backward FFT failed");
        AGPU_CHECK(pme_order_dispatch(order, true, g, pm, p->d_r, q, B, 1.0 / (M_PI * V), f, phi, s));
    }
    AGPU_CHECK(reduce_ev(pm->partial.as<double>(), nblk_g, 10, rec10, rec10 + 1, nullptr));
    return AGPU_OK;
}

}  // namespace agpu
