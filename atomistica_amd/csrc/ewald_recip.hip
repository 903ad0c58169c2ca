// Direct reciprocal Ewald sum as matrix products on the FP64 matrix cores.
//
//   E = (4 pi / V) sum_k c(k) |S(k)|^2,  c(k) = exp(-k^2 / 4 beta^2) / k^2,
//   S(k) = sum_j q_j exp(i k.r_j),  k = 2 pi Bbox^T n over the half space,
//   phi_j = (8 pi / V) Re sum_k conj(c S) exp(i k.r_j)
// (the reference's PME class sums the same series on a mesh,
// pme_kernel.f90:251-752).
//
// With s = Bbox r the phase factorises, exp(2 pi i n.s) = e(n1, n2) e(n3), so
// for a set of columns (n1, n2) the sum over the ions is a matrix product of
// the column phases (columns x ions) with cos and sin of 2 pi m s3 (ions x m),
// n3 = n3c +- m:
//   S(n3c + m) = (XC - YS) + i (XS + YC),   S(n3c - m) = (XC + YS) + i (YC - XS)
// with X + iY = q e(n1, n2, n3c), C + iS = e(m): four real products give two k.
// The way back is the product over m of conj(c S), combined for +-m into
// u, v, p, w, with C and S, per column and ion (G, and M with the factor m),
// after which the column phase is applied once per column:
//   phi_j ~ Re e G,  F_j ~ (n1, n2, n3c) Im e G + (0, 0, 1) Im e M.
// So S(k) costs 2 and the forces 4 fused multiply-adds per ion and half-space
// k; both run as v_mfma_f64_16x16x4 with the phases formed beside them.
//
// Columns come in patches of 4 x 4 (e = e(patch) e(a, b), a, b < 4: one
// sincospi per patch and ion, and 16 per ion shared by all patches), m in
// tiles of 8 (C in lanes 0-7, S in lanes 8-15 of a 16-wide operand) for S(k)
// and in steps of 4 (the product's depth) for the forces.  On a sphere of
// radius R (in units of the reciprocal lattice) this pads the work by 1.5 at
// R = 25, 1.12 at R = 93 for S(k) and by 1.36, 1.09 for the forces; 16-wide
// rows of columns padded more (1.9, 1.19 and worse below).  n3c centres each
// patch's range of n3, which a sheared cell shifts away from zero.
//
// Measured on 216 000 ions, 1.72 M k: S(k) 29.3 ms and forces 49.9 ms
// (137 and 248 ms with a complex rotation per ion and k on the VALU); the
// products alone take 23 and 44.5 ms at the 72.5 TFLOP/s of a large FP64 matrix
// product.  FP64 VALU and matrix instructions do not overlap here, so what is
// left is the phases and the epilogues beside the products.  256 cells of
// 64-4096 ions: 1.2 and 1.85 ms (5.2 and 7.1 ms).  The sums of a split of the
// ions are added in turn, which rounds less than one running sum over all
// ions: forces of 6400 ions differ from 80-bit sums by 9.7e-15 (4.6e-14 with
// the running sum), those of 216 000 ions from pairwise sums by 5.9e-14
// (1.8e-13).
#include <algorithm>
#include <cmath>
#include <cstring>

#include "ewald_recip.hpp"
#include "profile.hpp"

namespace agpu {

constexpr int EWR_TMAX = 12;            // 8-wide tiles of m per item
constexpr int EWR_MMAX = 8 * EWR_TMAX;  // m per item
constexpr int EWR_ST = 8;               // tiles of a workgroup of S(k): 128 accumulator registers, no spills
constexpr int EWR_IC = 32;              // ions per LDS chunk of S(k)
constexpr int EWR_ROW = 8 * EWR_ST + 8; // LDS row of e(m): 8 more, so that rows of consecutive ions start half the banks apart
constexpr int EWR_SW = 4;               // waves (items) per workgroup of S(k)
constexpr int EWR_FW = 4;               // waves (16 ions each) per workgroup of the forces
constexpr int EWR_FI = 16 * EWR_FW;
constexpr int EWR_FT = EWR_TMAX / 2;    // tiles of an item that the forces take through LDS at a time

typedef double v4d __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4d mfma64(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// n s less the nearest whole number of turns, the product taken exactly
__device__ __forceinline__ double ewr_turn(double n, double s)
{
    const double p = n * s;
    return (p - rint(p)) + fma(n, s, -p);
}

__device__ __forceinline__ double2 ewr_expi(double turns)
{
    double2 e;
    sincospi(2.0 * (turns - rint(turns)), &e.y, &e.x);
    return e;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b)
{
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// geometry per structure: b_d[x] (9), 4 pi / V, and the reciprocal vectors
// 2 pi b_d[x] (9) as the host formed them for the choice of the k
constexpr int EWR_GEO = 20;

// s = Bbox r less whole turns, and the charge
__global__ void k_ewr_frac(int n, const int *__restrict__ sof, const double *__restrict__ geo,
                           const double *__restrict__ r, const double *__restrict__ q, double4 *__restrict__ s4)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const double *b = geo + (sof ? EWR_GEO * (size_t)sof[j] : 0);
    const double x = r[3 * (size_t)j], y = r[3 * (size_t)j + 1], z = r[3 * (size_t)j + 2];
    double s[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        s[d] = b[3 * d] * x + b[3 * d + 1] * y + b[3 * d + 2] * z;
        s[d] -= rint(s[d]);
    }
    s4[j] = make_double4(s[0], s[1], s[2], q[j]);
}

// ---------------------------------------------------------------------------
// S(k)
// ---------------------------------------------------------------------------
struct EwrSLds {
    double2 e3[EWR_IC][EWR_ROW];    // e(m) per ion
    double2 e12[EWR_IC][16];        // e(a, b) per ion
    double2 pq[EWR_SW][EWR_IC];     // q e(n1, n2, n3c) per wave's patch and ion
};

template <int NT>
__device__ __forceinline__ void ewr_sk_body(EwrSLds &L, const EwrSBlock &B, const EwrItem &I, int wave,
                                            const EwrItem *__restrict__ items, const double4 *__restrict__ s4, double *__restrict__ S)
{
    const int lane = threadIdx.x & 63;
    v4d acc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t][0] = acc[t][1] = (v4d){0.0, 0.0, 0.0, 0.0};
    // 8 threads per ion stage it: one sincospi each, for the four waves'
    // patches and the four phases that the rest are products of
    const int si = threadIdx.x >> 3, sb = threadIdx.x & 7;
    double x1 = 0.0, x2 = 0.0, x3 = 0.0;
    if (sb < EWR_SW) {
        const EwrItem &P = items[B.item + min(sb, B.nitem - 1)];
        x1 = P.n1;
        x2 = P.n2;
        x3 = P.n3c;
    } else if (sb == 4) {
        x1 = 1.0;
    } else if (sb == 5) {
        x2 = 1.0;
    } else {
        x3 = sb == 6 ? 1 : I.mb + 8 * B.t0;
    }
    const int c = lane & 15, k = lane >> 4;
    const int boff = 2 * (c & 7) + (c >> 3);      // C of m = c, or S of m = c - 8
    for (int base = B.a0; base < B.a1; base += EWR_IC) {
        __syncthreads();
        {
            const double4 a = base + si < B.a1 ? s4[base + si] : make_double4(0.0, 0.0, 0.0, 0.0);
            const double2 p = ewr_expi(ewr_turn(x1, a.x) + ewr_turn(x2, a.y) + ewr_turn(x3, a.z));
            if (sb < EWR_SW) L.pq[sb][si] = make_double2(a.w * p.x, a.w * p.y);
            const double2 one = make_double2(1.0, 0.0);
            const double2 f1 = make_double2(__shfl(p.x, 4, 8), __shfl(p.y, 4, 8));
            const double2 f2 = make_double2(__shfl(p.x, 5, 8), __shfl(p.y, 5, 8));
            const double2 g1 = make_double2(__shfl(p.x, 6, 8), __shfl(p.y, 6, 8));
            double2 e = make_double2(__shfl(p.x, 7, 8), __shfl(p.y, 7, 8));
            // m = mb + sb + 8 t: e(mb) e(s3)^sb, then by rotation with e(8 s3)
            const double2 g2 = cmul(g1, g1), g4 = cmul(g2, g2), w = cmul(g4, g4);
            e = cmul(e, sb & 1 ? g1 : one);
            e = cmul(e, cmul(sb & 2 ? g2 : one, sb & 4 ? g4 : one));
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                L.e3[si][8 * t + sb] = e;
                e = cmul(e, w);
            }
            // column a * 4 + b of a patch: a s1 + b s2; a and a + 2
            double2 f = cmul(sb & 1 ? f2 : one, sb & 2 ? cmul(f2, f2) : one);
            f = cmul(f, sb & 4 ? f1 : one);
            L.e12[si][sb] = f;
            L.e12[si][sb + 8] = cmul(f, cmul(f1, f1));
        }
        __syncthreads();
#pragma unroll
        for (int st = 0; st < EWR_IC / 4; ++st) {
            const int ion = 4 * st + k;
            const double2 x = cmul(L.pq[wave][ion], L.e12[ion][c]);
            const double *row = reinterpret_cast<const double *>(L.e3[ion]) + boff;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const double b = row[16 * t];
                acc[t][0] = mfma64(x.x, b, acc[t][0]);
                acc[t][1] = mfma64(x.y, b, acc[t][1]);
            }
        }
    }
    if (wave >= B.nitem) return;
    // per tile: {X, Y} products, 4 accumulator rows, 64 lanes
    double *o = S + ((size_t)I.stile + B.t0 + (size_t)B.split * I.sstride) * 512 + lane;
    const int nt = I.nt - B.t0;
#pragma unroll
    for (int t = 0; t < NT; ++t)
        if (t < nt)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int g = 0; g < 4; ++g) o[((t * 2 + h) * 4 + g) * 64] = acc[t][h][g];
}

// A workgroup's four patches share the staged e(m) and e(a, b) of a chunk of
// ions; each wave multiplies its patch with the workgroup's tiles.
__global__ void __launch_bounds__(64 * EWR_SW, 2)
k_ewr_sk(const EwrSBlock *__restrict__ blks, const EwrItem *__restrict__ items, const double4 *__restrict__ s4,
         double *__restrict__ S)
{
    __shared__ __align__(16) EwrSLds L;
    const EwrSBlock B = blks[blockIdx.x];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const EwrItem I = items[B.item + min(wave, B.nitem - 1)];
    switch (B.nt) {
    case 1: ewr_sk_body<1>(L, B, I, wave, items, s4, S); break;
    case 2: ewr_sk_body<2>(L, B, I, wave, items, s4, S); break;
    case 3: ewr_sk_body<3>(L, B, I, wave, items, s4, S); break;
    case 4: ewr_sk_body<4>(L, B, I, wave, items, s4, S); break;
    case 5: ewr_sk_body<5>(L, B, I, wave, items, s4, S); break;
    case 6: ewr_sk_body<6>(L, B, I, wave, items, s4, S); break;
    case 7: ewr_sk_body<7>(L, B, I, wave, items, s4, S); break;
    default: ewr_sk_body<EWR_ST>(L, B, I, wave, items, s4, S); break;
    }
}

// Thread = (column, m) of a tile: the splits' sums, c(k), energy and virial
// record of the tile, and the coefficients of the way back,
//   {u, v} = {a + a', b - b'}, {p, -w} = {a - a', -(b + b')},
// a + ib = c S(n3c + m), a' + ib' = c S(n3c - m), as rows [m][column].
__global__ void __launch_bounds__(128)
k_ewr_energy(const int2 *__restrict__ map, const EwrItem *__restrict__ items, const double *__restrict__ geo,
             double kmax2, double inv4b2, const double *__restrict__ S, double2 *__restrict__ T,
             double *__restrict__ rec)
{
    __shared__ double red[2][7];
    const int2 mt = map[blockIdx.x];
    const EwrItem I = items[mt.x];
    const double *G = geo + EWR_GEO * (size_t)I.s;
    const int col = threadIdx.x & 15, mm = threadIdx.x >> 4;
    const int m = I.mb + 8 * mt.y + mm;
    // accumulator row of column i: register i / 4, lanes 16 (i % 4) + ...
    const int at = (col >> 2) * 64 + (col & 3) * 16 + mm;
    double xc = 0.0, xs = 0.0, yc = 0.0, ys = 0.0;
    for (int sp = 0; sp < I.nsplit; ++sp) {
        const double *p = S + ((size_t)I.stile + mt.y + (size_t)sp * I.sstride) * 512 + at;
        xc += p[0];
        xs += p[8];
        yc += p[256];
        ys += p[264];
    }
    const int n1 = I.n1 + (col >> 2), n2 = I.n2 + (col & 3);
    const double pref = G[9];
    double v[7] = {0, 0, 0, 0, 0, 0, 0};
    double ta[2] = {0.0, 0.0}, tb[2] = {0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int n3 = h ? I.n3c - m : I.n3c + m;
        bool use = n1 > 0 || (n1 == 0 && (n2 > 0 || (n2 == 0 && n3 > 0)));
        if (h && m == 0) use = false;
        {
#pragma clang fp contract(off)
            // the operations of the host's choice of columns, in its order
            double kh[3];
            for (int x = 0; x < 3; ++x)
                kh[x] = ((double)n1 * G[10 + x] + (double)n2 * G[13 + x]) + (double)n3 * G[16 + x];
            const double kh2 = (kh[0] * kh[0] + kh[1] * kh[1]) + kh[2] * kh[2];
            use = use && kh2 <= kmax2;
        }
        if (!use) continue;
        const double sr = h ? xc + ys : xc - ys, si = h ? yc - xs : xs + yc;
        double kv[3];
#pragma unroll
        for (int x = 0; x < 3; ++x)
            kv[x] = 2.0 * M_PI * ((double)n1 * G[x] + (double)n2 * G[3 + x] + (double)n3 * G[6 + x]);
        const double k2 = kv[0] * kv[0] + kv[1] * kv[1] + kv[2] * kv[2];
        const double c = exp(-k2 * inv4b2) / k2;
        ta[h] = c * sr;
        tb[h] = c * si;
        const double ek = pref * c * (sr * sr + si * si);
        const double fac = 2.0 * (inv4b2 + 1.0 / k2);
        v[0] += ek;
        v[1] += ek * (fac * kv[0] * kv[0] - 1.0);
        v[2] += ek * (fac * kv[1] * kv[1] - 1.0);
        v[3] += ek * (fac * kv[2] * kv[2] - 1.0);
        v[4] += ek * fac * kv[0] * kv[1];
        v[5] += ek * fac * kv[0] * kv[2];
        v[6] += ek * fac * kv[1] * kv[2];
    }
    double2 *o = T + (size_t)I.tile * 256 + mt.y * 128 + threadIdx.x;
    o[0] = make_double2(ta[0] + ta[1], tb[0] - tb[1]);
    o[I.nt * 128] = make_double2(ta[0] - ta[1], -(tb[0] + tb[1]));
#pragma unroll
    for (int c = 0; c < 7; ++c) v[c] = group_sum<64>(v[c]);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int c = 0; c < 7; ++c) red[threadIdx.x >> 6][c] = v[c];
    __syncthreads();
    if (threadIdx.x < 10) {
        // {e, W column-major} from {e, xx, yy, zz, xy, xz, yz}
        constexpr int from[10] = {0, 1, 4, 5, 4, 2, 6, 5, 6, 3};
        rec[(size_t)(I.tile + mt.y) * 10 + threadIdx.x] = red[0][from[threadIdx.x]] + red[1][from[threadIdx.x]];
    }
}

// ---------------------------------------------------------------------------
// forces and potential
// ---------------------------------------------------------------------------
// The coefficients of an item's tiles [t0, t0 + EWR_FT), 16 bytes a lane,
// straight into LDS (64 lanes' worth per wave and trip; a tile is two of
// them in each of its two arrays): {u, v} rows, then {p, -w} rows
__device__ __forceinline__ void ewr_fetch(const double2 *__restrict__ T, const EwrItem &I, int t0, double2 *lds,
                                          int wave, int lane)
{
    const int n = 2 * min(I.nt - t0, EWR_FT);
    const double2 *src = T + (size_t)I.tile * 256 + t0 * 128 + lane;
    for (int q = wave; q < 2 * n; q += EWR_FW) {
        const int at = q < n ? q * 64 : I.nt * 128 + (q - n) * 64;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + at),
                                         (__attribute__((address_space(3))) void *)(lds + q * 64), 16, 0, 0);
    }
}

struct EwrAcc {
    v4d gr, gi, mr, mi, nr, ni;    // G; M = (mr - nr) + i (mi - ni)
};

// steps [S0, S0 + 2 EWR_FT) of an item with ks of them: a depth of 4 m each
template <int S0>
__device__ __forceinline__ void ewr_force_steps(const double2 *__restrict__ uvp, int rows, int ks, double md,
                                                const double2 (&cs)[EWR_MMAX / 4], EwrAcc &A)
{
    const double2 *pwp = uvp + rows;
    double2 uv = uvp[0], pw = pwp[0];
#pragma unroll
    for (int q = 0; q < 2 * EWR_FT; ++q) {
        if (S0 + q < ks) {
            // the next step's coefficients; past the item's end some other
            // word of the buffer, not used
            double2 uvn = uv, pwn = pw;
            if (q + 1 < 2 * EWR_FT) {
                uvn = uvp[(q + 1) * 64];
                pwn = pwp[(q + 1) * 64];
            }
            const double c = cs[S0 + q].x, s = cs[S0 + q].y;
            const double mc = md * c, ms = md * s;
            A.gr = mfma64(uv.x, c, A.gr);
            A.gi = mfma64(pw.x, s, A.gi);
            A.mr = mfma64(pw.x, mc, A.mr);
            A.mi = mfma64(uv.x, ms, A.mi);
            A.gr = mfma64(uv.y, s, A.gr);
            A.gi = mfma64(pw.y, c, A.gi);
            A.nr = mfma64(pw.y, ms, A.nr);
            A.ni = mfma64(uv.y, mc, A.ni);
            md += 4.0;
            uv = uvn;
            pw = pwn;
        }
    }
}

// A wave keeps cos and sin of m s3 of its 16 ions for the 96 m of a group in
// registers and walks the patches; the coefficients go through LDS, shared by
// the workgroup's four waves and fetched one half item ahead.  Two such
// workgroups fit a CU, and their waves meet at no common barrier, so that one
// multiplies while the other applies its column phases (one workgroup of
// eight waves left the matrix cores idle there).
__global__ void __launch_bounds__(64 * EWR_FW, 2)
k_ewr_force(const EwrFBlock *__restrict__ blks, const EwrItem *__restrict__ items, const double4 *__restrict__ s4,
            const double2 *__restrict__ T, double4 *__restrict__ part)
{
    __shared__ __align__(16) double2 sT[2][EWR_FT * 256];
    const EwrFBlock B = blks[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = B.a0 + 16 * wave + (lane & 15), k = lane >> 4;
    const bool act = j < B.a1, busy = B.a0 + 16 * wave < B.a1;
    const double4 a = s4[act ? j : B.a0];
    // column r * 4 + k of a patch (accumulator row r, lane group k)
    double2 e12[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) e12[r] = ewr_expi(ewr_turn(r, a.x) + ewr_turn(k, a.y));
    double2 cs[EWR_MMAX / 4], ep = make_double2(0.0, 0.0);
    int mb = -1, cur = 0;
    double a1 = 0.0, a2 = 0.0, a3 = 0.0, ap = 0.0;
    EwrItem I = items[B.i0];
    ewr_fetch(T, I, 0, sT[0], wave, lane);
    for (int it = B.i0; it < B.i1; ++it) {
        const EwrItem N = items[min(it + 1, B.i1 - 1)];
        const bool two = I.nt > EWR_FT;
        // the coefficients have arrived, and every wave is done with the
        // other buffer, which takes the next ones
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (two) ewr_fetch(T, I, EWR_FT, sT[cur ^ 1], wave, lane);
        else if (it + 1 < B.i1) ewr_fetch(T, N, 0, sT[cur ^ 1], wave, lane);
        if (I.mb != mb) {
            mb = I.mb;
#pragma unroll
            for (int st = 0; st < EWR_MMAX / 4; ++st)
                if (st < I.nt * 2) cs[st] = ewr_expi(ewr_turn(mb + 4 * st + k, a.z));
        }
        // the phases of four patches at a time, one per lane group
        const int q = (it - B.i0) & 3;
        if (q == 0) {
            const EwrItem &P = items[min(it + k, B.i1 - 1)];
            ep = ewr_expi(ewr_turn(P.n1, a.x) + ewr_turn(P.n2, a.y) + ewr_turn(P.n3c, a.z));
        }
        EwrAcc A;
        A.gr = A.gi = A.mr = A.mi = A.nr = A.ni = (v4d){0.0, 0.0, 0.0, 0.0};
        if (busy) ewr_force_steps<0>(sT[cur] + lane, 128 * min(I.nt, EWR_FT), I.ks, mb + k, cs, A);
        cur ^= 1;
        if (two) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            if (it + 1 < B.i1) ewr_fetch(T, N, 0, sT[cur ^ 1], wave, lane);
            if (busy)
                ewr_force_steps<2 * EWR_FT>(sT[cur] + lane, 128 * (I.nt - EWR_FT), I.ks, mb + 8 * EWR_FT + k, cs, A);
            cur ^= 1;
        }
        const int from = 16 * q + (lane & 15);
        const double2 e0 = make_double2(__shfl(ep.x, from, 64), __shfl(ep.y, from, 64));
        double g = 0.0, g1 = 0.0, gm = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const double2 e = cmul(e0, e12[r]);
            ap += e.x * A.gr[r] - e.y * A.gi[r];
            const double im = e.x * A.gi[r] + e.y * A.gr[r];
            g += im;
            g1 += r * im;
            gm += e.x * (A.mi[r] - A.ni[r]) + e.y * (A.mr[r] - A.nr[r]);
        }
        a1 += (double)I.n1 * g + g1;
        a2 += (double)(I.n2 + k) * g;
        a3 += (double)I.n3c * g + gm;
        I = N;
    }
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
        a1 += __shfl_xor(a1, o, 64);
        a2 += __shfl_xor(a2, o, 64);
        a3 += __shfl_xor(a3, o, 64);
        ap += __shfl_xor(ap, o, 64);
    }
    if (act && lane < 16) part[B.rec + j] = make_double4(a1, a2, a3, ap);
}

// f += q E and phi += phi_rec from the ions' partial sums, as many as the ion's
// structure has splits
__global__ void k_ewr_apply(int nat, const int *__restrict__ sof, const EwrFRec *__restrict__ frec,
                            const double *__restrict__ geo, const double4 *__restrict__ s4,
                            const double4 *__restrict__ part, double *__restrict__ f, double *__restrict__ phi)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nat) return;
    const int s = sof ? sof[j] : 0;
    const EwrFRec R = frec[s];
    const double *G = geo + EWR_GEO * (size_t)s;
    double a1 = 0.0, a2 = 0.0, a3 = 0.0, ap = 0.0;
    for (int k = 0; k < R.nsplit; ++k) {
        const double4 v = part[R.rec + (long long)k * R.n + j];
        a1 += v.x;
        a2 += v.y;
        a3 += v.z;
        ap += v.w;
    }
    const double pref2 = 2.0 * G[9];
    if (f) {
        const double fq = pref2 * s4[j].w * 2.0 * M_PI;
#pragma unroll
        for (int x = 0; x < 3; ++x) f[3 * (size_t)j + x] += fq * (a1 * G[x] + a2 * G[3 + x] + a3 * G[6 + x]);
    }
    if (phi) phi[j] += pref2 * ap;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
// the patches of one structure with their ranges of n3
static int ewr_patches(int s, const double *A, const double (&b)[3][3], double kmax, std::vector<EwrItem> &out)
{
    int nmax[3];
    for (int d = 0; d < 3; ++d) {
        const double *a = A + 3 * d;
        const double len = std::sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
        nmax[d] = (int)std::floor(kmax * len / (2.0 * M_PI)) + 1;
        if (nmax[d] > 500) return set_error(AGPU_ERR_ARG, "Ewald: more than 500 k-vectors per axis");
    }
    const double b33 = b[2][0] * b[2][0] + b[2][1] * b[2][1] + b[2][2] * b[2][2];
    for (int p1 = 0; p1 <= nmax[0]; p1 += 4)
        for (int p2 = -4 * ((nmax[1] + 3) / 4); p2 <= nmax[1]; p2 += 4) {
            int lo = 1 << 20, hi = -(1 << 20);
            for (int n1 = p1; n1 < p1 + 4; ++n1)
                for (int n2 = p2; n2 < p2 + 4; ++n2) {
                    if (n1 > nmax[0] || n2 > nmax[1] || n2 < -nmax[1] || (n1 == 0 && n2 < 0)) continue;
                    double pp = 0.0, pb = 0.0;
                    for (int x = 0; x < 3; ++x) {
                        const double v = n1 * b[0][x] + n2 * b[1][x];
                        pp += v * v;
                        pb += v * b[2][x];
                    }
                    // |p + n3 b3| <= kmax, a little wide: the energy pass decides per k
                    const double c = -pb / b33, h2 = c * c - (pp - kmax * kmax * (1.0 + 1e-12)) / b33;
                    if (h2 < 0.0) continue;
                    const double h = std::sqrt(h2) + 1e-9;
                    const int l = std::max(-nmax[2], (int)std::ceil(c - h)), u = std::min(nmax[2], (int)std::floor(c + h));
                    if (u < l || (n1 == 0 && n2 == 0 && u < 1)) continue;
                    lo = std::min(lo, l);
                    hi = std::max(hi, u);
                }
            if (hi < lo) continue;
            EwrItem I{};
            I.n1 = p1;
            I.n2 = p2;
            I.n3c = (int)std::floor(0.5 * (lo + hi));
            const int M = std::max(hi - I.n3c, I.n3c - lo);
            for (I.mb = 0; I.mb <= M; I.mb += EWR_MMAX) {
                const int cnt = std::min(EWR_MMAX, M + 1 - I.mb);
                I.nt = (cnt + 7) / 8;
                I.ks = (cnt + 3) / 4;
                I.s = s;
                out.push_back(I);
            }
        }
    return AGPU_OK;
}

template <typename T> static int ewr_upload(DevBuf &d, const std::vector<T> &h, hipStream_t s)
{
    AGPU_CHECK(d.reserve(sizeof(T) * (h.size() + 1)));
    if (!h.empty()) AGPU_HIP(hipMemcpyAsync(d.ptr, h.data(), sizeof(T) * h.size(), hipMemcpyHostToDevice, s));
    return AGPU_OK;
}

int ewr_plan(EwrState &st, int ns, const double *cells, const int *off, double kmax)
{
    st.items.clear();
    st.sblk.clear();
    st.fblk.clear();
    st.tile0.assign(ns + 1, 0);
    std::vector<double> geo((size_t)EWR_GEO * ns, 0.0);
    std::vector<int> item0(ns + 1, 0);
    std::vector<EwrFRec> frec(ns);
    std::vector<int2> map;
    long long tiles = 0, stiles = 0, swork = 0, fwork = 0;
    for (int s = 0; s < ns; ++s) {
        const double *A = cells + 9 * (size_t)s;
        double Bi[9], b[3][3];
        AGPU_CHECK(compute_inverse(A, Bi));
        double *g = &geo[(size_t)EWR_GEO * s];
        for (int d = 0; d < 3; ++d)
            for (int x = 0; x < 3; ++x) {
                g[3 * d + x] = Bi[3 * x + d];
                b[d][x] = 2.0 * M_PI * Bi[3 * x + d];
                g[10 + 3 * d + x] = b[d][x];
            }
        g[9] = 4.0 * M_PI / std::fabs(A[0] * (A[4] * A[8] - A[5] * A[7]) - A[1] * (A[3] * A[8] - A[5] * A[6]) +
                                      A[2] * (A[3] * A[7] - A[4] * A[6]));
        item0[s] = (int)st.items.size();
        AGPU_CHECK(ewr_patches(s, A, b, kmax, st.items));
        if (off[s + 1] == off[s]) st.items.resize(item0[s]);   // no ions: no terms
        // waves of a workgroup take neighbouring items: similar ranges of m
        std::sort(st.items.begin() + item0[s], st.items.end(), [](const EwrItem &x, const EwrItem &y) {
            if (x.mb != y.mb) return x.mb < y.mb;
            if (x.ks != y.ks) return x.ks > y.ks;
            return x.n1 != y.n1 ? x.n1 < y.n1 : x.n2 < y.n2;
        });
        st.tile0[s] = (int)tiles;
        const long long n = off[s + 1] - off[s];
        for (size_t k = item0[s]; k < st.items.size(); ++k) {
            st.items[k].tile = (int)tiles;
            tiles += st.items[k].nt;
            swork += n * st.items[k].nt;
            fwork += ((n + EWR_FI - 1) / EWR_FI) * (st.items[k].ks + 2);
        }
        if (tiles > (1ll << 30)) return set_error(AGPU_ERR_ARG, "Ewald: too many k-vectors");
    }
    item0[ns] = (int)st.items.size();
    st.tile0[ns] = (int)tiles;
    st.ntile = (int)tiles;
    // Work per workgroup: S(k) in (ion, tile) units of its four waves, forces
    // in steps, so that each kernel has about 12 workgroups per resident place
    // (512 of either), but no less than costs its set-up.
    const long long starget = std::max(swork / (EWR_SW * 512ll * 12), 64ll * 2);
    const long long ftarget = std::max(fwork / (512ll * 12), 24ll);
    st.nfrec = 0;
    for (int s = 0; s < ns; ++s) {
        const int a0 = off[s], n = off[s + 1] - off[s];
        const int nt_s = st.tile0[s + 1] - st.tile0[s];
        frec[s] = EwrFRec{0, n, 0};
        if (nt_s == 0) continue;
        // splits of the ions: by the structure's largest item, whole LDS chunks
        int ntm = 1;
        long long fw = 0;
        for (int k = item0[s]; k < item0[s + 1]; ++k) {
            ntm = std::max(ntm, st.items[k].nt);
            fw += st.items[k].ks + 2;
        }
        long long nsp = ((long long)n * ntm + starget - 1) / starget;
        nsp = std::max(1ll, std::min(nsp, (long long)(n + 2 * EWR_IC - 1) / (2 * EWR_IC)));
        const int per = (int)(((n + nsp - 1) / nsp + EWR_IC - 1) / EWR_IC) * EWR_IC;
        const int nsplit = (n + per - 1) / per;
        long long so = stiles;
        for (int k = item0[s]; k < item0[s + 1]; ++k) {
            st.items[k].nsplit = nsplit;
            st.items[k].sstride = nt_s;
            st.items[k].stile = (int)so;
            so += st.items[k].nt;
        }
        stiles += (long long)nt_s * nsplit;
        if (stiles > 0x7fffffffll) return set_error(AGPU_ERR_ARG, "Ewald: too many k-vectors");
        for (int k = item0[s]; k < item0[s + 1];) {
            int c = 1;
            while (c < EWR_SW && k + c < item0[s + 1] && st.items[k + c].mb == st.items[k].mb) ++c;
            int nt = 0;
            for (int t = 0; t < c; ++t) nt = std::max(nt, st.items[k + t].nt);
            // more than EWR_ST tiles: two workgroups of half of them each
            const int step = nt > EWR_ST ? (nt + 1) / 2 : nt;
            for (int t0 = 0; t0 < nt; t0 += step)
                for (int sp = 0; sp < nsplit; ++sp)
                    st.sblk.push_back(EwrSBlock{k, c, a0 + sp * per, std::min(a0 + n, a0 + (sp + 1) * per), sp, t0,
                                                std::min(step, nt - t0), 0});
            k += c;
        }
        // splits of the items for the forces: equal steps
        const int ni = item0[s + 1] - item0[s];
        int nf = (int)std::max(1ll, std::min((fw + ftarget - 1) / ftarget, (long long)ni));
        std::vector<int> cut(1, item0[s]);
        long long acc = 0;
        for (int k = item0[s]; k < item0[s + 1]; ++k) {
            acc += st.items[k].ks + 2;
            if (acc * nf >= fw * (long long)cut.size() && k + 1 < item0[s + 1]) cut.push_back(k + 1);
        }
        nf = (int)cut.size();
        cut.push_back(item0[s + 1]);
        frec[s].nsplit = nf;
        frec[s].rec = st.nfrec - a0;
        st.nfrec += (long long)nf * n;
        for (int sp = 0; sp < nf; ++sp)
            for (int a = 0; a < n; a += EWR_FI)
                st.fblk.push_back(EwrFBlock{a0 + a, std::min(a0 + n, a0 + a + EWR_FI), cut[sp], cut[sp + 1],
                                            frec[s].rec + (long long)sp * n, 0});
    }
    // the longest workgroups first
    auto fcost = [&](const EwrFBlock &x) {
        return st.items[x.i1 - 1].tile + st.items[x.i1 - 1].nt - st.items[x.i0].tile;
    };
    std::stable_sort(st.sblk.begin(), st.sblk.end(), [](const EwrSBlock &x, const EwrSBlock &y) {
        return (long long)x.nt * (x.a1 - x.a0) > (long long)y.nt * (y.a1 - y.a0);
    });
    std::stable_sort(st.fblk.begin(), st.fblk.end(),
                     [&](const EwrFBlock &x, const EwrFBlock &y) { return fcost(x) > fcost(y); });
    map.reserve(st.ntile);
    for (size_t k = 0; k < st.items.size(); ++k)
        for (int t = 0; t < st.items[k].nt; ++t) map.push_back(make_int2((int)k, t));
    hipStream_t hs = stream();
    AGPU_CHECK(ewr_upload(st.d_items, st.items, hs));
    AGPU_CHECK(ewr_upload(st.d_sblk, st.sblk, hs));
    AGPU_CHECK(ewr_upload(st.d_fblk, st.fblk, hs));
    AGPU_CHECK(ewr_upload(st.d_map, map, hs));
    AGPU_CHECK(ewr_upload(st.d_geo, geo, hs));
    AGPU_CHECK(ewr_upload(st.d_frec, frec, hs));
    AGPU_CHECK(ewr_upload(st.d_tile0, st.tile0, hs));
    AGPU_CHECK(st.S.reserve(sizeof(double) * 512 * (size_t)(stiles + 1)));
    AGPU_CHECK(st.T.reserve(sizeof(double2) * 256 * (size_t)(tiles + 1)));
    AGPU_HIP(hipStreamSynchronize(hs));
    return AGPU_OK;
}

int ewr_run(EwrState &st, int nat, const double *r, const double *q, const int *sof, double kmax, double beta,
            double *rec, double *f, double *phi)
{
    if (nat == 0 || st.ntile == 0) return AGPU_OK;
    hipStream_t s = stream();
    const double *geo = st.d_geo.as<double>();
    const EwrItem *items = st.d_items.as<EwrItem>();
    AGPU_CHECK(st.s4.reserve(sizeof(double4) * (size_t)nat));
    double4 *s4 = st.s4.as<double4>();
    AGPU_LAUNCH("ewald_frac", k_ewr_frac, dim3((nat + 255) / 256), dim3(256), 0, s, nat, sof, geo, r, q, s4);
    AGPU_LAUNCH("ewald_sk", k_ewr_sk, dim3((unsigned)st.sblk.size()), dim3(64 * EWR_SW), 0, s,
                st.d_sblk.as<EwrSBlock>(), items, s4, st.S.as<double>());
    AGPU_LAUNCH("ewald_kenergy", k_ewr_energy, dim3(st.ntile), dim3(128), 0, s, st.d_map.as<int2>(), items, geo,
                kmax * kmax, 1.0 / (4.0 * beta * beta), st.S.as<double>(), st.T.as<double2>(), rec);
    if (!f && !phi) return AGPU_OK;
    AGPU_CHECK(st.fpart.reserve(sizeof(double4) * (size_t)st.nfrec));
    AGPU_LAUNCH("ewald_kforce", k_ewr_force, dim3((unsigned)st.fblk.size()), dim3(64 * EWR_FW), 0, s,
                st.d_fblk.as<EwrFBlock>(), items, s4, st.T.as<double2>(), st.fpart.as<double4>());
    AGPU_LAUNCH("ewald_kapply", k_ewr_apply, dim3((nat + 255) / 256), dim3(256), 0, s, nat, sof,
                st.d_frec.as<EwrFRec>(), geo, s4, st.fpart.as<double4>(), f, phi);
    return AGPU_OK;
}

}  // namespace agpu
