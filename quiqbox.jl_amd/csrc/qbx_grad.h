// qbx_grad.h -- adjoint ERI kernels of libqbx_hip.so (gfx950): the two-electron
// part of the RHF energy gradient with respect to the basis parameters.
//
// For every unique contracted shell quartet (the screened task lists of the
// Fock build, one wave per bra pair and 64 of its kets) the kernel
//   1. forms the seeds G = f (4 D_ab D_cd - D_ac D_bd - D_ad D_bc) s_a s_b s_c s_d
//      on the contracted (ab|cd) (D the total density, f the 8-fold degeneracy
//      of the unique quartet, s the component scales), so that the sum of
//      G (ab|cd) over all unique quartets is the two-electron energy
//      sum (1/2 D_mn D_ls - 1/4 D_ml D_ns) (mn|ls) over all index quartets;
//      for UHF (nset = 2: D holds D, D_alpha, D_beta) the exchange part is
//      2 sum_s (D^s_ac D^s_bd + D^s_ad D^s_bc), i.e. the energy
//      sum (1/2 D_mn D_ls - 1/2 sum_s D^s_ml D^s_ns) (mn|ls), which is the
//      RHF form when D_alpha = D_beta = D/2;
//   2. transposes the horizontal recurrence (EriAdj::hrr_adj): seeds on the
//      contracted [e0|f0], which need no integral;
//   3. runs one primitive loop: the vertical recurrence forward (the contracted
//      [e0|f0] are summed for step 4) and in reverse (EriAdj::vrr_adj_grp), and
//      the adjoint of the geometry, Boys function (dF_m/dT = -F_{m+1}) and
//      prefactor, down to the exponents a, b, c, d and the centres A, B, C, D of
//      the primitive quartet;
//   4. forms the seeds again (cheaper than holding them through the loop) and
//      from them and the contracted [e0|f0] the derivatives with respect to A-B
//      and C-D.
// Per radial primitive k of each shell it accumulates dE/d(alpha_k) at fixed
// weights and c_k dE/dc_k (the seeded value of the primitive quartets that
// contain k), per shell dE/d(centre).  The bra's primitive pairs are the outer
// loop, so its sums are wave-wide scalars reduced once per bra primitive pair; the
// kets' go to LDS sums per radial primitive with ds_add_f64, four per primitive
// quartet, and each block of a persistent grid adds its LDS sums to the result
// once.  (Register sums per lane and radial primitive, selected with a compare
// per slot, cost 190 VALU instructions a primitive quartet and 128 registers, and
// every lane's sums went out as global atomics on some 700 addresses.)  Measured on
// the 32-atom, 128-function s/p cluster (16 primitive pairs a shell pair), classes
// one after another: 40 ms before; 9.5 ms for the whole gradient call now, the
// classes concurrently.
#pragma once
#include "qbx_eri.h"

template <int LA, int LB, int LC, int LD> struct EriAdj;

namespace qbx {

struct GeomAdj {
    double da, db, dc, dd;
    double dA[3], dB[3], dC[3], dD[3];
};

// Adjoint of the primitive-quartet set-up.  Forward: p = a + b, P = (aA + bB)/p,
// PA = P - A, K_p = c_a c_b exp(-ab/p |A-B|^2)/p (likewise q, Q, QC, K_q), s =
// (p+q)^{-1/2}, PQ = P - Q, rho = pq/(p+q), T = rho |PQ|^2, pref = 2 pi^{5/2}
// K_p K_q s, F_m = pref B_m(T), WP = -q/(p+q) PQ, WQ = p/(p+q) PQ, inv2p =
// 1/2p, inv2q = 1/2q, inv2pq = 1/(2(p+q)), rho_p = q/(p+q), rho_q = p/(p+q).
// Given Fb[m] = dL/dF_m and bin[] = dL/d(PA, WP, QC, WQ, inv2p, inv2q, inv2pq,
// rho_p, rho_q), returns dL/d(a, b, c, d, A, B, C, D).  B_m for m <= LT + 1; ip =
// 1/p, iq = 1/q (thirty divisions a primitive quartet otherwise).
template <int LT>
__device__ __forceinline__ GeomAdj geom_adjoint(double a, double b, double c, double d, double ip, double iq,
                                                const double* PA, const double* QC, const double* AB,
                                                const double* CD, const double* PQ, double pref, double inv,
                                                const double* Bm, const double* Fb, const double* bin)
{
    const double p = a + b, q = c + d;
    const double rho_p = q * inv, rho_q = p * inv, rho = p * rho_p;
    const double R2 = PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2];
    double bpref = 0.0, bT = 0.0;
#pragma unroll
    for (int m = 0; m <= LT; ++m) {
        bpref += Fb[m] * Bm[m];
        bT -= Fb[m] * Bm[m + 1];
    }
    bT *= pref;
    const double blnK = bpref * pref;     // d pref / d ln K_p = d pref / d ln K_q = pref
    const double brho = bT * R2;
    double bPQ[3];
    double brho_p = bin[15], brho_q = bin[16];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        bPQ[t] = 2.0 * rho * bT * PQ[t] - rho_p * bin[3 + t] + rho_q * bin[9 + t];
        brho_p -= bin[3 + t] * PQ[t];
        brho_q += bin[9 + t] * PQ[t];
    }
    double bp = (brho * q + brho_q) * inv;
    double bq = (brho * p + brho_p) * inv;
    // inv = s^2 = 1/(p+q): d pref / d inv = pref / (2 inv)
    const double binv = brho * p * q + brho_p * q + brho_q * p + 0.5 * bin[14] + 0.5 * blnK * (p + q);
    const double ip2 = ip * ip, iq2 = iq * iq;
    bp -= binv * inv * inv + 0.5 * bin[12] * ip2;
    bq -= binv * inv * inv + 0.5 * bin[13] * iq2;
    GeomAdj g;
    // P = (aA + bB)/p: dP/da = (A - P)/p = -PA/p, dP/db = (B - P)/p = -(AB + PA)/p
    const double ab2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
    const double cd2 = CD[0] * CD[0] + CD[1] * CD[1] + CD[2] * CD[2];
    const double ap = a * ip, bo = b * ip, cq = c * iq, dq = d * iq;
    const double mu2 = 2.0 * a * bo * blnK, nu2 = 2.0 * c * dq * blnK;
    double ga = 0.0, gb = 0.0, gc = 0.0, gd = 0.0;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const double bP = bPQ[t] + bin[t];     // PQ = P - Q, PA = P - A
        const double bQ = -bPQ[t] + bin[6 + t];
        ga += bP * PA[t];
        gb += bP * (AB[t] + PA[t]);
        gc += bQ * QC[t];
        gd += bQ * (CD[t] + QC[t]);
        // ln K_p = ln c_a c_b - (ab/p)|A-B|^2 - ln p
        g.dA[t] = ap * bP - bin[t] - mu2 * AB[t];
        g.dB[t] = bo * bP + mu2 * AB[t];
        g.dC[t] = cq * bQ - bin[6 + t] - nu2 * CD[t];
        g.dD[t] = dq * bQ + nu2 * CD[t];
    }
    g.da = bp - ip * ga - blnK * (bo * bo * ab2 + ip);
    g.db = bp - ip * gb - blnK * (ap * ap * ab2 + ip);
    g.dc = bq - iq * gc - blnK * (dq * dq * cd2 + iq);
    g.dd = bq - iq * gd - blnK * (cq * cq * cd2 + iq);
    return g;
}

// Where a block's sums go: its LDS copy of the three outputs (sums: g_xpn, g_lin,
// g_cen in a row), or the outputs themselves where the copy does not fit.
struct GradSink {
    double* sums;
    double *x, *l, *c;
    int nr;
    bool lds;
    __device__ __forceinline__ GradSink(const EriArgs& a, double* s)
        : sums(s), x(a.g_xpn), l(a.g_lin), c(a.g_cen), nr(a.n_radial), lds(a.grad_lds > 0) {}
    __device__ __forceinline__ void xpn(int k, double v) const { lds ? (void)atomicAdd(sums + k, v) : (void)atomicAdd(x + k, v); }
    __device__ __forceinline__ void lin(int k, double v) const { lds ? (void)atomicAdd(sums + nr + k, v) : (void)atomicAdd(l + k, v); }
    __device__ __forceinline__ void cen(int k, double v) const { lds ? (void)atomicAdd(sums + 2 * nr + k, v) : (void)atomicAdd(c + k, v); }
};

// Seeds G on the contracted integrals of one shell quartet (f: its degeneracy weight).
template <int NA, int NB, int NC, int ND>
__device__ __forceinline__ void grad_seeds(const EriArgs& a, cptr<DevShell> SA, cptr<DevShell> SB, const DevShell* SC,
                                           const DevShell* SD, double f, double* G)
{
    const size_t N = (size_t)a.N;
    const double* D = a.D;
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
        for (int ib = 0; ib < NB; ++ib)
#pragma unroll
            for (int ic = 0; ic < NC; ++ic)
#pragma unroll
                for (int id = 0; id < ND; ++id) {
                    const int m = max(SA->bf[ia], 0), n = max(SB->bf[ib], 0);
                    const int l = max(SC->bf[ic], 0), s = max(SD->bf[id], 0);
                    const double sc = SA->sc[ia] * SB->sc[ib] * SC->sc[ic] * SD->sc[id];
                    double gam;
                    if (a.nset == 2) {
                        const double* Da = D + N * N;
                        const double* Db = D + 2 * N * N;
                        gam = 4.0 * D[m * N + n] * D[l * N + s] -
                              2.0 * (Da[m * N + l] * Da[n * N + s] + Db[m * N + l] * Db[n * N + s] +
                                     Da[m * N + s] * Da[n * N + l] + Db[m * N + s] * Db[n * N + l]);
                    } else {
                        gam = 4.0 * D[m * N + n] * D[l * N + s] - D[m * N + l] * D[n * N + s] -
                              D[m * N + s] * D[n * N + l];
                    }
                    G[((ia * NB + ib) * NC + ic) * ND + id] = f * sc * gam;
                }
}

// Bound by FP64 issue (and, for (pp|pp), by its register file: group GR of the
// class's seeds, see GRAD_GROUPS in gen_eri.py).
template <int LA, int LB, int LC, int LD, int GR>
__global__ __launch_bounds__(256) void eri_grad_kernel(EriArgs a)
{
    using Adj = EriAdj<LA, LB, LC, LD>;
    constexpr int NA = qbx_ncart(LA), NB = qbx_ncart(LB), NC = qbx_ncart(LC), ND = qbx_ncart(LD);
    constexpr int LT = LA + LB + LC + LD;
    constexpr int NACC = Adj::NACC;
    constexpr int NINT = Adj::NINT;
    __shared__ double2 sboys[BOYS_HEAD2 + boys_rows(LT + 1) * QBX_BOYSL_STRIDE / 2];
    extern __shared__ double sums[];    // [grad_lds]: g_xpn, g_lin, g_cen
    stage_boys<256, boys_rows(LT + 1)>(sboys, a.boysl);    // rows of order LT + 1
    for (int i = threadIdx.x; i < a.grad_lds; i += 256) sums[i] = 0.0;
    __syncthreads();
    const double* sb = (const double*)sboys + BOYS_HEAD;
    const GradSink sink(a, sums);

    const int lane = (int)threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const cptr<int> cpre = cst(a.cpre);
    for (int wave = (int)blockIdx.x * 4 + wib; wave < a.nwave; wave += (int)gridDim.x * 4) {
        int lo = 0, hi = a.nbra;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (cpre[mid] <= wave) lo = mid; else hi = mid;
        }
        const int bi = lo;
        const KetList kl(a.klist, a.nbk, bi);
        const int pos = (wave - cpre[bi]) * 64 + lane;
        const bool inrange = pos < kl.n;
        const int ki = kl.ket(inrange ? pos : 0);
        const int sA = cst(a.bra.shA)[bi], sB = cst(a.bra.shB)[bi];
        const int sC = a.ket.shA[ki], sD = a.ket.shB[ki];
        const int kn = inrange ? a.ket.ppn[ki] : 0;
        const bool live = kn > 0;
        if (__ballot(live) == 0) continue;

        const cptr<DevShell> SA = cst(a.sh + sA);
        const cptr<DevShell> SB = cst(a.sh + sB);
        const DevShell* SC = a.sh + sC;
        const DevShell* SD = a.sh + sD;
        double f = live ? 1.0 : 0.0;
        if (sA == sB) f *= 0.5;
        if (sC == sD) f *= 0.5;
        if (a.same && bi == ki) f *= 0.5;
        const cptr<double> ABp = cst(a.bra.AB + 3 * bi);
        const double AB[3] = {ABp[0], ABp[1], ABp[2]};
        const double CD[3] = {a.ket.AB[3 * ki], a.ket.AB[3 * ki + 1], a.ket.AB[3 * ki + 2]};
        double acc[NACC], accb[NACC];
#pragma unroll
        for (int n = 0; n < NACC; ++n) acc[n] = 0.0;
        {
            double G[NINT], x[3], y[3];
            grad_seeds<NA, NB, NC, ND>(a, SA, SB, SC, SD, f, G);
            Adj::hrr_adj(acc, G, accb, x, y, AB[0], AB[1], AB[2], CD[0], CD[1], CD[2]);
        }

        // ---- primitive loop: bra primitive pairs (wave-uniform) outside ----
        const int bo = cst(a.bra.ppo)[bi], bn = cst(a.bra.ppn)[bi];
        const cptr<PrimPair> BP = cst(a.pp + bo);
        const cptr<int> BK = cst(a.ppk + bo);
        const PrimPair* KP = a.pp + a.ket.ppo[ki];
        const int* KK = a.ppk + a.ket.ppo[ki];
        const int pA = cst(a.shell_poff)[sA], pB = cst(a.shell_poff)[sB];
        const int pC = a.shell_poff[sC], pD = a.shell_poff[sD];
        double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0}, gC[3] = {0.0, 0.0, 0.0}, gD[3] = {0.0, 0.0, 0.0};
        for (int u = 0; u < bn; ++u) {
            const double p = BP[u].p, inv2p = BP[u].inv2p, bx = BP[u].pad, Kp = BP[u].Kp;
            const double Px = BP[u].Px, Py = BP[u].Py, Pz = BP[u].Pz;
            const double PA[3] = {BP[u].PAx, BP[u].PAy, BP[u].PAz};
            double sa = 0.0, sbx = 0.0, sl = 0.0;
            for (int v = 0; v < kn; ++v) {
                const KetPrim Q = load_ket(KP + v);
                const double dx = KP[v].pad;
                const int kk = KK[v];
                const double QC[3] = {Q.QCx, Q.QCy, Q.QCz};
                const double PQ[3] = {Px - Q.Qx, Py - Q.Qy, Pz - Q.Qz};
                const double s = rsqrt_pos(p + Q.q), inv = s * s;
                const double T = p * Q.q * inv * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
                const double pref = Kp * Q.Kq * s;
                double Bm[LT + 2];
                boys_lds<LT + 1>(T, Bm, sb);
                double F[LT + 1];
#pragma unroll
                for (int m = 0; m <= LT; ++m) F[m] = Bm[m] * pref;
                const double rho_p = Q.q * inv, rho_q = p * inv;
                double Fb[LT + 1], bin[17];
                const double Lp = Adj::template vrr_adj_grp<GR>(
                    F, accb, acc, PA[0], PA[1], PA[2], -rho_p * PQ[0], -rho_p * PQ[1], -rho_p * PQ[2], QC[0], QC[1],
                    QC[2], rho_q * PQ[0], rho_q * PQ[1], rho_q * PQ[2], inv2p, Q.inv2q, 0.5 * inv, rho_p, rho_q, Fb,
                    bin);
                const GeomAdj g = geom_adjoint<LT>(p - bx, bx, Q.q - dx, dx, 2.0 * inv2p, 2.0 * Q.inv2q, PA, QC, AB,
                                                   CD, PQ, pref, inv, Bm, Fb, bin);
                sa += g.da;
                sbx += g.db;
                sl += Lp;
                const int kc = pC + (kk & 0xffff), kd = pD + (kk >> 16);
                sink.xpn(kc, g.dc);
                sink.xpn(kd, g.dd);
                sink.lin(kc, Lp);
                sink.lin(kd, Lp);
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    gA[t] += g.dA[t];
                    gB[t] += g.dB[t];
                    gC[t] += g.dC[t];
                    gD[t] += g.dD[t];
                }
            }
            sa = wave_sum(sa);
            sbx = wave_sum(sbx);
            sl = wave_sum(sl);
            if (lane == 0) {
                const int kab = BK[u];
                const int ka = pA + (kab & 0xffff), kb = pB + (kab >> 16);
                sink.xpn(ka, sa);
                sink.xpn(kb, sbx);
                sink.lin(ka, sl);
                sink.lin(kb, sl);
            }
        }

        // ---- derivatives with respect to A-B and C-D, and the centres' sums ----
        asm volatile("" ::: "memory");    // the seeds are formed again, not kept
        {
            double G[NINT], x[NACC], bAB[3], bCD[3];
            grad_seeds<NA, NB, NC, ND>(a, SA, SB, SC, SD, f, G);
            Adj::hrr_adj(acc, G, x, bAB, bCD, AB[0], AB[1], AB[2], CD[0], CD[1], CD[2]);
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                gA[t] += bAB[t];
                gB[t] -= bAB[t];
                gC[t] += bCD[t];
                gD[t] -= bCD[t];
            }
        }
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const double x1 = wave_sum(gA[t]), x2 = wave_sum(gB[t]);
            if (lane == 0) {
                sink.cen(3 * sA + t, x1);
                sink.cen(3 * sB + t, x2);
            }
            if (live) {
                sink.cen(3 * sC + t, gC[t]);
                sink.cen(3 * sD + t, gD[t]);
            }
        }
    }
    if (a.grad_lds > 0) {
        __syncthreads();
        for (int i = threadIdx.x; i < a.grad_lds; i += 256) {
            const double v = sums[i];
            if (v == 0.0) continue;
            double* out = i < a.n_radial ? a.g_xpn + i
                          : i < 2 * a.n_radial ? a.g_lin + (i - a.n_radial) : a.g_cen + (i - 2 * a.n_radial);
            atomicAdd(out, v);
        }
    }
}

constexpr int GRAD_LDS_MAX = 48 * 1024;   // LDS copy of the outputs (2 radial + 3 shells doubles)

template <int LA, int LB, int LC, int LD, int G>
void launch_grad_group(const EriArgs& a, unsigned blocks, size_t shm, hipStream_t s)
{
    hipLaunchKernelGGL((eri_grad_kernel<LA, LB, LC, LD, G>), dim3(blocks), dim3(256), shm, s, a);
    QBX_HIP(hipGetLastError());
}

template <int LA, int LB, int LC, int LD, int... Gs>
void launch_grad_groups(std::integer_sequence<int, Gs...>, const EriArgs& a, unsigned blocks, size_t shm,
                        hipStream_t* s, int ns)
{
    (launch_grad_group<LA, LB, LC, LD, Gs>(a, blocks, shm, s[Gs % ns]), ...);
}

template <int LA, int LB, int LC, int LD>
void launch_eri_grad(const EriArgs& a0, hipStream_t* s, int ns)
{
    if (a0.nwave <= 0) return;
    EriArgs a = a0;
    const size_t n = 2 * (size_t)a.n_radial + 3 * (size_t)a.nshell;
    const size_t boys = QBX_BOYSL_ROWS * QBX_BOYSL_STRIDE * sizeof(double) + BOYS_HEAD * sizeof(double);
    // the static rows and the copy stay within the 64 KB a block gets without asking
    const size_t shm = n * sizeof(double);
    a.grad_lds = shm + boys <= 64 * 1024 && shm <= (size_t)GRAD_LDS_MAX ? (int)n : 0;
    // a persistent grid: each block adds its copy to the outputs once
    const int64_t need = ((int64_t)a.nwave + 3) / 4;
    const int64_t cap = a.grad_lds > 0 ? 512 : need;
    launch_grad_groups<LA, LB, LC, LD>(std::make_integer_sequence<int, EriAdj<LA, LB, LC, LD>::NGRP>{}, a,
                                       (unsigned)(need < cap ? need : cap), a.grad_lds > 0 ? shm : 0, s, ns);
}

}  // namespace qbx
