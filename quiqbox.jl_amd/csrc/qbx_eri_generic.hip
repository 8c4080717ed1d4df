// qbx_eri_generic.hip -- two-electron integrals of the shell quartets that
// hold an f or g shell (angular momentum above the generated classes), in
// every mode: J/K digest, dense tensor, Schwarz bounds.
//
// Contracted quartets run the McMurchie-Davidson kernel below (eri_md_kernel).
// Primitive quartets handed in by a caller (qbx_prim_eri) run the Obara-Saika
// recurrences axis by axis for one Cartesian component quartet (Obara & Saika, J.
// Chem. Phys. 84, 3963 (1986)), the Boys auxiliary index carried from axis to
// axis: on each axis the vertical recurrence on electron 1 up to the axis's total
// power, the electron transfer to electron 2, then the horizontal transfers on
// the ket and the bra.  This is the per-component form of the recurrences that
// Quiqbox evaluates (GaussianOrbitals.jl:525-663); here every primitive quartet is
// first put in the orientation where the transfer steps do not amplify rounding:
// within each pair the larger exponent first, and the electron whose pair has the
// smaller exponent sum first (the transfer multiplies by p/q <= 1).
#include "qbx_eri.h"

#include <algorithm>

namespace qbx {
namespace {

constexpr double kTwoPi52 = 34.986836655249725693;   // 2 pi^{5/2}

struct PrimGeom {
    double p, Px, Py, Pz;     // exponent sum, product centre
    double PA[3];             // P - A (first centre of the pair)
    double AB[3];             // A - B
    double ea, eb;            // exponents of the pair's first and second primitive
    double K;                 // c_a c_b exp(-ab/p |A-B|^2) / p
};

// One axis: vals[0..nUp] hold the values carried from the previous axes
// (index = Boys auxiliary order); on return vals[0..nUp-S] hold this axis
// processed, S = a + b + c + d its total power.
template <int NM>
__device__ void axis_pass(double* vals, int& nUp, int a, int b, int c, int d, double xPA, double xPQ, double xAB,
                          double xCD, double fac, double i2p, double iq, double poq, double shiftq)
{
    const int S = a + b + c + d;
    if (S == 0) return;
    double T[NM + 1][NM + 1];
    for (int j = 0; j <= nUp; ++j) T[0][j] = vals[j];
    // vertical recurrence on electron 1:
    // [i+1]^(j) = PA [i]^(j) - (rho/p) PQ [i]^(j+1) + i/(2p) ([i-1]^(j) - (rho/p) [i-1]^(j+1))
    for (int i = 0; i < S; ++i)
        for (int j = 0; j + i < nUp; ++j) {
            double v = xPA * T[i][j] - fac * xPQ * T[i][j + 1];
            if (i > 0) v += (i * i2p) * (T[i - 1][j] - fac * T[i - 1][j + 1]);
            T[i + 1][j] = v;
        }
    const int nOut = nUp - S, cd = c + d;
    const double i2q = 0.5 * iq;
    for (int m = 0; m <= nOut; ++m) {
        // electron transfer: [i, o+1] = (i [i-1, o] + o [i, o-1]) / (2q)
        //                               - (b X_AB + d X_CD) / q [i, o] - p/q [i+1, o]
        double E[NM + 1][NM + 1];
        for (int i = 0; i <= S; ++i) E[i][0] = T[i][m];
        for (int o = 0; o < cd; ++o)
            for (int i = 0; i + o < S; ++i) {
                double t1 = 0.0;
                if (i > 0) t1 += i * E[i - 1][o];
                if (o > 0) t1 += o * E[i][o - 1];
                E[i][o + 1] = t1 * i2q - shiftq * E[i][o] - poq * E[i + 1][o];
            }
        // horizontal transfers: (k, t+1) = (k+1, t) + X (k, t), ket then bra
        double g[NM + 1];
        for (int i = a; i <= a + b; ++i) {
            double h[NM + 1];
            for (int o = c; o <= cd; ++o) h[o] = E[i][o];
            for (int s = 0; s < d; ++s)
                for (int k = c; k < cd - s; ++k) h[k] = h[k + 1] + xCD * h[k];
            g[i] = h[c];
        }
        for (int s = 0; s < b; ++s)
            for (int k = a; k < a + b - s; ++k) g[k] = g[k + 1] + xAB * g[k];
        vals[m] = g[a];
    }
    nUp = nOut;
}

__device__ inline void flip_pair(PrimGeom& g, int* la, int* lb)
{
    for (int t = 0; t < 3; ++t) {
        g.PA[t] += g.AB[t];       // P - B = (P - A) + (A - B)
        g.AB[t] = -g.AB[t];
        const int x = la[t];
        la[t] = lb[t];
        lb[t] = x;
    }
    const double e = g.ea;
    g.ea = g.eb;
    g.eb = e;
}

// One primitive quartet of one Cartesian component quartet, weights included.
template <int NM>
__device__ double prim_quartet(PrimGeom X, PrimGeom Y, int la[3], int lb[3], int lc[3], int ld[3],
                               const double* boys, const double* bexp)
{
    if (X.eb > X.ea) flip_pair(X, la, lb);
    if (Y.eb > Y.ea) flip_pair(Y, lc, ld);
    int* a = la;
    int* b = lb;
    int* c = lc;
    int* d = ld;
    if (X.p > Y.p) {
        const PrimGeom t = X;
        X = Y;
        Y = t;
        a = lc;
        b = ld;
        c = la;
        d = lb;
    }
    const double p = X.p, q = Y.p, pq = p + q;
    const double PQ[3] = {X.Px - Y.Px, X.Py - Y.Py, X.Pz - Y.Pz};
    const double rho = p * q / pq;
    const double T = rho * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
    const int Lt = a[0] + a[1] + a[2] + b[0] + b[1] + b[2] + c[0] + c[1] + c[2] + d[0] + d[1] + d[2];
    double vals[NM + 1];
    qbx_boys_rt(Lt, T, vals, boys, bexp);
    const double fac = q / pq, i2p = 0.5 / p, iq = 1.0 / q, poq = p / q;
    int nUp = Lt;
    for (int t = 0; t < 3; ++t) {
        const double shiftq = (X.eb * X.AB[t] + Y.eb * Y.AB[t]) * iq;
        axis_pass<NM>(vals, nUp, a[t], b[t], c[t], d[t], X.PA[t], PQ[t], X.AB[t], Y.AB[t], fac, i2p, iq, poq,
                      shiftq);
    }
    return kTwoPi52 * X.K * Y.K / sqrt(pq) * vals[0];
}

// ---------------------------------------------------------------------------
// Contracted shell quartets: McMurchie-Davidson (J. Comput. Phys. 26, 218
// (1978)).  A block takes one shell quartet, W teams of TS threads: each team takes a
// share of the ket's primitive pairs with its own LDS for what follows.  Four teams
// of one wave where kets are contracted (a single wave's chain through the 512
// primitive quartets of an f and three core s shells took 0.6 ms); one team of four
// waves for few primitive quartets of high angular momentum (one wave on (ff|ff):
// 0.9 ms), one of one wave otherwise.  For each primitive quartet the Hermite
// integrals
//   R_tuv^(m): R_000^(m) = (-2 alpha)^m F_m,  R_{t+1,u,v}^(m) = t R_{t-1,u,v}^(m+1)
//                                                            + X R_tuv^(m+1)
// are built in LDS, lanes over (t, u, v), one level of m after another; the ket's
// Hermite coefficients of every ket component are applied to them and summed over
// the ket's primitive pairs,
//   T[h][cd] = sum_kets sum_k E^cd_k (-1)^k R_{h+k},  h = (t, u, v) of the bra,
// and the bra's coefficients are applied once per bra primitive pair,
//   (ab|cd) = sum_bras sum_h E^ab_h T[h][cd].
// No step is repeated per component quartet: one recurrence per component quartet
// and primitive quartet, with its tables in scratch memory, took 52 ms for the 7,449
// such shell quartets (126,000 primitive quartets) of N2 in cc-pVTZ; the launches of
// this kernel sum to 7 ms there, on three streams.  Bound by LDS
// latency along the chain of the R levels (as many blocks per CU as the class's LDS
// allows).  Exchanges within a wave need no barrier: a wave's LDS instructions
// complete in order (team_sync then only keeps the compiler from reordering them).
//
// LDS (doubles), sized per pair of pair classes: per team R as a cube of side L + 1,
// the scaled Boys values and P - Q of 64 primitive quartets (one per lane,
// evaluated together), the E table [axis][i][j][t] of the current ket pair (its odd
// t negated) and T for `ub` bra primitive pairs and `cdc` ket components; per block
// the bra pairs' E tables, the sums of those components, and per ket component the
// places and sizes of its E rows.
// ---------------------------------------------------------------------------
constexpr int MD_LMAX = 4 * QBX_MAXL;
constexpr int md_nherm(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }

// (t, u, v) of Hermite index h, ordered by t + u + v, then as Cartesian components
__host__ __device__ constexpr int md_index(int t, int u, int v)
{
    const int N = t + u + v, r = N - t;
    return N * (N + 1) * (N + 2) / 6 + r * (r + 1) / 2 + v;
}

struct HermTable {
    unsigned short tuv[md_nherm(MD_LMAX)];   // t | u << 5 | v << 10
    constexpr HermTable() : tuv()
    {
        for (int t = 0; t <= MD_LMAX; ++t)
            for (int u = 0; t + u <= MD_LMAX; ++u)
                for (int v = 0; t + u + v <= MD_LMAX; ++v)
                    tuv[md_index(t, u, v)] = (unsigned short)(t | u << 5 | v << 10);
    }
};
__device__ const HermTable d_herm{};

template <int TS> __device__ __forceinline__ void team_sync()
{
    if constexpr (TS > 64) {
        __syncthreads();    // the team is the block
    } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

struct MdSizes {
    int S, eb, ek, nhab, nab, ncd;
    __host__ __device__ MdSizes(int la, int lb, int lc, int ld)
    {
        S = la + lb + lc + ld + 1;
        eb = 3 * (la + 1) * (lb + 1) * (la + lb + 1);
        ek = 3 * (lc + 1) * (ld + 1) * (lc + ld + 1);
        nhab = md_nherm(la + lb);
        nab = qbx_ncart(la) * qbx_ncart(lb);
        ncd = qbx_ncart(lc) * qbx_ncart(ld);
    }
    __host__ __device__ size_t wave(int ub, int cdc) const
    {
        return (size_t)S * S * S + 64 * (S + 3) + ek + (size_t)cdc * ub * nhab;
    }
    __host__ __device__ size_t doubles(int ub, int cdc, int waves) const
    {
        return waves * wave(ub, cdc) + (size_t)ub * eb + (size_t)cdc * (nab + 1);
    }
};

// Hermite coefficients E_t^{ij} (without the pair's exponential) of n primitive
// pairs into [pair][axis][i][j][t], threads of one team over (pair, axis, t), team
// `first` of `step`; NEG: times (-1)^t.
//   E_t^{i+1,j} = E_{t-1}^{ij} / 2p + X_PA E_t^{ij} + (t+1) E_{t+1}^{ij}, j with X_PB
template <bool NEG, int TS>
__device__ void md_coefficients(double* E, const PrimPair* P, int n, int la, int lb, const double* AB, int lane,
                                int first, int step)
{
    const int nt = la + lb + 1, per = 3 * nt, size = 3 * (la + 1) * (lb + 1) * nt;
    const int group = TS / per;   // pairs evaluated together (per <= 27)
    for (int p0 = first * group; p0 < n; p0 += step * group) {
        const int w = lane / per, r = lane - w * per, ax = r / nt, t = r - ax * nt;
        const bool on = w < group && p0 + w < n;
        double* e = E + (size_t)(on ? p0 + w : 0) * size + (size_t)(on ? ax : 0) * (la + 1) * (lb + 1) * nt;
        const PrimPair* q = P + (on ? p0 + w : 0);
        const double s = NEG ? -1.0 : 1.0;
        const double h = s * q->inv2p, up = s * (t + 1);
        const double xa = ax == 0 ? q->PAx : ax == 1 ? q->PAy : q->PAz;
        const double xb = xa + AB[ax < 3 ? ax : 0];
        if (on) e[t] = t == 0 ? 1.0 : 0.0;
        team_sync<TS>();
        for (int i = 0; i <= la; ++i) {
            if (i > 0) {
                const double* f = e + (size_t)(i - 1) * (lb + 1) * nt;
                if (on)
                    e[(size_t)i * (lb + 1) * nt + t] =
                        (t > 0 ? h * f[t - 1] : 0.0) + xa * f[t] + (t + 1 < nt ? up * f[t + 1] : 0.0);
                team_sync<TS>();
            }
            for (int j = 1; j <= lb; ++j) {
                const double* f = e + ((size_t)i * (lb + 1) + j - 1) * nt;
                if (on)
                    e[((size_t)i * (lb + 1) + j) * nt + t] =
                        (t > 0 ? h * f[t - 1] : 0.0) + xb * f[t] + (t + 1 < nt ? up * f[t + 1] : 0.0);
                team_sync<TS>();
            }
        }
    }
}

// F_0..F_n into LDS (qbx_boys_rt with the running order in a register)
__device__ void md_boys(int n, double T, double* F, const double* __restrict__ tab, const double* __restrict__ etab)
{
    if (T < QBX_BOYS_TMAX) {
        const int i = __double2int_rn(T * QBX_BOYS_INVDT);
        const double md = (double)i * QBX_BOYS_DT - T;
        const double* __restrict__ row = tab + i * QBX_BOYS_NCOL + n;
        double acc = row[QBX_BOYS_TAYLOR - 1];
#pragma unroll
        for (int k = QBX_BOYS_TAYLOR - 1; k >= 1; --k) acc = row[k - 1] + (md * (1.0 / k)) * acc;
        double ex = 1.0;
#pragma unroll
        for (int k = 8; k >= 1; --k) ex = 1.0 + (md * (1.0 / k)) * ex;
        const double e = etab[i] * ex;
        F[n] = acc;
        for (int m = n - 1; m >= 0; --m) {
            acc = (2.0 * T * acc + e) / (2 * m + 1);
            F[m] = acc;
        }
    } else {
        const double rt = rsqrt(T);
        const double h = 0.5 * rt * rt;
        double acc = 0.88622692545275801365 * rt;
        F[0] = acc;
        for (int m = 0; m < n; ++m) {
            acc *= (2 * m + 1) * h;
            F[m + 1] = acc;
        }
    }
}

template <int NSLOT, int MODE, int TS, int W>
__global__ __launch_bounds__(TS * W) void eri_md_kernel(GenArgs a)
{
    extern __shared__ double lds[];
    const int tid = (int)threadIdx.x, lane = tid % TS;      // thread of the team
    const int w = __builtin_amdgcn_readfirstlane(tid / TS); // team
    const int la = a.l[0], lb = a.l[1], lc = a.l[2], ld = a.l[3];
    const int L = la + lb + lc + ld;
    const MdSizes z(la, lb, lc, ld);
    const int S = z.S, S2 = S * S, ub = a.ub, cdc = a.cdc, nh = z.nhab;
    const size_t per = z.wave(ub, cdc);
    double* R = lds + w * per;
    double* Fs = R + S * S2;                 // [64][S]
    double* PQ = Fs + 64 * S;                // [64][3]
    double* Ek = PQ + 64 * 3;
    double* T = Ek + z.ek;                   // [ub][cdc][nh]
    double* Eb = lds + W * per;              // [ub][eb]
    double* out = Eb + (size_t)ub * z.eb;    // [cdc][nab]
    int2* info = (int2*)(out + (size_t)cdc * z.nab);   // per ket component

    // the thread's Hermite indices: place in the cube, the axis stepped down and its power
    int place[NSLOT], step[NSLOT], pw[NSLOT], level[NSLOT], axis[NSLOT];
#pragma unroll
    for (int s = 0; s < NSLOT; ++s) {
        const int h = lane + TS * s;
        const int c = h < md_nherm(L) ? d_herm.tuv[h] : 0;
        const int t = c & 31, u = (c >> 5) & 31, v = c >> 10;
        place[s] = t * S2 + u * S + v;
        axis[s] = t ? 0 : u ? 1 : 2;
        step[s] = t ? S2 : u ? S : 1;
        pw[s] = t ? t : u ? u : v;
        level[s] = h < md_nherm(L) && h > 0 ? t + u + v : 1 << 20;
    }

    // shell quartet of this block
    const int64_t task = a.first + (int64_t)blockIdx.x;
    int lo = 0, hi = a.nbra;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (a.prefix[mid] <= task) lo = mid; else hi = mid;
    }
    const int bi = lo;
    const int ki = MODE == MODE_SCHWARZ ? bi : (int)(task - a.prefix[bi]);
    const int sA = a.bra.shA[bi], sB = a.bra.shB[bi], sC = a.ket.shA[ki], sD = a.ket.shB[ki];
    const int bn = a.bra.ppn[bi], kn = a.ket.ppn[ki];
    if (bn == 0 || kn == 0) return;
    if (MODE == MODE_JK && a.pdmax) {
        const int ns = a.nshell;
        const double* dm = a.pdmax;
        double dmax = fmax(fmax(dm[sA * ns + sB], dm[sC * ns + sD]), fmax(dm[sA * ns + sC], dm[sA * ns + sD]));
        dmax = fmax(dmax, fmax(dm[sB * ns + sC], dm[sB * ns + sD]));
        if (a.bra.Q[bi] * a.ket.Q[ki] * dmax < a.dthr) return;
    }
    const PrimPair* BP = a.pp + a.bra.ppo[bi];
    const PrimPair* KP = a.pp + a.ket.ppo[ki];
    const double AB[3] = {a.bra.AB[3 * bi], a.bra.AB[3 * bi + 1], a.bra.AB[3 * bi + 2]};
    const double CD[3] = {a.ket.AB[3 * ki], a.ket.AB[3 * ki + 1], a.ket.AB[3 * ki + 2]};
    const DevShell* SA = a.sh + sA;
    const DevShell* SB = a.sh + sB;
    const DevShell* SC = a.sh + sC;
    const DevShell* SD = a.sh + sD;
    const int NB = qbx_ncart(lb), ND = qbx_ncart(ld);
    const int ntb = la + lb + 1, ntk = lc + ld + 1;
    double f = 1.0;
    if (sA == sB) f *= 0.5;
    if (sC == sD) f *= 0.5;
    if (a.same && bi == ki) f *= 0.5;
    const size_t N = (size_t)a.N;
    const JKSink sink(a);
    double qmax = 0.0;

    for (int c0 = 0; c0 < z.ncd; c0 += cdc) {
        const int nc = min(cdc, z.ncd - c0);
        __syncthreads();    // the previous components' sums and rows are read
        for (int c = tid; c < nc; c += TS * W) {
            const int ic = (c0 + c) / ND, id = (c0 + c) - ic * ND;
            int gc[3], gd[3];
            qbx_cart(lc, ic, gc);
            qbx_cart(ld, id, gd);
            int2 v;
            // rows of Ek (each below 1024) and their lengths (each below 16)
            v.x = 0;
            v.y = 0;
            for (int x = 0; x < 3; ++x) {
                v.x |= (((x * (lc + 1) + gc[x]) * (ld + 1) + gd[x]) * ntk) << (10 * x);
                v.y |= (gc[x] + gd[x] + 1) << (8 * x);
            }
            info[c] = v;
        }
        for (int k = tid; k < nc * z.nab; k += TS * W) out[k] = 0.0;
        const int v0 = kn * w / W, vn = kn * (w + 1) / W - v0;   // this team's ket primitive pairs
        for (int u0 = 0; u0 < bn; u0 += ub) {
            const int nu = min(ub, bn - u0);
            __syncthreads();
            md_coefficients<false, TS>(Eb, BP + u0, nu, la, lb, AB, lane, w, W);
            for (int k = lane; k < nu * nc * nh; k += TS) T[k] = 0.0;
            const int total = vn * nu;
            int vcur = -1;
            for (int j0 = 0; j0 < total; j0 += 64) {
                team_sync<TS>();    // the previous batch's values are read
                if (lane < 64 && j0 + lane < total) {
                    const int v = (j0 + lane) / nu, u = (j0 + lane) - v * nu;
                    const PrimPair& X = BP[u0 + u];
                    const PrimPair& Y = KP[v0 + v];
                    const double p = X.p, q = Y.p, is = rsqrt(p + q), alpha = p * q * is * is;
                    const double x = X.Px - Y.Px, y = X.Py - Y.Py, zz = X.Pz - Y.Pz;
                    double* F = Fs + lane * S;
                    md_boys(L, alpha * (x * x + y * y + zz * zz), F, a.boys, a.bexp);
                    double pref = kTwoPi52 * X.Kp * Y.Kp * is;
                    for (int m = 0; m <= L; ++m) {
                        F[m] *= pref;
                        pref *= -2.0 * alpha;
                    }
                    PQ[3 * lane] = x;
                    PQ[3 * lane + 1] = y;
                    PQ[3 * lane + 2] = zz;
                }
                team_sync<TS>();
                const int jn = min(64, total - j0);
                for (int j = 0; j < jn; ++j) {
                    const int v = (j0 + j) / nu, u = (j0 + j) - v * nu;
                    if (v != vcur) {
                        md_coefficients<true, TS>(Ek, KP + v0 + v, 1, lc, ld, CD, lane, 0, 1);
                        vcur = v;
                    }
                    // Hermite integrals: level m from level m + 1 in place (every lane reads before any writes)
                    double xs[NSLOT];
#pragma unroll
                    for (int s = 0; s < NSLOT; ++s) xs[s] = PQ[3 * j + axis[s]];
                    if (lane == 0) R[0] = Fs[j * S + L];
                    for (int m = L - 1; m >= 0; --m) {
                        team_sync<TS>();
                        double nv[NSLOT];
#pragma unroll
                        for (int s = 0; s < NSLOT; ++s)
                            if (level[s] <= L - m) {
                                nv[s] = xs[s] * R[place[s] - step[s]];
                                if (pw[s] > 1) nv[s] += (pw[s] - 1) * R[place[s] - 2 * step[s]];
                            }
                        team_sync<TS>();
#pragma unroll
                        for (int s = 0; s < NSLOT; ++s)
                            if (level[s] <= L - m) R[place[s]] = nv[s];
                        if (lane == 0) R[0] = Fs[j * S + m];
                    }
                    team_sync<TS>();
                    // ket coefficients: T[u][c][h] += sum_k Ek_k R[h + k]
                    double* Tu = T + (size_t)u * nc * nh;
                    int c = lane / nh, h = lane - c * nh;
                    const int dc = TS / nh, dh = TS - dc * nh;
                    for (; c < nc;) {
                        const int hh = d_herm.tuv[h];
                        const double* r = R + (hh & 31) * S2 + ((hh >> 5) & 31) * S + (hh >> 10);
                        const int2 o = info[c];
                        const double* ex = Ek + (o.x & 1023);
                        const double* ey = Ek + ((o.x >> 10) & 1023);
                        const double* ez = Ek + (o.x >> 20);
                        const int nx = o.y & 255, ny = (o.y >> 8) & 255, nz = o.y >> 16;
                        double sum = 0.0;
                        for (int t = 0; t < nx; ++t) {
                            double sy = 0.0;
                            for (int q = 0; q < ny; ++q) {
                                const double* rr = r + t * S2 + q * S;
                                double sz = ez[0] * rr[0];
                                for (int k = 1; k < nz; ++k) sz += ez[k] * rr[k];
                                sy += ey[q] * sz;
                            }
                            sum += ex[t] * sy;
                        }
                        Tu[c * nh + h] += sum;
                        c += dc;
                        h += dh;
                        if (h >= nh) {
                            h -= nh;
                            ++c;
                        }
                    }
                    team_sync<TS>();    // R and Ek are rewritten by the next primitive quartet
                }
            }
            // bra coefficients, on the teams' T together
            __syncthreads();
            for (int k = tid; k < nc * z.nab; k += TS * W) {
                const int c = k / z.nab, ab = k - c * z.nab;
                const int ia = ab / NB, ib = ab - ia * NB;
                int ga[3], gb[3];
                qbx_cart(la, ia, ga);
                qbx_cart(lb, ib, gb);
                double sum = 0.0;
                for (int u = 0; u < nu; ++u) {
                    const double* e = Eb + (size_t)u * z.eb;
                    const double* t0 = lds + (T - R) + ((size_t)u * nc + c) * nh;   // team 0's
                    const double* ex = e + ((0 * (la + 1) + ga[0]) * (lb + 1) + gb[0]) * ntb;
                    const double* ey = e + ((1 * (la + 1) + ga[1]) * (lb + 1) + gb[1]) * ntb;
                    const double* ez = e + ((2 * (la + 1) + ga[2]) * (lb + 1) + gb[2]) * ntb;
                    for (int t = 0; t <= ga[0] + gb[0]; ++t)
                        for (int q = 0; q <= ga[1] + gb[1]; ++q) {
                            const double exy = ex[t] * ey[q];
                            for (int r = 0; r <= ga[2] + gb[2]; ++r) {
                                const double* th = t0 + md_index(t, q, r);
                                double v = th[0];
#pragma unroll
                                for (int o = 1; o < W; ++o) v += th[o * per];
                                sum += exy * ez[r] * v;
                            }
                        }
                }
                out[k] += sum;
            }
        }
        // ---- digest of these ket components: element k is written and read by one thread ----
        for (int k = tid; k < nc * z.nab; k += TS * W) {
            const int c = k / z.nab, ab = k - c * z.nab;
            const int ia = ab / NB, ib = ab - ia * NB;
            const int ic = (c0 + c) / ND, id = (c0 + c) - ic * ND;
            const int fa = SA->bf[ia], fb = SB->bf[ib], fc = SC->bf[ic], fd = SD->bf[id];
            if (fa < 0 || fb < 0 || fc < 0 || fd < 0) continue;
            const double val = out[k] * (SA->sc[ia] * SB->sc[ib]) * (SC->sc[ic] * SD->sc[id]);
            if (MODE == MODE_SCHWARZ) {
                if (ab == c0 + c) qmax = fmax(qmax, fabs(val));
            } else if (MODE == MODE_DENSE) {
                // an element that several components reach (A = B, C = D, bra = ket) is written by one
                if ((sA == sB && ia < ib) || (sC == sD && ic < id) || (a.same && bi == ki && ab < c0 + c))
                    continue;
                const size_t i = fa, j = fb, kk = fc, l = fd;
                a.eri[((i * N + j) * N + kk) * N + l] = val;
                a.eri[((j * N + i) * N + kk) * N + l] = val;
                a.eri[((i * N + j) * N + l) * N + kk] = val;
                a.eri[((j * N + i) * N + l) * N + kk] = val;
                a.eri[((kk * N + l) * N + i) * N + j] = val;
                a.eri[((l * N + kk) * N + i) * N + j] = val;
                a.eri[((kk * N + l) * N + j) * N + i] = val;
                a.eri[((l * N + kk) * N + j) * N + i] = val;
            } else {
                // J_ab += 4f v D_cd, J_cd += 4f v D_ab, K_ac/K_ad/K_bd/K_bc += 2f v D
                // (the symmetrization G = (J + J^T)/2 - (K + K^T)/2 completes the 8-fold sum)
                const double fj = 4.0 * f * val, fk = 2.0 * f * val;
                for (int s = 0; s < a.nset; ++s) {
                    const double* DJ = a.D + (size_t)s * N * N;
                    const double* DK = a.D + (size_t)(a.nset + s) * N * N;
                    double* Js = sink.J + (size_t)s * N * N;
                    double* Ks = sink.K + (size_t)s * N * N;
                    sink.add(Js + fa * N + fb, fj * DJ[fc * N + fd]);
                    sink.add(Js + fc * N + fd, fj * DJ[fa * N + fb]);
                    sink.add(Ks + fa * N + fc, fk * DK[fb * N + fd]);
                    sink.add(Ks + fa * N + fd, fk * DK[fb * N + fc]);
                    sink.add(Ks + fb * N + fd, fk * DK[fa * N + fc]);
                    sink.add(Ks + fb * N + fc, fk * DK[fa * N + fd]);
                }
            }
        }
    }
    if (MODE == MODE_SCHWARZ) {
        for (int o = 32; o > 0; o >>= 1) qmax = fmax(qmax, __shfl_xor(qmax, o, 64));
        __syncthreads();
        if ((tid & 63) == 0) lds[tid >> 6] = qmax;
        __syncthreads();
        for (int o = 0; o < TS * W / 64; ++o) qmax = fmax(qmax, lds[o]);
        if (tid == 0) a.qout[bi] = sqrt(qmax);
    }
}

// One block a quartet; a grid holds below 2^32 threads (16.8 million blocks of 256), so
// longer lists take several launches.
template <int NSLOT, int TS, int W> void launch_slots(GenArgs a, size_t shm, int mode, hipStream_t s)
{
    constexpr int64_t MAX_BLOCKS = 0xffffffffLL / (TS * W);
    auto go = [&](void (*kern)(GenArgs)) {
        // above 64 KB the limit has to be raised
        if (shm > 64 * 1024)
            QBX_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
        for (a.first = 0; a.first < a.total; a.first += MAX_BLOCKS) {
            const int64_t n = std::min(a.total - a.first, MAX_BLOCKS);
            hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(TS * W), shm, s, a);
            QBX_HIP(hipGetLastError());
        }
    };
    switch (mode) {
    case MODE_JK: go(eri_md_kernel<NSLOT, MODE_JK, TS, W>); break;
    case MODE_DENSE: go(eri_md_kernel<NSLOT, MODE_DENSE, TS, W>); break;
    case MODE_SCHWARZ: go(eri_md_kernel<NSLOT, MODE_SCHWARZ, TS, W>); break;
    default: throw QbxError(QBX_EINTERNAL, "unknown ERI mode");
    }
}

// Primitive quartets one thread each (unit coefficients): the reference's
// per-primitive engine computePGTOrbTwoBodyRepulsion! (GaussianOrbitals.jl:594-663).
__global__ __launch_bounds__(64) void prim_eri_kernel(int n, const double* __restrict__ cen,
                                                      const double* __restrict__ xpn, const int* __restrict__ ang,
                                                      const double* boys, const double* bexp, double* __restrict__ out)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= n) return;
    int l[4][3];
    double c[4][3], e[4];
    for (int k = 0; k < 4; ++k) {
        e[k] = xpn[4 * i + k];
        for (int t = 0; t < 3; ++t) {
            c[k][t] = cen[12 * i + 3 * k + t];
            l[k][t] = ang[12 * i + 3 * k + t];
        }
    }
    PrimGeom G[2];
    for (int h = 0; h < 2; ++h) {
        const int ka = 2 * h, kb = 2 * h + 1;
        PrimGeom& g = G[h];
        g.ea = e[ka];
        g.eb = e[kb];
        g.p = e[ka] + e[kb];
        double r2 = 0.0, P[3];
        for (int t = 0; t < 3; ++t) {
            g.AB[t] = c[ka][t] - c[kb][t];
            r2 += g.AB[t] * g.AB[t];
            P[t] = (e[ka] * c[ka][t] + e[kb] * c[kb][t]) / g.p;
            g.PA[t] = P[t] - c[ka][t];
        }
        g.Px = P[0];
        g.Py = P[1];
        g.Pz = P[2];
        g.K = exp(-e[ka] * e[kb] / g.p * r2) / g.p;
    }
    out[i] = prim_quartet<QBX_PRIM_ERI_LTOT>(G[0], G[1], l[0], l[1], l[2], l[3], boys, bexp);
}

}  // namespace

void prim_eri(int n, const double* cen, const double* xpn, const int* ang, const double* boys, const double* bexp,
              double* out, hipStream_t s)
{
    static_assert(QBX_PRIM_ERI_LTOT <= QBX_BOYS_NMAX, "Boys table orders for the primitive ERIs");
    if (n <= 0) return;
    hipLaunchKernelGGL(prim_eri_kernel, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, n, cen, xpn, ang, boys, bexp,
                       out);
    QBX_HIP(hipGetLastError());
}

// LDS a block may take: four (one wave) or two blocks a CU, all of it where the
// integrals of two g pairs need it
constexpr size_t kMdLds = 40 * 1024, kMdLds4 = 80 * 1024, kMdLdsMax = 128 * 1024;

void launch_eri_generic(const GenArgs& a0, int mode, hipStream_t s)
{
    static_assert(MD_LMAX <= 16 && MD_LMAX <= QBX_BOYS_NMAX, "generic kernel sizes");
    if (a0.total <= 0) return;
    GenArgs a = a0;
    const int L = a.l[0] + a.l[1] + a.l[2] + a.l[3];
    if (L > MD_LMAX) throw QbxError(QBX_EUNSUP, "angular momentum above the generic kernel");
    const MdSizes z(a.l[0], a.l[1], a.l[2], a.l[3]);
    if (z.ek > 1024) throw QbxError(QBX_EINTERNAL, "Hermite rows of a ket pair above their encoding");
    const int ub = std::max(1, std::min(a.bn_max, 8));
    // four teams where some ket has as many primitive pairs for them and their LDS
    // fits; else one team, of four waves from 84 Hermite integrals (L = 6) on
    const bool teams = a.kn_max >= 4 && z.doubles(ub, std::min(z.ncd, 3), 4) * sizeof(double) <= kMdLds4;
    const bool wide = !teams && L >= 6;
    const int W = teams ? 4 : 1;
    const size_t usual = teams || wide ? kMdLds4 : kMdLds;
    // bra primitive pairs and ket components held at a time: up to eight pairs, then
    // as many components as fit
    a.ub = ub;
    while (a.ub > 1 && z.doubles(a.ub, 1, W) * sizeof(double) > usual) --a.ub;
    a.cdc = 1;
    while (a.cdc < z.ncd && z.doubles(a.ub, a.cdc + 1, W) * sizeof(double) <= usual) ++a.cdc;
    // the team's part alone is near the usual size: a few components beyond it
    while (a.cdc < z.ncd && a.cdc < 8 && z.doubles(a.ub, a.cdc + 1, W) * sizeof(double) <= kMdLdsMax) ++a.cdc;
    // equal shares of the components
    const int parts = (z.ncd + a.cdc - 1) / a.cdc;
    a.cdc = (z.ncd + parts - 1) / parts;
    const size_t shm = z.doubles(a.ub, a.cdc, W) * sizeof(double);
    if (shm > kMdLdsMax) throw QbxError(QBX_EINTERNAL, "generic ERI kernel beyond its LDS");
    const int slots = (md_nherm(L) + (wide ? 255 : 63)) / (wide ? 256 : 64);
    if (wide) {
        if (slots <= 1) launch_slots<1, 256, 1>(a, shm, mode, s);
        else if (slots <= 2) launch_slots<2, 256, 1>(a, shm, mode, s);
        else launch_slots<4, 256, 1>(a, shm, mode, s);
    } else if (!teams) {
        launch_slots<1, 64, 1>(a, shm, mode, s);    // up to L = 5, 56 integrals
    } else {
        if (slots <= 1) launch_slots<1, 64, 4>(a, shm, mode, s);
        else if (slots <= 2) launch_slots<2, 64, 4>(a, shm, mode, s);
        else if (slots <= 4) launch_slots<4, 64, 4>(a, shm, mode, s);
        else if (slots <= 8) launch_slots<8, 64, 4>(a, shm, mode, s);
        else launch_slots<16, 64, 4>(a, shm, mode, s);
    }
}

}  // namespace qbx
