// qbx_one_e.hip -- nuclear attraction of every pair class up to (g, g) and the
// one-electron part of the energy gradient of the s and p pair classes.
//
// Both are sums over (primitive pair, nucleus) of values that depend on the
// pair of shells only through a few linear steps, so a wave takes one shell
// pair and its lanes the (primitive pair, nucleus) items: per item the Boys
// values of the class's order from the rows staged in LDS and the one-body
// vertical recurrence to [e] on the first centre, summed in registers; the
// lanes' sums are then added and the horizontal transfer to (a b) runs once
// per shell pair.
#include "qbx_eri.h"
#include "qbx_one_e.h"
#include "gen/one_e_classes.inc"

namespace qbx {
namespace {

constexpr int kWaves = 4;              // waves (shell pairs) per block
constexpr double kTwoPi = 6.28318530717958647693;
constexpr double kPi32 = 5.568327996831707845;   // pi^(3/2)

// Lane's walk over the items (u, n), u < np primitive pairs, n < nn nuclei, in
// steps of 64 items.
struct ItemWalk {
    int u, n, du, dn, nn;
    __device__ __forceinline__ ItemWalk(int lane, int nnuc) : nn(nnuc)
    {
        u = lane / nnuc;
        n = lane - u * nnuc;
        du = 64 / nnuc;
        dn = 64 - du * nnuc;
    }
    __device__ __forceinline__ void next()
    {
        u += du;
        n += dn;
        if (n >= nn) {
            n -= nn;
            ++u;
        }
    }
};

// Nuclear attraction.  Bound by FP64 issue: per item 16 + 11 L_total Boys and
// geometry operations plus the recurrence.  With one thread per Cartesian
// component pair (every component repeating the Boys values and a recurrence
// in scratch memory) the 592-function, 160-nucleus cluster took 37.0 ms a call;
// it takes 0.50 ms, the copy to the host included.
template <int LA, int LB>
__global__ __launch_bounds__(64 * kWaves) void nuclear_kernel(NucArgs a)
{
    using Cls = OneE<LA, LB>;
    constexpr int L = LA + LB, NA = qbx_ncart(LA), NB = qbx_ncart(LB), NAB = NA * NB;
    constexpr int TPB = 64 * kWaves;
    __shared__ double2 sboys[BOYS_HEAD2 + boys_rows(L) * QBX_BOYSL_STRIDE / 2];
    stage_boys<TPB, boys_rows(L)>(sboys, a.boysl);
    __syncthreads();
    const double* sb = (const double*)sboys + BOYS_HEAD;
    const int lane = (int)threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    for (int pair = (int)blockIdx.x * kWaves + wib; pair < a.pairs.n; pair += (int)gridDim.x * kWaves) {
        const int np = cst(a.pairs.ppn)[pair];
        const PrimPair* P = a.pp + cst(a.pairs.ppo)[pair];
        double acc[Cls::NACC];
#pragma unroll
        for (int k = 0; k < Cls::NACC; ++k) acc[k] = 0.0;
        for (ItemWalk it(lane, a.nnuc); it.u < np; it.next()) {
            const PrimPair* Q = P + it.u;
            const double* R = a.R + 3 * it.n;
            const double p = Q->p;
            const double PCx = Q->Px - R[0], PCy = Q->Py - R[1], PCz = Q->Pz - R[2];
            double F[L + 1];
            boys_lds<L>(p * (PCx * PCx + PCy * PCy + PCz * PCz), F, sb);
            const double pref = -kTwoPi * Q->Kp * a.Z[it.n];
#pragma unroll
            for (int m = 0; m <= L; ++m) F[m] *= pref;
            Cls::vrr(F, acc, Q->PAx, Q->PAy, Q->PAz, PCx, PCy, PCz, Q->inv2p);
        }
#pragma unroll
        for (int k = 0; k < Cls::NACC; ++k) acc[k] = wave_sum(acc[k]);
        const double* AB = a.pairs.AB + 3 * pair;
        double out[NAB];
        Cls::hrr(acc, out, AB[0], AB[1], AB[2]);
        // component pair k to lane k % 64
        const DevShell* SA = a.sh + cst(a.pairs.shA)[pair];
        const DevShell* SB = a.sh + cst(a.pairs.shB)[pair];
#pragma unroll
        for (int k0 = 0; k0 < NAB; k0 += 64) {
            double v = 0.0;
#pragma unroll
            for (int k = k0; k < (k0 + 64 < NAB ? k0 + 64 : NAB); ++k) v = (k - k0) == lane ? out[k] : v;
            const int k = k0 + lane;
            if (k >= NAB) continue;
            const int ia = k / NB, ib = k - ia * NB;
            const int fa = SA->bf[ia], fb = SB->bf[ib];
            if (fa < 0 || fb < 0) continue;
            v *= SA->sc[ia] * SB->sc[ib];
            a.out[(size_t)fa * a.N + fb] = v;
            a.out[(size_t)fb * a.N + fa] = v;
        }
    }
}

// One-electron energy gradient: a lane takes one primitive pair and, where the
// pair has fewer than 64 of them, a share of the nuclei.  The attraction enters
// through [e], |e| <= la + lb + 2, summed over the nuclei first; every raised
// and lowered integral is then a combination of those sums (OneGrad), formed
// once per lane.  The 32-atom s/p cluster (2080 shell pairs, 16 primitive pairs
// each) took 32 ms with one thread per primitive pair that evaluated each raised
// component pair for each nucleus; now below 0.2 ms (the gradient call 70.2 -> 38.7
// ms).
template <int LA, int LB>
__global__ __launch_bounds__(64 * kWaves) void one_e_grad_kernel(NucArgs a)
{
    using Cls = OneGrad<LA, LB>;
    constexpr int L = LA + LB + 2, NA = qbx_ncart(LA), NB = qbx_ncart(LB);
    constexpr int TPB = 64 * kWaves;
    constexpr int MP = QBX_GRAD_MAXP;
    __shared__ double2 sboys[BOYS_HEAD2 + boys_rows(L) * QBX_BOYSL_STRIDE / 2];
    __shared__ double sums[kWaves][4][MP];   // dE/da, dE/db and c dE/dc of A's and B's radial primitives
    stage_boys<TPB, boys_rows(L)>(sboys, a.boysl);
    __syncthreads();
    const double* sb = (const double*)sboys + BOYS_HEAD;
    const int lane = (int)threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int npass = (a.pairs.n + (int)gridDim.x * kWaves - 1) / ((int)gridDim.x * kWaves);
    for (int pass = 0; pass < npass; ++pass) {
        const int pair = (pass * (int)gridDim.x + (int)blockIdx.x) * kWaves + wib;
        const bool on = pair < a.pairs.n;
        const int np = on ? cst(a.pairs.ppn)[pair] : 0;
        const int sA = on ? cst(a.pairs.shA)[pair] : 0, sB = on ? cst(a.pairs.shB)[pair] : 0;
        if (lane < 4 * MP) sums[wib][lane / MP][lane % MP] = 0.0;
        __syncthreads();
        double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
        if (np > 0) {
            const int nsl = 64 / np > 0 ? 64 / np : 1;       // shares of the nuclei (np <= 64)
            const int u = lane % np, slice = lane / np;
            if (slice < nsl) {
                const PrimPair P = a.pp[cst(a.pairs.ppo)[pair] + u];
                double acc[Cls::NACC];
#pragma unroll
                for (int k = 0; k < Cls::NACC; ++k) acc[k] = 0.0;
                const double w = -kTwoPi * P.Kp;
                for (int n = slice; n < a.nnuc; n += nsl) {
                    const double PCx = P.Px - a.R[3 * n], PCy = P.Py - a.R[3 * n + 1], PCz = P.Pz - a.R[3 * n + 2];
                    double F[L + 1];
                    boys_lds<L>(P.p * (PCx * PCx + PCy * PCy + PCz * PCz), F, sb);
                    const double pref = w * a.Z[n];
#pragma unroll
                    for (int m = 0; m <= L; ++m) F[m] *= pref;
                    Cls::vrr(F, acc, P.PAx, P.PAy, P.PAz, PCx, PCy, PCz, P.inv2p);
                }
                // overlap and second-derivative factors per axis; the first share adds T and S
                const double* ABp = a.pairs.AB + 3 * pair;
                const double AB[3] = {ABp[0], ABp[1], ABp[2]};
                const double PA[3] = {P.PAx, P.PAy, P.PAz};
                const double beta = P.pad, alpha = P.p - P.pad;
                double s[3][LA + 3][LB + 5], k[3][LA + 3][LB + 3];
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const double PB = PA[t] + AB[t];
#pragma unroll
                    for (int i = 0; i < LA + 3; ++i) {
                        if (i == 0) s[t][0][0] = 1.0;
                        else s[t][i][0] = PA[t] * s[t][i - 1][0] + (i > 1 ? P.inv2p * (i - 1) * s[t][i - 2][0] : 0.0);
#pragma unroll
                        for (int j = 1; j < LB + 5; ++j)
                            s[t][i][j] = PB * s[t][i][j - 1] + (i > 0 ? P.inv2p * i * s[t][i - 1][j - 1] : 0.0) +
                                         (j > 1 ? P.inv2p * (j - 1) * s[t][i][j - 2] : 0.0);
                    }
#pragma unroll
                    for (int i = 0; i < LA + 3; ++i)
#pragma unroll
                        for (int j = 0; j < LB + 3; ++j)
                            k[t][i][j] = -2.0 * beta * (2 * j + 1) * s[t][i][j] + 4.0 * beta * beta * s[t][i][j + 2] +
                                         (j > 1 ? (double)(j * (j - 1)) * s[t][i][j - 2] : 0.0);
                }
                const double pre = slice == 0 ? kPi32 * P.Kp * rsqrt(P.p) : 0.0;
                const double fac = sA == sB ? 1.0 : 2.0;
                double wd[NA * NB], ww[NA * NB];
#pragma unroll
                for (int ia = 0; ia < NA; ++ia)
#pragma unroll
                    for (int ib = 0; ib < NB; ++ib) {
                        const int fa = a.sh[sA].bf[ia], fb = a.sh[sB].bf[ib];
                        const bool have = fa >= 0 && fb >= 0;
                        const size_t o = have ? (size_t)fa * a.N + fb : 0;
                        const double sc = have ? fac * a.sh[sA].sc[ia] * a.sh[sB].sc[ib] : 0.0;
                        wd[ia * NB + ib] = sc * a.Dt[o];
                        ww[ia * NB + ib] = sc * a.W[o];
                    }
                double gl = 0.0, gxa = 0.0, gxb = 0.0;
                Cls::derivatives(acc, s, k, pre, wd, ww, alpha, beta, AB[0], AB[1], AB[2], gl, gxa, gxb, gA, gB);
                const int kab = a.ppk[cst(a.pairs.ppo)[pair] + u];
                const int ka = kab & 0xffff, kb = kab >> 16;
                atomicAdd(&sums[wib][0][ka], gxa);
                atomicAdd(&sums[wib][1][kb], gxb);
                atomicAdd(&sums[wib][2][ka], gl);
                atomicAdd(&sums[wib][3][kb], gl);
            }
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            gA[t] = wave_sum(gA[t]);
            gB[t] = wave_sum(gB[t]);
        }
        if (np > 0) {
            if (lane < 4 * MP) {
                const int q = lane / MP, k = lane % MP;
                const int sh = q & 1 ? sB : sA;
                if (k < a.sh[sh].nprim) atomicAdd((q < 2 ? a.g_xpn : a.g_lin) + a.poff[sh] + k, sums[wib][q][k]);
            } else if (lane < 4 * MP + 6) {
                const int c = lane - 4 * MP;
                const double v = c == 0 ? gA[0] : c == 1 ? gA[1] : c == 2 ? gA[2] : c == 3 ? gB[0] : c == 4 ? gB[1] : gB[2];
                atomicAdd(a.g_cen + 3 * (c < 3 ? sA : sB) + c % 3, v);
            }
        }
        __syncthreads();    // the sums are cleared by the next pass
    }
}

// Blocks of a launch over n shell pairs: one wave a pair, at most 8 blocks a CU
// (a block stages 14-24 KB of Boys rows once and then walks its pairs).
unsigned pair_blocks(int n)
{
    const int b = (n + kWaves - 1) / kWaves;
    return (unsigned)(b < 2048 ? b : 2048);
}

}  // namespace

void launch_nuclear(int la, int lb, const NucArgs& a, hipStream_t s)
{
    static_assert(2 * QBX_MAXL <= QBX_BOYSL_LMAX, "Boys rows for the nuclear attraction");
    if (a.pairs.n <= 0) return;
    const dim3 grid(pair_blocks(a.pairs.n)), block(64 * kWaves);
#define QBX_NUC(A, B) \
    if (la == A && lb == B) hipLaunchKernelGGL((nuclear_kernel<A, B>), grid, block, 0, s, a);
    QBX_NUC(0, 0) QBX_NUC(1, 0) QBX_NUC(1, 1) QBX_NUC(2, 0) QBX_NUC(2, 1) QBX_NUC(2, 2)
    QBX_NUC(3, 0) QBX_NUC(3, 1) QBX_NUC(3, 2) QBX_NUC(3, 3)
    QBX_NUC(4, 0) QBX_NUC(4, 1) QBX_NUC(4, 2) QBX_NUC(4, 3) QBX_NUC(4, 4)
#undef QBX_NUC
    QBX_HIP(hipGetLastError());
}

void launch_one_e_grad(int la, int lb, const NucArgs& a, hipStream_t s)
{
    static_assert(QBX_GRAD_MAXP * QBX_GRAD_MAXP <= 64 && 4 * QBX_GRAD_MAXP + 6 <= 64, "lanes of a shell pair");
    if (a.pairs.n <= 0) return;
    const dim3 grid(pair_blocks(a.pairs.n)), block(64 * kWaves);
    if (la == 0 && lb == 0) hipLaunchKernelGGL((one_e_grad_kernel<0, 0>), grid, block, 0, s, a);
    else if (la == 1 && lb == 0) hipLaunchKernelGGL((one_e_grad_kernel<1, 0>), grid, block, 0, s, a);
    else if (la == 1 && lb == 1) hipLaunchKernelGGL((one_e_grad_kernel<1, 1>), grid, block, 0, s, a);
    else throw QbxError(QBX_EINTERNAL, "no one-electron gradient kernel for the pair class");
    QBX_HIP(hipGetLastError());
}

}  // namespace qbx
