// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4f64) and the
// small kernels of trace-correcting purification.
//
// MFMA f64 16x16x4 operand layout (one wave): lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16]; the four result registers r hold
// D[4 r + l / 16][l % 16].
#include <cstdint>

#include "qbx_common.h"
#include "qbx_linalg.h"

namespace qbx {
namespace {

constexpr int GK = 16;   // K step (four MFMA steps)

typedef double dbl4 __attribute__((ext_vector_type(4)));

struct GemmF64 {
    const double* A;
    const double* B;
    const double* Z;
    double* C;
    int M, N, K, lda, ldb, ldz, ldc;
    double alpha, beta;
};

// Block of four waves in a 2 x 2 arrangement; each wave owns WT x WT tiles of
// 16 x 16 outputs, so the block tile is 32 WT square.  WT = 2 reads half the
// LDS bytes per MFMA of WT = 1 and is taken where the grid still has several
// blocks per CU.
template <bool TA, bool TB, int WT>
__global__ __launch_bounds__(256) void gemm_f64_kernel(GemmF64 g)
{
    constexpr int BT = 32 * WT;
    constexpr int LOADS = GK * BT / 256;
    __shared__ double As[GK][BT + 1];   // As[k][i] = op(A)[row0 + i][k0 + k]
    __shared__ double Bs[GK][BT + 1];   // Bs[k][j] = op(B)[k0 + k][col0 + j]
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int w = t >> 6;
    const int wr = w >> 1, wc = w & 1;
    // 1-D grid, the column tiles of one row panel adjacent: a tall operand
    // (M up to 2^31 rows) is read from HBM once and reused from L2
    const int ntile = (g.N + BT - 1) / BT;
    const int row0 = (int)(blockIdx.x / ntile) * BT, col0 = (int)(blockIdx.x % ntile) * BT;
    dbl4 acc[WT][WT];
#pragma unroll
    for (int a = 0; a < WT; ++a)
#pragma unroll
        for (int b = 0; b < WT; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
    // tile loads: GK x BT elements of each operand, LOADS per thread,
    // coalesced along the operand's contiguous index; the next K step's loads
    // are issued before the current step's MFMAs
    double ra[LOADS], rb[LOADS];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int h = 0; h < LOADS; ++h) {
            const int e = t + 256 * h;
            int i, k;
            if (TA) { k = e / BT; i = e % BT; } else { i = e / GK; k = e % GK; }
            const int gi = row0 + i, gk = k0 + k;
            ra[h] = (gi < g.M && gk < g.K) ? (TA ? g.A[(size_t)gk * g.lda + gi] : g.A[(size_t)gi * g.lda + gk]) : 0.0;
            int j;
            if (TB) { j = e / GK; k = e % GK; } else { k = e / BT; j = e % BT; }
            const int gj = col0 + j, gk2 = k0 + k;
            rb[h] = (gj < g.N && gk2 < g.K) ? (TB ? g.B[(size_t)gj * g.ldb + gk2] : g.B[(size_t)gk2 * g.ldb + gj]) : 0.0;
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < g.K; k0 += GK) {
#pragma unroll
        for (int h = 0; h < LOADS; ++h) {
            const int e = t + 256 * h;
            int i, k;
            if (TA) { k = e / BT; i = e % BT; } else { i = e / GK; k = e % GK; }
            As[k][i] = ra[h];
            int j;
            if (TB) { j = e / GK; k = e % GK; } else { k = e / BT; j = e % BT; }
            Bs[k][j] = rb[h];
        }
        __syncthreads();
        if (k0 + GK < g.K) fetch(k0 + GK);
#pragma unroll
        for (int kk = 0; kk < GK / 4; ++kk) {
            double a[WT], b[WT];
#pragma unroll
            for (int m = 0; m < WT; ++m) {
                a[m] = As[4 * kk + (lane >> 4)][(wr * WT + m) * 16 + (lane & 15)];
                b[m] = Bs[4 * kk + (lane >> 4)][(wc * WT + m) * 16 + (lane & 15)];
            }
#pragma unroll
            for (int m = 0; m < WT; ++m)
#pragma unroll
                for (int n = 0; n < WT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[m], b[n], acc[m][n], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < WT; ++m)
#pragma unroll
        for (int n = 0; n < WT; ++n) {
            const int j = col0 + (wc * WT + n) * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = row0 + (wr * WT + m) * 16 + 4 * r + (lane >> 4);
                if (i < g.M && j < g.N) {
                    double v = g.alpha * acc[m][n][r];
                    if (g.beta != 0.0) v += g.beta * g.Z[(size_t)i * g.ldz + j];
                    g.C[(size_t)i * g.ldc + j] = v;
                }
            }
        }
}

// Four k values (k0 + 4 (l/16) + 0..3) of op(X)'s row r for MFMA steps 0..3: an
// MFMA may take its four k in any order as long as both operands take the same,
// so a lane's four are neighbours in memory where k is the contiguous index (two
// 16-byte loads with VEC) and no LDS pass is needed.  T: X is stored [k][r].
template <bool T, bool VEC> __device__ __forceinline__ dbl4 load_k4(const double* X, int ld, int r, int k)
{
    if (T) {
        const double* p = X + (size_t)k * ld + r;
        return dbl4{p[0], p[ld], p[2 * (size_t)ld], p[3 * (size_t)ld]};
    }
    const double* p = X + (size_t)r * ld + k;
    if (VEC) {
        const double2 a = ((const double2*)p)[0], b = ((const double2*)p)[1];
        return dbl4{a.x, a.y, b.x, b.y};
    }
    return dbl4{p[0], p[1], p[2], p[3]};
}

// the same at the end of K
template <bool T> __device__ __forceinline__ dbl4 load_k4_tail(const double* X, int ld, int r, int k, int K)
{
    dbl4 v = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s)
        if (k + s < K) v[s] = T ? X[(size_t)(k + s) * ld + r] : X[(size_t)r * ld + k + s];
    return v;
}

__device__ __forceinline__ void mfma_16k(const dbl4* a, const dbl4* b, dbl4 (*acc)[2])
{
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n)
                acc[m][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[m][k], b[n][k], acc[m][n], 0, 0, 0);
}

// GEMMs whose 64 x 64 tiles would not fill the chip: a block owns 32 x 32 outputs
// and its four waves split K, each summing all four 16 x 16 tiles over its share,
// 16 MFMAs for every eight 16-byte loads, two steps in flight, no barriers; the
// shares are added in wave order.  Rows beyond the operand read its last row
// (their outputs are not stored), and steps beyond the share its last step, so that
// every load is unconditional and the waits are exact (with guarded loads the
// compiler waited for all of them at every step: 27 us at 600^3).  Against four
// waves on one 16 x 16 tile each and K through LDS, two barriers every 16 k: 600^3
// 27.8 -> 22 us, 301^3 10.3 -> 7.8, 1024^3 61.6 -> 53, 70 x 4900 x 4900 187 -> 124.
// Below KSPLIT_MIN the other form is as fast or faster (20000 x 33 x 33: 7.0
// against 9.1 us).
constexpr int SPLIT = 4;
constexpr int KSPLIT_MIN = 256;

template <bool TA, bool TB, bool VEC>
__global__ __launch_bounds__(64 * SPLIT) void gemm_f64_split_kernel(GemmF64 g)
{
    __shared__ double red[SPLIT][4 * 256];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int ntile = (g.N + 31) / 32;
    const int row0 = (int)(blockIdx.x / ntile) * 32, col0 = (int)(blockIdx.x % ntile) * 32;
    const int r = lane & 15, q = lane >> 4;
    const int steps = g.K / 16;       // whole steps (K >= KSPLIT_MIN: every wave has some)
    const int s0 = steps * w / SPLIT, s1 = steps * (w + 1) / SPLIT;
    const int ra[2] = {min(row0 + r, g.M - 1), min(row0 + 16 + r, g.M - 1)};
    const int rb[2] = {min(col0 + r, g.N - 1), min(col0 + 16 + r, g.N - 1)};
    dbl4 acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = dbl4{0.0, 0.0, 0.0, 0.0};
    dbl4 a[3][2], b[3][2];
    auto fetch = [&](int s, int d) {
        const int k = 16 * min(s, s1 - 1) + 4 * q;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            a[d][m] = load_k4<TA, VEC>(g.A, g.lda, ra[m], k);
            b[d][m] = load_k4<!TB, VEC>(g.B, g.ldb, rb[m], k);
        }
    };
    fetch(s0, 0);
    fetch(s0 + 1, 1);
    int s = s0;
    for (; s + 3 <= s1; s += 3) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            fetch(s + d + 2, (d + 2) % 3);
            mfma_16k(a[d], b[d], acc);
        }
    }
    if (s < s1) mfma_16k(a[0], b[0], acc);
    if (s + 1 < s1) mfma_16k(a[1], b[1], acc);
    if (w == SPLIT - 1 && 16 * steps < g.K) {
        const int k = 16 * steps + 4 * q;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            a[0][m] = load_k4_tail<TA>(g.A, g.lda, ra[m], k, g.K);
            b[0][m] = load_k4_tail<!TB>(g.B, g.ldb, rb[m], k, g.K);
        }
        mfma_16k(a[0], b[0], acc);
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[w][(16 * m + 4 * e + q) * 32 + 16 * n + r] = acc[m][n][e];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        const int e = t + 256 * h;
        const int i = row0 + e / 32, j = col0 + e % 32;
        if (i >= g.M || j >= g.N) continue;
        double v = red[0][e];
#pragma unroll
        for (int k = 1; k < SPLIT; ++k) v += red[k][e];
        v *= g.alpha;
        if (g.beta != 0.0) v += g.beta * g.Z[(size_t)i * g.ldz + j];
        g.C[(size_t)i * g.ldc + j] = v;
    }
}

// out[(a nao + b) nmo + m] = C[a][m] C[b][m]: the orbital-pair columns of the
// opposite-spin Coulomb matrix
__global__ void pair_columns_kernel(const double* C, int nao, int nmo, size_t tot, double* out)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= tot) return;
    const int m = (int)(e % nmo);
    const size_t ab = e / nmo;
    const int a = (int)(ab / nao), b = (int)(ab % nao);
    out[e] = C[(size_t)a * nmo + m] * C[(size_t)b * nmo + m];
}

// one wave a row
__global__ __launch_bounds__(256) void gershgorin_kernel(const double* P, int n, double* lohi)
{
    const int lane = threadIdx.x & 63, i = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    double r = 0.0;
    for (int j = lane; j < n; j += 64)
        if (j != i) r += fabs(P[(size_t)i * n + j]);
    for (int o = 32; o > 0; o >>= 1) r += __shfl_xor(r, o);
    const double c = P[(size_t)i * n + i];
    if (lane == 0) {
        lohi[2 * i] = c - r;
        lohi[2 * i + 1] = c + r;
    }
}

// ---------------------------------------------------------------------------
// Trace-correcting purification (SP2) without a host decision per product.  The
// matrices are symmetric and padded with zeros to a multiple of 32 rows, so the
// products take the 32 x 32 tiles on and above the diagonal only (block b of
// sp2_tile), read both operands as rows, and need no bounds checks.  Every kernel
// leaves each tile's share of tr P and |P|_F^2; the next product's blocks all add
// the shares in the same order and so all take the same decision.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void sp2_tile(int b, int& ti, int& tj)
{
    tj = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
    while ((tj + 1) * (tj + 2) / 2 <= b) ++tj;
    while (tj * (tj + 1) / 2 > b) --tj;
    ti = b - tj * (tj + 1) / 2;
}

// Adds tile b's values (v of element e = thread + 256 h, row e / 32, column e %
// 32) to its shares of tr P and |P|_F^2: an off-diagonal tile stands for two.
template <int TPB>
__device__ __forceinline__ void sp2_shares(double tr, double fr, bool diag, int b, double* shares)
{
    __shared__ double s_tr[TPB / 64], s_fr[TPB / 64];
    for (int o = 32; o > 0; o >>= 1) {
        tr += __shfl_xor(tr, o);
        fr += __shfl_xor(fr, o);
    }
    if ((threadIdx.x & 63) == 0) {
        s_tr[threadIdx.x >> 6] = tr;
        s_fr[threadIdx.x >> 6] = fr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, f = 0.0;
        for (int k = 0; k < TPB / 64; ++k) {
            a += s_tr[k];
            f += s_fr[k];
        }
        shares[2 * b] = a;
        shares[2 * b + 1] = diag ? f : 2.0 * f;
    }
}

// tr P and |P|_F^2 from the shares; every thread of the block gets them
template <int TPB>
__device__ __forceinline__ void sp2_measure(const double* shares, int nblk, double& tr, double& fr)
{
    __shared__ double s_tr[TPB / 64], s_fr[TPB / 64];
    double a = 0.0, f = 0.0;
    for (int k = threadIdx.x; k < nblk; k += TPB) {
        a += shares[2 * k];
        f += shares[2 * k + 1];
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        f += __shfl_xor(f, o);
    }
    if ((threadIdx.x & 63) == 0) {
        s_tr[threadIdx.x >> 6] = a;
        s_fr[threadIdx.x >> 6] = f;
    }
    __syncthreads();
    tr = 0.0;
    fr = 0.0;
    for (int k = 0; k < TPB / 64; ++k) {
        tr += s_tr[k];
        fr += s_fr[k];
    }
}

// P = (hi - F) / (hi - lo), F's symmetric part (n x n), padded to np
__global__ __launch_bounds__(256) void sp2_start_kernel(const double* F, int n, int np, const double* lohi, double* P,
                                                        double* shares, Sp2State* state)
{
    int ti, tj;
    sp2_tile(blockIdx.x, ti, tj);
    const double lo = lohi[0];
    double hi = lohi[1];
    if (!(hi > lo)) hi = lo + 1.0;
    double tr = 0.0, fr = 0.0;
    for (int h = 0; h < 4; ++h) {
        const int e = threadIdx.x + 256 * h;
        const int i = 32 * ti + e / 32, j = 32 * tj + e % 32;
        double v = 0.0;
        if (i < n && j < n)
            v = ((i == j ? hi : 0.0) - 0.5 * (F[(size_t)i * n + j] + F[(size_t)j * n + i])) / (hi - lo);
        P[(size_t)i * np + j] = v;
        if (ti != tj) P[(size_t)j * np + i] = v;
        fr += v * v;
        if (i == j) tr += v;
    }
    sp2_shares<256>(tr, fr, ti == tj, blockIdx.x, shares);
    if (blockIdx.x == 0 && threadIdx.x == 0) state[0] = Sp2State{-1, 0, 0, 0};
}

// Product k: Q = P^2 or 2P - P^2, whichever moves the trace toward nocc, or
// nothing once the projector has settled (two products after |tr P - |P|_F^2| and
// the trace's error are small).  A block's eight waves split K as in
// gemm_f64_split_kernel.  Half the tiles, no separate pass for the trace and the
// norm (one block read the matrix for 85 us) and no host round trip: 140 -> 15 us a
// product at n = 600, of which 4.5 us is an empty launch with its shares and 4 us
// the MFMA time of the 190 blocks.
constexpr int SP2_WAVES = 8;

__global__ __launch_bounds__(64 * SP2_WAVES) void sp2_product_kernel(const double* P, double* Q, int np, int nblk,
                                                                    double nocc, const double* shares_in,
                                                                    double* shares_out, const Sp2State* in,
                                                                    Sp2State* out)
{
    constexpr int TPB = 64 * SP2_WAVES;
    __shared__ double red[SP2_WAVES / 2][32 * 33];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    int ti, tj;
    sp2_tile(blockIdx.x, ti, tj);
    const int r = lane & 15, q = lane >> 4;
    const int steps = np / 16;
    const int s0 = steps * w / SP2_WAVES, s1 = steps * (w + 1) / SP2_WAVES;
    const double* pa = P + (size_t)(32 * ti + r) * np + 4 * q;
    const double* pb = P + (size_t)(32 * tj + r) * np + 4 * q;
    // two steps in flight, the first ones (and P's own tile) while the shares are added
    dbl4 acc[2][2], a[3][2], b[3][2];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[m][n] = dbl4{0.0, 0.0, 0.0, 0.0};
    auto fetch = [&](int s, int d) {    // unconditional: steps beyond the share read its last one
        const int k = 16 * min(s, steps - 1);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            a[d][m] = *(const dbl4*)(pa + (size_t)(16 * m) * np + k);
            b[d][m] = *(const dbl4*)(pb + (size_t)(16 * m) * np + k);
        }
    };
    fetch(s0, 0);
    fetch(s0 + 1, 1);
    double own[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = t + TPB * h;
        own[h] = P[(size_t)(32 * ti + e / 32) * np + 32 * tj + e % 32];
    }
    Sp2State st = *in;
    double tr, fr;
    sp2_measure<TPB>(shares_in, nblk, tr, fr);
    if (!st.stop) {
        if (st.tail < 0 && fabs(tr - fr) < 1e-8 * fmax(1.0, nocc) && fabs(tr - nocc) < 1e-6) st.tail = 2;
        if (st.tail == 0) st.stop = 1;
        else if (st.tail > 0) --st.tail;
    }
    if (!st.stop) ++st.it;
    if (blockIdx.x == 0 && t == 0) *out = st;
    if (st.stop) return;
    const bool square = fabs(fr - nocc) <= fabs(2.0 * tr - fr - nocc);
    int s = s0;
    for (; s + 3 <= s1; s += 3) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            fetch(s + d + 2, (d + 2) % 3);
            mfma_16k(a[d], b[d], acc);
        }
    }
    if (s < s1) mfma_16k(a[0], b[0], acc);
    if (s + 1 < s1) mfma_16k(a[1], b[1], acc);
    // shares of K: the upper waves' to LDS, the lower waves add theirs
    constexpr int H = SP2_WAVES / 2;
    auto each = [&](auto f) {
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) f(red[w % H][(16 * m + 4 * e + q) * 33 + 16 * n + r], acc[m][n][e]);
    };
    if (w >= H) each([](double& x, double v) { x = v; });
    __syncthreads();
    if (w < H) each([](double& x, double v) { x = v + x; });
    __syncthreads();
    double tr1 = 0.0, fr1 = 0.0;
    double v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int e = t + TPB * h, i = e / 32, j = e % 32;
        double x = red[0][i * 33 + j];
#pragma unroll
        for (int k = 1; k < H; ++k) x += red[k][i * 33 + j];
        const size_t o = (size_t)(32 * ti + i) * np + 32 * tj + j;
        if (!square) x = 2.0 * own[h] - x;
        v[h] = x;
        Q[o] = x;
        fr1 += x * x;
        if (ti == tj && i == j) tr1 += x;
    }
    if (ti != tj) {    // the mirrored tile, rows along its own memory
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = t + TPB * h;
            red[0][(e / 32) * 33 + e % 32] = v[h];
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int e = t + TPB * h, i = e / 32, j = e % 32;
            Q[(size_t)(32 * tj + i) * np + 32 * ti + j] = red[0][j * 33 + i];
        }
    }
    sp2_shares<TPB>(tr1, fr1, ti == tj, blockIdx.x, shares_out);
}

// state and measures of the latest matrix, for the host
__global__ __launch_bounds__(256) void sp2_status_kernel(const double* shares, int nblk, const Sp2State* s,
                                                         Sp2Status* out)
{
    double tr, fr;
    // the shares alternate with the products made (none more once stopped)
    sp2_measure<256>(shares + (size_t)(s->it & 1) * 2 * nblk, nblk, tr, fr);
    if (threadIdx.x == 0) *out = Sp2Status{*s, tr, fr};
}

// P <- (P + P^T) / 2 in place, one thread per (i, j) with i < j
__global__ void symmetrize_square_kernel(double* P, int n)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    const size_t i = e / n, j = e % n;
    if (i >= j) return;
    const double v = 0.5 * (P[i * n + j] + P[j * n + i]);
    P[i * n + j] = v;
    P[j * n + i] = v;
}

// column signs: sgn[j] = -1 where C[0][j] < 0, else 1
__global__ void column_sign_kernel(const double* C, int n, double* sgn)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) sgn[j] = C[j] < 0.0 ? -1.0 : 1.0;
}

__global__ void scale_columns_kernel(double* C, int n, const double* sgn)
{
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)n * n) return;
    C[e] *= sgn[e % n];
}

// out[0] = min_i lohi[2i], out[1] = max_i lohi[2i+1]: the spectral interval
// from the rows' Gershgorin intervals (one block; min and max are exact in
// any order)
__global__ __launch_bounds__(1024) void interval_kernel(const double* lohi, int n, double* out)
{
    __shared__ double s_lo[16], s_hi[16];
    double lo = lohi[0], hi = lohi[1];
    for (int i = threadIdx.x; i < n; i += 1024) {
        lo = fmin(lo, lohi[2 * i]);
        hi = fmax(hi, lohi[2 * i + 1]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o));
        hi = fmax(hi, __shfl_xor(hi, o));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s_lo[w] = lo;
        s_hi[w] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < 16; ++k) {
            lo = fmin(lo, s_lo[k]);
            hi = fmax(hi, s_hi[k]);
        }
        out[0] = fmin(lo, s_lo[0]);
        out[1] = fmax(hi, s_hi[0]);
    }
}

}  // namespace

void gemm_f64(bool trans_a, bool trans_b, int M, int N, int K, double alpha, const double* A, int lda,
              const double* B, int ldb, double beta, const double* Z, int ldz, double* C, int ldc, hipStream_t s)
{
    if (M <= 0 || N <= 0) return;
    if (beta != 0.0 && !Z) throw QbxError(QBX_EINVAL, "GEMM addend missing");
    GemmF64 g{A, B, Z, C, M, N, K, lda, ldb, ldz, ldc, alpha, beta};
    // 64 x 64 blocks where they give 1024 or more (four a CU), else 32 x 32 blocks,
    // with K split over the block's waves from K = KSPLIT_MIN on
    const size_t big = (size_t)((N + 63) / 64) * (size_t)((M + 63) / 64);
    const int bt = big >= 1024 ? 64 : 32;
    const size_t tiles = (size_t)((N + bt - 1) / bt) * (size_t)((M + bt - 1) / bt);
    if (tiles > 0x7fffffffu) throw QbxError(QBX_EUNSUP, "GEMM too large for one grid");
    const dim3 grid((unsigned)tiles), block(256);
    auto launch = [&](void (*kern)(GemmF64)) {
        void* args[] = {&g};
        QBX_HIP(hipLaunchKernel((const void*)kern, grid, block, args, 0, s));
    };
    const int op = (trans_a ? 2 : 0) + (trans_b ? 1 : 0);
    static void (*const k64[4])(GemmF64) = {gemm_f64_kernel<false, false, 2>, gemm_f64_kernel<false, true, 2>,
                                            gemm_f64_kernel<true, false, 2>, gemm_f64_kernel<true, true, 2>};
    static void (*const k32[4])(GemmF64) = {gemm_f64_kernel<false, false, 1>, gemm_f64_kernel<false, true, 1>,
                                            gemm_f64_kernel<true, false, 1>, gemm_f64_kernel<true, true, 1>};
    static void (*const ksplit[2][4])(GemmF64) = {
        {gemm_f64_split_kernel<false, false, false>, gemm_f64_split_kernel<false, true, false>,
         gemm_f64_split_kernel<true, false, false>, gemm_f64_split_kernel<true, true, false>},
        {gemm_f64_split_kernel<false, false, true>, gemm_f64_split_kernel<false, true, true>,
         gemm_f64_split_kernel<true, false, true>, gemm_f64_split_kernel<true, true, true>}};
    // 16-byte loads along k where every row of an operand with contiguous k starts on 16 bytes
    const bool vec = (trans_a || (((uintptr_t)A & 15) == 0 && (lda & 1) == 0)) &&
                     (!trans_b || (((uintptr_t)B & 15) == 0 && (ldb & 1) == 0));
    launch(bt == 64 ? k64[op] : K >= KSPLIT_MIN ? ksplit[vec][op] : k32[op]);
    QBX_HIP(hipGetLastError());
}

void pair_columns(const double* C, int nao, int nmo, double* out, hipStream_t s)
{
    const size_t tot = (size_t)nao * nao * nmo;
    if (tot == 0) return;
    hipLaunchKernelGGL(pair_columns_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s, C, nao, nmo, tot,
                       out);
    QBX_HIP(hipGetLastError());
}

void gershgorin(const double* P, int n, double* lohi, hipStream_t s)
{
    hipLaunchKernelGGL(gershgorin_kernel, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, P, n, lohi);
    QBX_HIP(hipGetLastError());
}

void symmetrize_square(double* P, int n, hipStream_t s)
{
    const size_t nn = (size_t)n * n;
    hipLaunchKernelGGL(symmetrize_square_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, s, P, n);
    QBX_HIP(hipGetLastError());
}

void fix_column_signs(double* C, int n, double* sgn, hipStream_t s)
{
    const size_t nn = (size_t)n * n;
    hipLaunchKernelGGL(column_sign_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, C, n, sgn);
    QBX_HIP(hipGetLastError());
    hipLaunchKernelGGL(scale_columns_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, s, C, n, sgn);
    QBX_HIP(hipGetLastError());
}

void spectral_interval(const double* lohi, int n, double* out, hipStream_t s)
{
    hipLaunchKernelGGL(interval_kernel, dim3(1), dim3(1024), 0, s, lohi, n, out);
    QBX_HIP(hipGetLastError());
}

int sp2_padded(int n) { return (n + 31) / 32 * 32; }
int sp2_blocks(int n)
{
    const int t = sp2_padded(n) / 32;
    return t * (t + 1) / 2;
}

void sp2_start(const double* F, int n, const double* lohi, double* P, double* shares, Sp2State* state, hipStream_t s)
{
    hipLaunchKernelGGL(sp2_start_kernel, dim3((unsigned)sp2_blocks(n)), dim3(256), 0, s, F, n, sp2_padded(n), lohi, P,
                       shares, state);
    QBX_HIP(hipGetLastError());
}

void sp2_product(const double* P, double* Q, int n, int nocc, int k, double* shares, Sp2State* state, hipStream_t s)
{
    const int nb = sp2_blocks(n);
    hipLaunchKernelGGL(sp2_product_kernel, dim3((unsigned)nb), dim3(64 * SP2_WAVES), 0, s, P, Q, sp2_padded(n), nb,
                       (double)nocc, shares + (size_t)(k & 1) * 2 * nb, shares + (size_t)((k + 1) & 1) * 2 * nb,
                       state + (k & 1), state + ((k + 1) & 1));
    QBX_HIP(hipGetLastError());
}

void sp2_status(const double* shares, int n, int k, const Sp2State* state, Sp2Status* out, hipStream_t s)
{
    hipLaunchKernelGGL(sp2_status_kernel, dim3(1), dim3(256), 0, s, shares, sp2_blocks(n), state + (k & 1), out);
    QBX_HIP(hipGetLastError());
}

}  // namespace qbx

extern "C" {

int qbx_gemm_f64(int32_t trans_a, int32_t trans_b, int32_t M, int32_t N, int32_t K, double alpha, const double* A,
                 int32_t lda, const double* B, int32_t ldb, double beta, double* C, int32_t ldc, void* stream)
{
    return qbx::guarded([&] {
        if (M < 0 || N < 0 || K < 0) throw qbx::QbxError(QBX_EINVAL, "negative GEMM size");
        if (!A || !B || !C) throw qbx::QbxError(QBX_EINVAL, "null GEMM operand");
        if ((trans_a ? lda < M : lda < K) || (trans_b ? ldb < K : ldb < N) || ldc < N)
            throw qbx::QbxError(QBX_EINVAL, "leading dimension too small");
        qbx::gemm_f64(trans_a != 0, trans_b != 0, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, C, ldc,
                      (hipStream_t)stream);
    });
}

}  // extern "C"
