// FP64 GEMM on the CDNA4 matrix cores (v_mfma_f64_16x16x4f64), trace-correcting
// purification on the device, and the Householder tridiagonalization of the Fock solve.
//
// MFMA f64 16x16x4 operand layout (one wave): lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16]; the four result registers r hold
// D[4 r + l / 16][l % 16].
#include <algorithm>
#include <cmath>
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
// Which form takes a product (split_k) follows from times of both at 100 to 3600
// tiles and K of 256 to 6000: below KSPLIT_MIN the other is as fast or faster (20000 x
// 33 x 33: 7.0 against 9.1 us); many tiles fill the chip without splitting K, and a
// short K then does not pay for the sum over the waves (20000 x 33 x 300, 1250 tiles:
// 40 us against 34; 60000 x 32 x 256, 1875: 42 against 39; but 1200^3, 1444 tiles,
// 8-15% faster).  Where both operands are stored along k, a load takes 16 rows of 32
// bytes each of both, and the bounds lie lower (60000 x 32 x 256: 50 us against 39;
// 1000 x 1000 x 2000 8% slower).
constexpr int SPLIT = 4;
constexpr int KSPLIT_MIN = 256;
constexpr int KSPLIT_LONG = 512;
bool split_k(bool along_k, size_t tiles, int K)
{
    if (K < KSPLIT_MIN) return false;
    return tiles <= (along_k ? (K >= KSPLIT_LONG ? 640 : 256) : (K >= KSPLIT_LONG ? 1536 : 640));
}

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
    // with K split over the block's waves where that pays (split_k)
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
    launch(bt == 64 ? k64[op] : split_k(!trans_a && trans_b, tiles, K) ? ksplit[vec][op] : k32[op]);
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

// ---------------------------------------------------------------------------
// Householder tridiagonalization.  A step needs the whole pivot column and the
// whole product A v before any row can be updated, so a library that launches a
// few kernels a column pays their latency 600 times over (n = 600: 6000 launches,
// 9.7 of the 13.9 ms of a Fock solve).  Here one persistent grid holds the matrix in
// LDS, rows dealt to the blocks in turn, and the blocks exchange two numbers per
// row and step: p_r = (A v)_r and the next pivot column's element before the
// step's update.  From those every block forms the update's w, the next column
// and its reflector for itself, so one exchange a step is all; the latency of the
// exchange and of two block-wide sums (4 to 5 us a step) bounds it.  A Fock solve of
// n = 100, 250, 600, 1000 and 1800: 1.94 -> 1.70, 5.9 -> 3.4, 13.3 -> 7.5, 24.0 ->
// 13.7 and 49.5 -> 32.3 ms.
//
// The exchange needs no barrier: every value has a place of its own, filled with
// TRI_EMPTY before the launch, and a reader polls until it holds something else.
// Values cross the XCDs, so they are stored and loaded at agent scope.  A NaN is
// published as the plain quiet NaN, which is not TRI_EMPTY.  The launch is
// cooperative (all blocks resident), and a block that has polled one value `spins`
// times more sets *status and ends; the others then end the same way.
// ---------------------------------------------------------------------------
constexpr uint64_t TRI_EMPTY = ~0ull;
constexpr int TRI_MAX_N = 2048;   // 1024 threads, two elements each; 160 KB of LDS a block end at 1850

size_t tridiag_exchange(int n) { return 2 * (size_t)n * n; }

__global__ void tri_empty_kernel(uint64_t* p, size_t n, int* status)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = TRI_EMPTY;
    if (blockIdx.x == 0 && threadIdx.x == 0) *status = 0;
}

__device__ __forceinline__ void tri_put(uint64_t* p, double v)
{
    const uint64_t u = v != v ? 0x7ff8000000000000ull : __builtin_bit_cast(uint64_t, v);
    __hip_atomic_store(p, u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t tri_get(const uint64_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double tri_wave_sum(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// E elements of every length-n vector per thread: element e of a thread is
// threadIdx.x + e * blockDim.x.
template <int E>
__global__ __launch_bounds__(1024) void tridiag_kernel(int n, const double* A, double* V, double* d, double* e_out,
                                                       double* tau_out, uint64_t* exchange, int* status, int spins)
{
    extern __shared__ double lds[];
    __shared__ double red[3][16];
    __shared__ int fail;
    const int B = (int)gridDim.x, b = (int)blockIdx.x, T = (int)blockDim.x, tid = (int)threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, nwave = T >> 6;
    const int R = (n + B - 1) / B;
    double* rows = lds;                  // rows b, b + B, ...
    double* va = rows + (size_t)R * n;   // last step's reflector,
    double* wa = va + n;                 // its w,
    double* vb = wa + n;                 // this step's column, then reflector
    for (int i = tid; i < R * n; i += T) {
        const int r = b + (i / n) * B;
        if (r < n) rows[i] = A[(size_t)r * n + i % n];
    }
    if (tid == 0) fail = 0;
    auto block_sum = [&](double v, int which) {
        v = tri_wave_sum(v);
        if (lane == 0) red[which][wave] = v;
        __syncthreads();
        double sum = 0.0;
        for (int w = 0; w < nwave; ++w) sum += red[which][w];
        return sum;
    };
    double tau = 0.0;
    for (int k = 0; k < n - 1; ++k) {
        double x[E];
        if (k == 0) {
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                x[q] = r < n ? A[r] : 0.0;
            }
        } else {
            // last step's products and the column before its update
            const uint64_t* in = exchange + (size_t)(k - 1) * 2 * n;
            uint64_t up[E], ux[E];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                const bool on = r >= k && r < n;
                up[q] = on ? tri_get(in + r) : 0;
                ux[q] = on ? tri_get(in + n + r) : 0;
            }
            bool ok = true;
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                for (int i = 0; i < spins && (up[q] == TRI_EMPTY || ux[q] == TRI_EMPTY); ++i) {
                    up[q] = tri_get(in + r);
                    ux[q] = tri_get(in + n + r);
                }
                ok = ok && up[q] != TRI_EMPTY && ux[q] != TRI_EMPTY;
            }
            if (!ok) fail = 1;
            double dot = 0.0;
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                if (r >= k && r < n) dot += __builtin_bit_cast(double, up[q]) * va[r];
            }
            dot = block_sum(dot, 0);
            if (fail) {     // uniform: written before block_sum's barrier, and never reset
                if (tid == 0) *status = 1;
                return;
            }
            // w = tau (p - tau/2 (p.v) v); A <- A - v w' - w v'
            double w[E];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                w[q] = 0.0;
                if (r >= k && r < n) {
                    w[q] = tau * (__builtin_bit_cast(double, up[q]) - 0.5 * tau * dot * va[r]);
                    wa[r] = w[q];
                }
            }
            __syncthreads();
            const double wk = wa[k], vk = va[k];
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                x[q] = r >= k && r < n ? __builtin_bit_cast(double, ux[q]) - va[r] * wk - w[q] * vk : 0.0;
            }
        }
        // reflector of the column's part below the diagonal
        double ssq = 0.0, big = 0.0;
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int r = tid + q * T;
            if (r >= k && r < n) vb[r] = x[q];
            if (r == k && b == 0) d[k] = x[q];
            if (r >= k + 2 && r < n) ssq += x[q] * x[q];
        }
        ssq = block_sum(ssq, 1);
        const double alpha = vb[k + 1];
        double norm = sqrt(alpha * alpha + ssq);
        bool tail = true;    // entries below alpha
        if (!(ssq > 1e-280 && norm < 1e140)) {
            // no entries, or squares that may have lost digits or overflowed:
            // scaled by the largest entry
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                if (r >= k + 2 && r < n) big = fmax(big, fabs(x[q]));
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
            if (lane == 0) red[2][wave] = big;
            __syncthreads();
            for (int w = 0; w < nwave; ++w) big = fmax(big, red[2][w]);
            __syncthreads();
            tail = big > 0.0;
            big = fmax(big, fabs(alpha));
            double y2 = 0.0;
#pragma unroll
            for (int q = 0; q < E; ++q) {
                const int r = tid + q * T;
                const double y = tail && r >= k + 2 && r < n ? x[q] / big : 0.0;
                y2 += y * y;
            }
            y2 = block_sum(y2, 2);
            norm = tail ? big * sqrt(y2 + (alpha / big) * (alpha / big)) : fabs(alpha);
        }
        double beta = alpha, scale = 0.0, tau_k = 0.0;
        if (tail) {
            beta = alpha > 0.0 ? -norm : norm;
            tau_k = (beta - alpha) / beta;
            scale = 1.0 / (alpha - beta);
        }
        __syncthreads();    // alpha read
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int r = tid + q * T;
            if (r < k + 1 || r >= n) continue;
            const double v = r == k + 1 ? 1.0 : x[q] * scale;
            vb[r] = v;
            if (b == 0 && r > k + 1) V[(size_t)k * n + r] = v;
        }
        if (b == 0 && tid == 0) {
            e_out[k] = beta;
            tau_out[k] = tau_k;
        }
        __syncthreads();
        // this block's rows: last step's update, and their products with the reflector
        uint64_t* out = exchange + (size_t)k * 2 * n;
        for (int rr = wave; rr < R; rr += nwave) {
            const int r = b + rr * B;
            if (r <= k || r >= n) continue;
            double* row = rows + (size_t)rr * n;
            const double vr = k > 0 ? va[r] : 0.0, wr = k > 0 ? wa[r] : 0.0;
            double acc = 0.0, first = 0.0;
            for (int c = k + 1 + lane; c < n; c += 64) {
                double a = row[c];
                if (k > 0) {
                    a -= vr * wa[c] + wr * va[c];
                    row[c] = a;
                }
                if (c == k + 1) first = a;
                acc += a * vb[c];
            }
            acc = tri_wave_sum(acc);
            if (lane == 0) {
                tri_put(out + r, acc);
                tri_put(out + n + r, first);
                if (k == n - 2) d[n - 1] = first;
            }
        }
        __syncthreads();
        double* t = va;
        va = vb;
        vb = t;
        tau = tau_k;
    }
}

TridiagPlan tridiag_plan(int n)
{
    TridiagPlan plan;
    if (n < 2 || n > TRI_MAX_N) return plan;
    int dev = 0, cus = 0, coop = 0, lds_max = 0;
    QBX_HIP(hipGetDevice(&dev));
    QBX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    QBX_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    QBX_HIP(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    if (!coop || cus <= 0) return plan;
    const int threads = std::min(1024, (n + 63) / 64 * 64);
    const void* f = n > 1024 ? (const void*)tridiag_kernel<2> : (const void*)tridiag_kernel<1>;
    // the fewest blocks whose LDS holds the matrix: each value then has fewer readers
    // (n = 600: 64, 128 and 256 blocks 7.47, 7.64 and 7.95 ms a solve)
    int B = 64;
    size_t shm = 0;
    for (;; B *= 2) {
        B = std::min(std::min(B, cus), n);
        shm = ((size_t)((n + B - 1) / B) + 3) * n * sizeof(double);
        if (shm + 1024 <= (size_t)lds_max) break;
        if (B >= 256 || B >= cus || B >= n) return plan;
    }
    int per_cu = 0;
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, threads, shm) != hipSuccess || per_cu * cus < B) {
        (void)hipGetLastError();
        return plan;
    }
    plan.n = n;
    plan.blocks = B;
    plan.threads = threads;
    plan.shm = shm;
    return plan;
}

bool tridiagonalize(const TridiagPlan& plan, const double* A, double* V, double* d, double* e, double* tau,
                    uint64_t* exchange, int* status, int spins, hipStream_t s)
{
    if (plan.blocks <= 0) return false;
    int n = plan.n;
    const void* f = n > 1024 ? (const void*)tridiag_kernel<2> : (const void*)tridiag_kernel<1>;
    const size_t nx = tridiag_exchange(n);
    hipLaunchKernelGGL(tri_empty_kernel, dim3((unsigned)std::min<size_t>((nx + 255) / 256, 2048)), dim3(256), 0, s,
                       exchange, nx, status);
    QBX_HIP(hipGetLastError());
    void* args[] = {&n, &A, &V, &d, &e, &tau, &exchange, &status, &spins};
    if (hipLaunchCooperativeKernel(f, dim3(plan.blocks), dim3(plan.threads), args, (unsigned)plan.shm, s) !=
        hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// One block: d (n) and e (n - 1) times the power of two that brings their largest
// entry into [1, 2); *back undoes it.  Where the tridiagonalization gave up, its outputs
// are partly unwritten: the zero matrix and no reflectors instead, so that the solver
// queued behind never sees them.
__global__ void tri_scale_kernel(int n, double* d, double* e, double* tau, const int* status, double* back)
{
    __shared__ double red[16];
    if (*status != 0) {
        for (int i = threadIdx.x; i < n; i += blockDim.x) {
            d[i] = 0.0;
            if (i < n - 1) e[i] = tau[i] = 0.0;
        }
        if (threadIdx.x == 0) *back = 0.0;
        return;
    }
    double big = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) big = fmax(big, fmax(fabs(d[i]), i < n - 1 ? fabs(e[i]) : 0.0));
    for (int o = 32; o >= 1; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = big;
    __syncthreads();
    for (int w = 0; w < (int)blockDim.x / 64; ++w) big = fmax(big, red[w]);
    const int x = big > 0.0 && big < HUGE_VAL ? -ilogb(big) : 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        d[i] = ldexp(d[i], x);
        if (i < n - 1) e[i] = ldexp(e[i], x);
    }
    if (threadIdx.x == 0) *back = (double)-x;
}
__global__ void tri_unscale_kernel(int n, double* d, const double* back)
{
    for (int i = threadIdx.x; i < n; i += blockDim.x) d[i] = ldexp(d[i], (int)*back);
}

void tridiag_scale(int n, double* d, double* e, double* tau, const int* status, double* back, hipStream_t s)
{
    hipLaunchKernelGGL(tri_scale_kernel, dim3(1), dim3(1024), 0, s, n, d, e, tau, status, back);
    QBX_HIP(hipGetLastError());
}
void tridiag_unscale(int n, double* d, const double* back, hipStream_t s)
{
    hipLaunchKernelGGL(tri_unscale_kernel, dim3(1), dim3(1024), 0, s, n, d, back);
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
