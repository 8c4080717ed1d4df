// qbx_mlp.hip -- BF16 matrix-core kernels for the learned SCF initial guess
// (a pair-feature MLP): an MFMA GEMM with FP32 accumulation and the
// elementwise pieces of its forward and backward passes.  All pointers are
// device pointers; every call is enqueued on the given stream (NULL: the
// default stream) and returns without synchronizing.
//
// Storage: matrices row-major; BF16 values as raw 16-bit patterns (the upper
// half of an IEEE float, round-to-nearest-even on conversion).
#include "qbx.h"
#include "qbx_common.h"

#include <hip/hip_runtime.h>
#include <cstdint>

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ unsigned short f2bf(float x)
{
    unsigned u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)((u >> 16) | 0x40u);   // quiet NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

struct GemmArgs {
    const unsigned short* A;
    const unsigned short* B;
    float* C;
    const float* bias;
    unsigned short* Cb;   // BF16 copy of the output (epilogues EPI_BIAS_RELU_BF16, EPI_RELU_BACK)
    const unsigned short* H;   // BF16 activations (EPI_RELU_BACK), laid out as C
    int M, N, K, lda, ldb, ldc;
    float alpha, beta;
};

enum { EPI_STORE = 0, EPI_BIAS_RELU_BF16 = 1, EPI_BIAS = 2, EPI_RELU_BACK = 3 };

// The MFMA of both GEMM kernels is v_mfma_f32_32x32x8_bf16: per instruction lane
// l supplies A[m0 + l%32][k0 + 4(l/32) + j] and B[k0 + 4(l/32) + j][n0 + l%32] (j
// = 0..3) and holds the accumulators D[m0 + 8(i/4) + 4(l/32) + i%4][n0 + l%32], i
// = 0..15.  op(A) = A (M x K, row stride lda) or A^T (A stored K x M); likewise B.
__device__ __forceinline__ int acc_row(int i, int kq) { return 8 * (i / 4) + 4 * kq + (i % 4); }

template <int EPI> __device__ __forceinline__ void store_out(const GemmArgs& g, int row, int n, float acc)
{
    const size_t o = (size_t)row * g.ldc + n;
    float v = g.alpha * acc;
    if (EPI == EPI_STORE) {
        if (g.beta != 0.0f) v += g.beta * g.C[o];
        g.C[o] = v;
    } else if (EPI == EPI_RELU_BACK) {
        v = bf2f(g.H[o]) > 0.0f ? v : 0.0f;
        g.C[o] = v;
        g.Cb[o] = f2bf(v);
    } else {
        v += g.bias[n];
        if (EPI == EPI_BIAS_RELU_BF16) {
            v = v > 0.0f ? v : 0.0f;
            g.Cb[o] = f2bf(v);
        }
        g.C[o] = v;
    }
}

// 64 x 64 outputs per block, one 32 x 32 tile a wave, K in steps of 32 through LDS
// (both operands as [row][k], so that a lane's four k values are one 8-byte read)
// with the next step's loads in flight.  Each output is one chain of MFMAs in
// ascending k.  Loading every operand value from memory as the wave needed it took
// 38 us for the 4096 x 256 x 464 layer and 24 us for the 4096 x 256 x 256 one.
constexpr int TM = 64, TN = 64, BK = 32;
constexpr int LDK = BK + 4;   // 72-byte rows: 8-byte aligned, bank-spread

// Eight operand values of one thread of the tile load: rows r of op (a row of
// the tile, k contiguous) or, for a transposed source, one k and eight rows.
struct Frag8 {
    unsigned short v[8];
};

template <bool T>
__device__ __forceinline__ Frag8 load8(const unsigned short* X, int ld, int R, int K, int r0, int k0, int t, bool vec)
{
    Frag8 f;
    if (!T) {
        const int r = r0 + t / 4, k = k0 + (t % 4) * 8;
        const unsigned short* p = X + (size_t)r * ld + k;
        if (vec && r < R && k + 8 <= K) {
            *(uint4*)f.v = *(const uint4*)p;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) f.v[j] = (r < R && k + j < K) ? p[j] : (unsigned short)0;
        }
    } else {
        const int k = k0 + t / 8, r = r0 + (t % 8) * 8;
        const unsigned short* p = X + (size_t)k * ld + r;
        if (vec && k < K && r + 8 <= R) {
            *(uint4*)f.v = *(const uint4*)p;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) f.v[j] = (k < K && r + j < R) ? p[j] : (unsigned short)0;
        }
    }
    return f;
}

template <bool T> __device__ __forceinline__ void stage8(unsigned short* S, const Frag8& f, int t)
{
    if (!T) {
        unsigned short* p = S + (t / 4) * LDK + (t % 4) * 8;
        ((uint2*)p)[0] = ((const uint2*)f.v)[0];
        ((uint2*)p)[1] = ((const uint2*)f.v)[1];
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) S[((t % 8) * 8 + j) * LDK + t / 8] = f.v[j];
    }
}

template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(GemmArgs g)
{
    __shared__ __align__(16) unsigned short As[TM * LDK];
    __shared__ __align__(16) unsigned short Bs[TN * LDK];
    const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
    const int tiles_n = (g.N + TN - 1) / TN;
    const int row0 = (int)(blockIdx.x / tiles_n) * TM, col0 = (int)(blockIdx.x % tiles_n) * TN;
    const int r = lane & 31, kq = lane >> 5;
    const int mw = (w >> 1) * 32, nw = (w & 1) * 32;
    // 16-byte loads where every tile row starts on 16 bytes
    const bool va = ((uintptr_t)g.A & 15) == 0 && (g.lda & 7) == 0;
    const bool vb = ((uintptr_t)g.B & 15) == 0 && (g.ldb & 7) == 0;
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    Frag8 fa = load8<TA>(g.A, g.lda, g.M, g.K, row0, 0, t, va);
    Frag8 fb = load8<!TB>(g.B, g.ldb, g.N, g.K, col0, 0, t, vb);
    for (int k0 = 0; k0 < g.K; k0 += BK) {
        stage8<TA>(As, fa, t);
        stage8<!TB>(Bs, fb, t);
        __syncthreads();
        if (k0 + BK < g.K) {
            fa = load8<TA>(g.A, g.lda, g.M, g.K, row0, k0 + BK, t, va);
            fb = load8<!TB>(g.B, g.ldb, g.N, g.K, col0, k0 + BK, t, vb);
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 8) {
            const bf16x4 a = *(const bf16x4*)(As + (mw + r) * LDK + kk + 4 * kq);
            const bf16x4 b = *(const bf16x4*)(Bs + (nw + r) * LDK + kk + 4 * kq);
            acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    const int n = col0 + nw + r;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = row0 + mw + acc_row(i, kq);
        if (row < g.M && n < g.N) store_out<EPI>(g, row, n, acc[i]);
    }
}

// Weight gradients (few outputs, K = the batch): one 32 x 32 tile a block, its 16
// waves each take a sixteenth of K, straight from memory, and the block adds the
// partial tiles in wave order.  One wave per tile left the 464 x 256 x 4096
// gradient on 120 waves and 512 dependent steps: 252 us.
constexpr int SPLIT_WAVES = 16;

template <bool TA, bool TB>
__global__ __launch_bounds__(64 * SPLIT_WAVES) void gemm_bf16_splitk_kernel(GemmArgs g)
{
    __shared__ float red[SPLIT_WAVES][16 * 64];
    const int t = (int)threadIdx.x, lane = t & 63, w = t >> 6;
    const int tiles_n = (g.N + 31) / 32;
    const int row0 = (int)(blockIdx.x / tiles_n) * 32, col0 = (int)(blockIdx.x % tiles_n) * 32;
    const int r = lane & 31, kq = lane >> 5;
    const int m = row0 + r, n = col0 + r;
    const int steps = (g.K + 7) / 8;
    const int s0 = (int)((int64_t)steps * w / SPLIT_WAVES), s1 = (int)((int64_t)steps * (w + 1) / SPLIT_WAVES);
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll 4
    for (int s = s0; s < s1; ++s) {
        bf16x4 a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = 8 * s + 4 * kq + j;
            unsigned short av = 0, bv = 0;
            if (m < g.M && k < g.K) av = TA ? g.A[(size_t)k * g.lda + m] : g.A[(size_t)m * g.lda + k];
            if (n < g.N && k < g.K) bv = TB ? g.B[(size_t)n * g.ldb + k] : g.B[(size_t)k * g.ldb + n];
            a[j] = (short)av;
            b[j] = (short)bv;
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) red[w][i * 64 + lane] = acc[i];
    __syncthreads();
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < SPLIT_WAVES; ++k) v += red[k][t];
    const int row = row0 + acc_row(w, kq);
    if (row < g.M && n < g.N) store_out<EPI_STORE>(g, row, n, v);
}

// elementwise operations
__global__ void to_bf16_kernel(const float* x, unsigned short* y, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// dZ = dH * [H > 0] (ReLU backward), as BF16 for the next GEMMs
__global__ void relu_back_kernel(const float* dH, const unsigned short* H, unsigned short* dZb, float* dZ, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = bf2f(H[i]) > 0.0f ? dH[i] : 0.0f;
    dZ[i] = v;
    dZb[i] = f2bf(v);
}

// weighted squared error: loss_i = w_r (Y - T)^2, dY = 2 w_r (Y - T) * scale, with the
// per-row weight w_r (0 for padding rows and masked columns via the mask).  MEAN:
// scale = 1 / max(sum_r w_r, 1), summed by every block.  One atomic a block (one
// an element, on one address, took 187 us for 4096 x 225).
template <bool MEAN>
__global__ __launch_bounds__(256) void mse_kernel(const float* Y, const float* T, const float* rw, const float* cmask,
                                                  int rows, int cols, float scale, float* dY, unsigned short* dYb,
                                                  float* loss)
{
    __shared__ float part[4];
    const int lane = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
    if (MEAN) {
        float s = 0.0f;
        for (int r = threadIdx.x; r < rows; r += 256) s += rw[r];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) part[w] = s;
        __syncthreads();
        s = (part[0] + part[1]) + (part[2] + part[3]);
        scale = (float)(1.0 / fmax((double)s, 1.0));
        __syncthreads();
    }
    float sum = 0.0f;
    const int64_t n = (int64_t)rows * cols, step = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
        const int rr = (int)(i / cols), cc = (int)(i - (int64_t)rr * cols);
        const float wt = rw[rr] * cmask[cc];
        const float d = Y[i] - T[i];
        const float gval = 2.0f * wt * d * scale;
        dY[i] = gval;
        dYb[i] = f2bf(gval);
        sum += wt * d * d * scale;
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) part[w] = sum;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss, (part[0] + part[1]) + (part[2] + part[3]));
}

// column sums of an FP32 rows x cols matrix (bias gradients): a block takes 16
// columns at a time, its 64 thread rows every 64th row, added in a fixed order.  One
// thread a column took 930 us for 4096 x 256.  At most COLSUM_BLOCKS blocks walk the
// columns (a grid holds below 2^32 threads, 67 million columns).
constexpr unsigned COLSUM_BLOCKS = 1u << 16;
__global__ __launch_bounds__(1024) void colsum_kernel(const float* X, int rows, int cols, float* out)
{
    __shared__ float red[64][17];
    const int c = (int)threadIdx.x & 15, q = (int)threadIdx.x >> 4;
    for (int64_t c0 = (int64_t)blockIdx.x * 16; c0 < cols; c0 += (int64_t)gridDim.x * 16) {
        const int64_t col = c0 + c;
        float s = 0.0f;
        if (col < cols) {
#pragma unroll 8
            for (int r = q; r < rows; r += 64) s += X[(size_t)r * cols + col];
        }
        __syncthreads();    // the last columns' sums are read
        red[q][c] = s;
        for (int h = 32; h > 0; h >>= 1) {
            __syncthreads();
            if (q < h) red[q][c] += red[q + h][c];
        }
        if (q == 0 && col < cols) out[col] = red[0][c];
    }
}

// The same for few rows, one thread a column: 5 x 20000 14.7 us against 15.9, 16 x 225
// 14.3 against 14.4, 100 x 256 21.2 against 14.5.
constexpr int COLSUM_FEW = 16;
__global__ __launch_bounds__(256) void colsum_few_kernel(const float* X, int rows, int cols, float* out)
{
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (c >= cols) return;
    float s = 0.0f;
    for (int r = 0; r < rows; ++r) s += X[(size_t)r * cols + c];
    out[c] = s;
}

// Adam (Kingma & Ba, 2015) on FP32 master weights; writes the BF16 copy
__device__ __forceinline__ void adam_one(float* w, float* mo, float* ve, const float* gr, unsigned short* wb, int64_t i,
                                         float lr, float b1, float b2, float eps, float c1, float c2)
{
    const float gi = gr[i];
    const float m1 = b1 * mo[i] + (1.0f - b1) * gi;
    const float v1 = b2 * ve[i] + (1.0f - b2) * gi * gi;
    mo[i] = m1;
    ve[i] = v1;
    const float wi = w[i] - lr * (m1 / c1) / (sqrtf(v1 / c2) + eps);
    w[i] = wi;
    if (wb) wb[i] = f2bf(wi);
}

// Adam over several tensors in one launch: tensor t owns the blocks from first[t]
constexpr int ADAM_MAX = 16;
struct AdamArgs {
    float *w[ADAM_MAX], *mo[ADAM_MAX], *ve[ADAM_MAX];
    const float* gr[ADAM_MAX];
    unsigned short* wb[ADAM_MAX];
    int64_t n[ADAM_MAX];
    unsigned first[ADAM_MAX + 1];
    int count;
    float lr, b1, b2, eps, c1, c2;
};

// ONE: a single tensor, whose pointers need no search (25.6 million parameters: 132 us
// with it, 127 without)
template <bool ONE> __global__ __launch_bounds__(256) void adam_multi_kernel(AdamArgs a)
{
    int t = 0;
    if (!ONE)
        while (t + 1 < a.count && blockIdx.x >= a.first[t + 1]) ++t;
    const int64_t i = (int64_t)(blockIdx.x - a.first[t]) * 256 + threadIdx.x;
    if (i < a.n[t])
        adam_one(a.w[t], a.mo[t], a.ve[t], a.gr[t], a.wb[t], i, a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
}

unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }
unsigned mse_blocks(int64_t n) { return (unsigned)(n > 256 * 512 ? 512 : (n + 255) / 256); }

}  // namespace

extern "C" {

int qbx_gemm_bf16(int32_t trans_a, int32_t trans_b, int32_t M, int32_t N, int32_t K, float alpha, const void* A,
                  int32_t lda, const void* B, int32_t ldb, float beta, float* C, int32_t ldc, int32_t epilogue,
                  const float* bias, void* Cb, void* stream)
{
    return qbx::guarded([&] {
        if (M < 0 || N < 0 || K < 0) throw qbx::QbxError(QBX_EINVAL, "negative GEMM size");
        if (!A || !B || !C) throw qbx::QbxError(QBX_EINVAL, "null GEMM operand");
        if (epilogue < 0 || epilogue > 2) throw qbx::QbxError(QBX_EINVAL, "unknown GEMM epilogue");
        if (epilogue != EPI_STORE && !bias) throw qbx::QbxError(QBX_EINVAL, "the epilogue needs a bias");
        if (epilogue == EPI_BIAS_RELU_BF16 && !Cb) throw qbx::QbxError(QBX_EINVAL, "the epilogue needs a BF16 output");
        if ((trans_a ? lda < M : lda < K) || (trans_b ? ldb < K : ldb < N) || ldc < N)
            throw qbx::QbxError(QBX_EINVAL, "leading dimension too small");
        if (M == 0 || N == 0) return;
        GemmArgs g{};
        g.A = (const unsigned short*)A;
        g.B = (const unsigned short*)B;
        g.C = C;
        g.bias = bias;
        g.Cb = (unsigned short*)Cb;
        g.M = M;
        g.N = N;
        g.K = K;
        g.lda = lda;
        g.ldb = ldb;
        g.ldc = ldc;
        g.alpha = alpha;
        g.beta = beta;
        if (epilogue != EPI_STORE && (trans_a || trans_b))
            throw qbx::QbxError(QBX_EUNSUP, "bias epilogues take untransposed operands");
        const int64_t blocks = (int64_t)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
        const int64_t tiles = (int64_t)((M + 31) / 32) * ((N + 31) / 32);
        if (blocks > 0x7fffffffLL) throw qbx::QbxError(QBX_EUNSUP, "GEMM too large for one grid");
        hipStream_t st = (hipStream_t)stream;
        // K split over the waves of a block where the 64 x 64 tiles would occupy
        // under half of the CUs and each wave still gets 32 or more k: 464 x 256 x
        // 4096 (32 blocks) 252 -> 17 us.  Shorter K, or more tiles, keep one chain
        // of MFMAs per output.
        if (epilogue == EPI_STORE && blocks < 128 && K >= 32 * SPLIT_WAVES) {
            const dim3 grid((unsigned)tiles), block(64 * SPLIT_WAVES);
            auto launch = [&](void (*kern)(GemmArgs)) { hipLaunchKernelGGL(kern, grid, block, 0, st, g); };
            if (!trans_a && !trans_b) launch(gemm_bf16_splitk_kernel<false, false>);
            else if (trans_a && !trans_b) launch(gemm_bf16_splitk_kernel<true, false>);
            else if (!trans_a && trans_b) launch(gemm_bf16_splitk_kernel<false, true>);
            else launch(gemm_bf16_splitk_kernel<true, true>);
        } else {
            const dim3 grid((unsigned)blocks), block(256);
            auto launch = [&](void (*kern)(GemmArgs)) { hipLaunchKernelGGL(kern, grid, block, 0, st, g); };
            if (epilogue == EPI_BIAS_RELU_BF16) launch(gemm_bf16_kernel<false, false, EPI_BIAS_RELU_BF16>);
            else if (epilogue == EPI_BIAS) launch(gemm_bf16_kernel<false, false, EPI_BIAS>);
            else if (!trans_a && !trans_b) launch(gemm_bf16_kernel<false, false, EPI_STORE>);
            else if (trans_a && !trans_b) launch(gemm_bf16_kernel<true, false, EPI_STORE>);
            else if (!trans_a && trans_b) launch(gemm_bf16_kernel<false, true, EPI_STORE>);
            else launch(gemm_bf16_kernel<true, true, EPI_STORE>);
        }
        QBX_HIP(hipGetLastError());
    });
}

int qbx_gemm_bf16_relu_back(int32_t M, int32_t N, int32_t K, const void* A, int32_t lda, const void* B, int32_t ldb,
                            const void* H, float* C, void* Cb, int32_t ldc, void* stream)
{
    return qbx::guarded([&] {
        if (M < 0 || N < 0 || K < 0) throw qbx::QbxError(QBX_EINVAL, "negative GEMM size");
        if (!A || !B || !H || !C || !Cb) throw qbx::QbxError(QBX_EINVAL, "null GEMM operand");
        if (lda < K || ldb < K || ldc < N) throw qbx::QbxError(QBX_EINVAL, "leading dimension too small");
        if (M == 0 || N == 0) return;
        GemmArgs g{};
        g.A = (const unsigned short*)A;
        g.B = (const unsigned short*)B;
        g.H = (const unsigned short*)H;
        g.C = C;
        g.Cb = (unsigned short*)Cb;
        g.M = M;
        g.N = N;
        g.K = K;
        g.lda = lda;
        g.ldb = ldb;
        g.ldc = ldc;
        g.alpha = 1.0f;
        const int64_t blocks = (int64_t)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
        if (blocks > 0x7fffffffLL) throw qbx::QbxError(QBX_EUNSUP, "GEMM too large for one grid");
        hipLaunchKernelGGL((gemm_bf16_kernel<false, true, EPI_RELU_BACK>), dim3((unsigned)blocks), dim3(256), 0,
                           (hipStream_t)stream, g);
        QBX_HIP(hipGetLastError());
    });
}

int qbx_mlp_elementwise(int32_t op, int64_t n, const void* x, const void* y, void* out0, void* out1, void* stream)
{
    // op 0: out0(bf16) = bf16(x f32)
    // op 1: ReLU backward: x = dH (f32), y = H (bf16) -> out1 = dZ (f32), out0 = dZ (bf16)
    return qbx::guarded([&] {
        if (n < 0) throw qbx::QbxError(QBX_EINVAL, "negative size");
        if (n == 0) return;
        hipStream_t st = (hipStream_t)stream;
        if (op == 0) {
            hipLaunchKernelGGL(to_bf16_kernel, dim3(blocks_for(n)), dim3(256), 0, st, (const float*)x,
                               (unsigned short*)out0, n);
        } else if (op == 1) {
            hipLaunchKernelGGL(relu_back_kernel, dim3(blocks_for(n)), dim3(256), 0, st, (const float*)x,
                               (const unsigned short*)y, (unsigned short*)out0, (float*)out1, n);
        } else {
            throw qbx::QbxError(QBX_EINVAL, "unknown elementwise op");
        }
        QBX_HIP(hipGetLastError());
    });
}

int qbx_mlp_mse(int32_t rows, int32_t cols, const float* Y, const float* T, const float* row_w, const float* col_mask,
                float scale, float* dY, void* dYb, float* loss, void* stream)
{
    return qbx::guarded([&] {
        if (rows < 0 || cols < 0) throw qbx::QbxError(QBX_EINVAL, "negative size");
        const int64_t n = (int64_t)rows * cols;
        if (n == 0) return;
        hipLaunchKernelGGL(mse_kernel<false>, dim3(mse_blocks(n)), dim3(256), 0, (hipStream_t)stream, Y, T, row_w,
                           col_mask, rows, cols, scale, dY, (unsigned short*)dYb, loss);
        QBX_HIP(hipGetLastError());
    });
}

int qbx_mlp_mse_mean(int32_t rows, int32_t cols, const float* Y, const float* T, const float* row_w,
                     const float* col_mask, float* dY, void* dYb, float* loss, void* stream)
{
    return qbx::guarded([&] {
        if (rows < 0 || cols < 0) throw qbx::QbxError(QBX_EINVAL, "negative size");
        if (!Y || !T || !row_w || !col_mask || !dY || !dYb || !loss) throw qbx::QbxError(QBX_EINVAL, "null argument");
        const int64_t n = (int64_t)rows * cols;
        if (n == 0) return;
        hipLaunchKernelGGL(mse_kernel<true>, dim3(mse_blocks(n)), dim3(256), 0, (hipStream_t)stream, Y, T, row_w,
                           col_mask, rows, cols, 0.0f, dY, (unsigned short*)dYb, loss);
        QBX_HIP(hipGetLastError());
    });
}

int qbx_mlp_colsum(int32_t rows, int32_t cols, const float* X, float* out, void* stream)
{
    return qbx::guarded([&] {
        if (rows < 0 || cols < 0) throw qbx::QbxError(QBX_EINVAL, "negative size");
        if (cols == 0) return;
        const unsigned blocks = (unsigned)(((int64_t)cols + 15) / 16);
        if (rows <= COLSUM_FEW)
            hipLaunchKernelGGL(colsum_few_kernel, dim3(blocks_for(cols)), dim3(256), 0, (hipStream_t)stream, X, rows,
                               cols, out);
        else
            hipLaunchKernelGGL(colsum_kernel, dim3(blocks < COLSUM_BLOCKS ? blocks : COLSUM_BLOCKS), dim3(1024), 0,
                               (hipStream_t)stream, X, rows, cols, out);
        QBX_HIP(hipGetLastError());
    });
}

int qbx_mlp_adam(int64_t n, float* w, float* m, float* v, const float* g, void* wb, float lr, float b1, float b2,
                 float eps, int32_t step, void* stream)
{
    float* const ws[1] = {w};
    float* const ms[1] = {m};
    float* const vs[1] = {v};
    const float* const gs[1] = {g};
    void* const wbs[1] = {wb};
    return qbx_mlp_adam_multi(1, &n, ws, ms, vs, gs, wbs, lr, b1, b2, eps, step, stream);
}

int qbx_mlp_adam_multi(int32_t count, const int64_t* n, float* const* w, float* const* m, float* const* v,
                       const float* const* g, void* const* wb, float lr, float b1, float b2, float eps, int32_t step,
                       void* stream)
{
    return qbx::guarded([&] {
        if (step < 1) throw qbx::QbxError(QBX_EINVAL, "bad Adam arguments");
        if (count < 1 || count > ADAM_MAX) throw qbx::QbxError(QBX_EINVAL, "Adam takes 1 to 16 tensors a call");
        if (!n || !w || !m || !v || !g || !wb) throw qbx::QbxError(QBX_EINVAL, "null Adam array");
        AdamArgs a{};
        int64_t blocks = 0;
        for (int t = 0; t < count; ++t) {
            if (n[t] < 0) throw qbx::QbxError(QBX_EINVAL, "bad Adam arguments");
            a.w[t] = w[t];
            a.mo[t] = m[t];
            a.ve[t] = v[t];
            a.gr[t] = g[t];
            a.wb[t] = (unsigned short*)wb[t];
            a.n[t] = n[t];
            a.first[t] = (unsigned)blocks;
            blocks += (n[t] + 255) / 256;
            if (blocks > 0x7fffffffLL) throw qbx::QbxError(QBX_EUNSUP, "Adam tensors too large for one grid");
        }
        if (blocks == 0) return;
        a.first[count] = (unsigned)blocks;
        a.count = count;
        a.lr = lr;
        a.b1 = b1;
        a.b2 = b2;
        a.eps = eps;
        a.c1 = 1.0f - powf(b1, (float)step);
        a.c2 = 1.0f - powf(b2, (float)step);
        hipLaunchKernelGGL(count == 1 ? adam_multi_kernel<true> : adam_multi_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
        QBX_HIP(hipGetLastError());
    });
}

}  // extern "C"
