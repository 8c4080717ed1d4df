// Dense FP64 linear algebra on the device for the SCF step: a GEMM on the
// FP64 matrix cores and the pieces of trace-correcting purification.
// Row-major matrices, device pointers, launches on the given stream.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace qbx {

// C = alpha * op(A) op(B) + beta * Z   (op = transpose when the flag is set;
// op(A) is M x K, op(B) is K x N; Z may be C itself, or null when beta == 0)
void gemm_f64(bool trans_a, bool trans_b, int M, int N, int K, double alpha, const double* A, int lda,
              const double* B, int ldb, double beta, const double* Z, int ldz, double* C, int ldc, hipStream_t s);

// out[(a nao + b) nmo + m] = C[a][m] C[b][m] for the nao x nmo matrix C
void pair_columns(const double* C, int nao, int nmo, double* out, hipStream_t s);

// Gershgorin interval of each row of the symmetric n x n matrix P:
// lohi[2i] = P_ii - sum_j!=i |P_ij|, lohi[2i+1] = P_ii + sum_j!=i |P_ij|
void gershgorin(const double* P, int n, double* lohi, hipStream_t s);

// P <- (P + P^T) / 2 for the n x n matrix P
void symmetrize_square(double* P, int n, hipStream_t s);

// flip the columns j of the n x n matrix C whose first-row entry C[0][j] is
// negative (sgn: n doubles of work space)
void fix_column_signs(double* C, int n, double* sgn, hipStream_t s);

// out[0] = min of lohi[2i], out[1] = max of lohi[2i+1] over the n rows
void spectral_interval(const double* lohi, int n, double* out, hipStream_t s);

// Trace-correcting purification on the device.  Matrices are symmetric,
// sp2_padded(n) square with zero rows and columns beyond n; `shares` holds 2 x 2 x
// sp2_blocks(n) doubles, `state` two entries.
struct Sp2State {
    int tail;   // products still to make once the projector has settled, -1: not settled
    int stop;   // no product any more
    int it;     // products made
    int pad;
};
struct Sp2Status {
    Sp2State s;
    double tr, fr;   // tr P and |P|_F^2 of the latest matrix
};
int sp2_padded(int n);
int sp2_blocks(int n);

// P = (hi I - F) / (hi - lo), F's symmetric part (n x n, row stride n), [lo, hi] =
// lohi (hi = lo + 1 where the interval is empty); state[0] and shares of P
void sp2_start(const double* F, int n, const double* lohi, double* P, double* shares, Sp2State* state, hipStream_t s);

// Product k (0, 1, ...): Q = P^2 or 2P - P^2, whichever moves tr P toward nocc, or
// nothing after the projector has settled.  Matrix k is in the first buffer for
// even k, in the second for odd k.
void sp2_product(const double* P, double* Q, int n, int nocc, int k, double* shares, Sp2State* state, hipStream_t s);

// state and measures after k launches of sp2_product
void sp2_status(const double* shares, int n, int k, const Sp2State* state, Sp2Status* out, hipStream_t s);

// Launch of the tridiagonalization of order n on the current device; no blocks where
// the matrix does not fit the device's LDS or the device cannot run the whole grid at
// once (above order 1850 with 256 CUs and 160 KB of LDS).
struct TridiagPlan {
    int n = 0, blocks = 0, threads = 0;
    size_t shm = 0;
};
TridiagPlan tridiag_plan(int n);

// Householder tridiagonalization of the symmetric n x n matrix A (LAPACK's lower
// form): diagonal d (n), off-diagonal e (n - 1), reflector k (its first entry, 1,
// left out) in V[k n + k + 2 ...], factors tau (n - 1).  exchange: tridiag_exchange(n)
// values of work space.  false where nothing was launched (no blocks, or the launch
// was refused).  *status (device) is 0, or 1 when a block gave up waiting for
// another after `spins` more polls of a value: the outputs are partly unwritten then.
constexpr int TRI_SPINS = 1 << 20;
size_t tridiag_exchange(int n);
bool tridiagonalize(const TridiagPlan& plan, const double* A, double* V, double* d, double* e, double* tau,
                    uint64_t* exchange, int* status, int spins, hipStream_t s);

// The tridiagonal matrix times a power of two, its largest entry in [1, 2) (the
// divide and conquer solver drops what is small in absolute terms), and the
// eigenvalues d brought back; back: one double of device memory.  Where *status is not 0
// the matrix and the factors tau become zero.
void tridiag_scale(int n, double* d, double* e, double* tau, const int* status, double* back, hipStream_t s);
void tridiag_unscale(int n, double* d, const double* back, hipStream_t s);

}  // namespace qbx
