// qbx_one_e.h -- nuclear attraction and the one-electron energy gradient by
// pair class (qbx_one_e.hip).
#pragma once
#include "qbx_eri_api.h"

namespace qbx {

// One pair class (la >= lb) of a basis and the point charges.
struct NucArgs {
    PairClassDev pairs;
    const PrimPair* pp;
    const DevShell* sh;
    const double* boysl;   // Boys rows of order la + lb (la + lb + 2 for the gradient)
    int N;
    int nnuc;
    const double* Z;
    const double* R;
    double* out;           // N x N
    // gradient: densities, radial indices of every primitive pair, first radial
    // primitive of every shell, outputs as in EriArgs
    const double* Dt;
    const double* W;
    const int* ppk;
    const int* poff;
    double* g_xpn;
    double* g_lin;
    double* g_cen;
};

// out[i][j] = out[j][i] = -sum_n Z_n <i| 1/|r - R_n| |j> over the class's pairs
void launch_nuclear(int la, int lb, const NucArgs& a, hipStream_t s);

// dE/d(exponent), c dE/dc and dE/d(centre) of sum D (T + V) - W S over the
// class's pairs (s and p shells)
void launch_one_e_grad(int la, int lb, const NucArgs& a, hipStream_t s);

}  // namespace qbx
