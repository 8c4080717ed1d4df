// qbx_eri_api.h -- argument block and launcher declaration of the ERI kernels.
#pragma once
#include "qbx_device.h"
#include <hip/hip_runtime.h>
#include <cstdint>

namespace qbx {
enum EriMode { MODE_JK = 0, MODE_DENSE = 1, MODE_SCHWARZ = 2 };

// J/K kernel with the bra's K rows in LDS: ROW_WAVES waves per block, at most
// ROW_LDS_MAX bytes of rows (larger bases use the one-wave-per-chunk kernel).
#ifndef QBX_ROW_WAVES
#define QBX_ROW_WAVES 4
#endif
constexpr int ROW_WAVES = QBX_ROW_WAVES;
// One K-row task (one block): items item0 .. item1 - 1 of bra `list`.  Item j is the 64-ket chunk chunk0 + j / (kparts bparts)
// with one of kparts parts of every ket's primitive pairs and one of bparts parts
// of the bra's: the digest is linear in the integrals, so the waves that share a
// heavy chunk each digest the integrals of their own primitive quartets.
struct RowTask {
    int list, chunk0, kparts, bparts, item0, item1;
};
// Most items per task of the low-L K-row kernels, and of the staged
// K-row kernel (whose waves are long, so that smaller tasks balance better).
// Fewer and larger tasks flush fewer K rows: with chunks alone as items, 24 H2O
// in cc-pVDZ took 50.9 ms per build at 16 and 49.6 at 32, the 592-function
// cluster lost at 64 (38.6 -> 39.4 ms), and its (dp|pp) took 5.05 ms at 16 and
// 4.33 at 8.
constexpr int ROW_ITEMS = 32;
constexpr int STAGED_ROW_ITEMS = 8;
constexpr int ROW_LDS_MAX = 64 * 1024;
struct PairClassDev {
    int n;
    const int* shA;
    const int* shB;
    const int* ppo;
    const int* ppn;
    const double* AB;
    const double* Q;    // Schwarz bound per pair (sorted descending)
};

struct EriArgs {
    PairClassDev bra, ket;
    const PrimPair* pp;
    const DevShell* sh;
    const double* boys;
    const double* bexp;
    const double* boysl;      // per-order Boys rows of the class's total L
    const int* klist;         // [nbra][2 nbk + 1]: ket lists of the bras (KetList)
    const int* cpre;          // [nbra+1] prefix over bras of ceil(kets / 64): waves
    const RowTask* rtask;     // K-row tasks of the bras (null: the one-wave-per-chunk kernels run)
    int nsuper;               // their number
    int nbk;                  // ket buckets of the class
    int lds_max;              // LDS bytes a block may use on this device
    int64_t total;            // Schwarz mode: number of diagonal pairs
    int nwave;                // J/K and dense modes: number of waves
    int nbra;
    int same;
    const double* D;   // [2*nset][N][N]: DJ sets then DK sets
    double* J;         // [copies][nset][N][N]
    double* K;
    // xcd_local: each XCD accumulates into its own copy of J and K (copy =
    // the XCC_ID of the wave, stride jk_stride doubles) with workgroup-scope
    // atomics, which the XCD's L2 resolves; otherwise one copy, device scope
    int xcd_local;
    size_t jk_stride;
    // ket sums J_cd in pair order (null: straight to J): the ket class's block
    // [component cd][pair], per density set (stride jp_set) and copy (jp_stride)
    double* jp;
    size_t jp_set, jp_stride;
    int nset;
    int N;
    double* eri;       // dense mode, N^4
    double* qout;      // Schwarz mode, per bra pair
    // density screening (J/K mode): skip quartets with Q_ab Q_cd max|D| < dthr,
    // max|D| over the six shell-pair blocks that the quartet reads
    const double* pdmax;  // [n_shell][n_shell], NULL: off
    int nshell;
    double dthr;
    void* scratch_stream;  // main stream: kernels with scratch are launched there
    // staged classes: workspace of ws_slots wave slots, each
    // EriClass::NE * NCD * 64 values of the kernel's arithmetic type
    void* ws;
    int ws_slots;
    int split;                // classes with Cls::SPLIT > 1: share each wave task among SPLIT waves (0: off)
    // gradient kernels: radial indices (k_a | k_b << 16) of every primitive pair,
    // first radial primitive of every shell, and the outputs: per radial
    // primitive dE/d(exponent) and c dE/dc, per shell dE/d(centre)
    const int* ppk;
    const int* shell_poff;
    int n_radial;             // radial primitives (length of g_xpn and g_lin)
    int grad_lds;             // doubles of a block's LDS copy of the three outputs (0: none)
    double* g_xpn;
    double* g_lin;
    double* g_cen;
};


// Defined (explicitly instantiated) in the generated per-class translation units.
template <int LA, int LB, int LC, int LD, typename R, int MODE>
void launch_eri(const EriArgs& a, hipStream_t s);

// Gradient kernels (classes whose shells are all s or p), generated units
// eri_<class>_grad.hip: group g of a class goes to stream s[g % ns].
template <int LA, int LB, int LC, int LD>
void launch_eri_grad(const EriArgs& a, hipStream_t* s, int ns);
typedef void (*EriGradLaunch)(const EriArgs&, hipStream_t*, int);

typedef void (*EriLaunch)(const EriArgs&, hipStream_t);

// Shell quartets with a shell above the generated classes (f and g): the
// generic kernel of qbx_eri_generic.hip, one launch per pair of pair classes
// (bra (l0 l1), ket (l2 l3)).  Both classes are in descending Schwarz order; the
// kets of bra i are the first prefix[i + 1] - prefix[i] of the ket class.  One
// block per shell quartet.
struct GenArgs {
    PairClassDev bra, ket;
    const DevShell* sh;
    const PrimPair* pp;
    const double* boys;       // one-electron Boys table (F_0..F_32 on the 0.1 grid)
    const double* bexp;
    int l[4];
    int bn_max, kn_max;       // largest primitive-pair counts of the two classes
    int ub, cdc;              // bra primitive pairs and ket components held at a time (set by the launcher)
    int nbra;
    int same;                 // bra and ket are one class
    int64_t total;            // quartets (blocks)
    int64_t first;            // this launch's first one (set by the launcher)
    const int64_t* prefix;    // [nbra + 1]
    int N;
    // J/K mode (as EriArgs)
    const double* D;
    double* J;
    double* K;
    int xcd_local;
    size_t jk_stride;
    int nset;
    const double* pdmax;
    int nshell;
    double dthr;
    // dense mode
    double* eri;
    // Schwarz mode: every bra with itself, sqrt(max |(ab|ab)|)
    double* qout;
};

// mode: MODE_JK, MODE_DENSE or MODE_SCHWARZ
void launch_eri_generic(const GenArgs& a, int mode, hipStream_t s);

// Primitive-quartet ERIs with unit coefficients (qbx_eri_generic.hip), one
// thread each: cen [n][4][3], xpn [n][4], ang [n][4][3] (order a, b, c, d of
// (ab|cd)), total angular momentum at most QBX_PRIM_ERI_LTOT.
#define QBX_PRIM_ERI_LTOT 24
void prim_eri(int n, const double* cen, const double* xpn, const int* ang, const double* boys, const double* bexp,
              double* out, hipStream_t s);

// The ERI kernels' Boys function alone (qbx_boys_probe.hip): F_0..F_L at n
// device arguments T from the order-L table rows, into F (n x (L+1)).
void boys_probe(const double* rows, int L, const double* T, int n, double* F, hipStream_t s);
}  // namespace qbx
