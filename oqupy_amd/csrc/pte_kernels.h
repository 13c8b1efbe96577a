// Argument blocks and kernel declarations of the process-tensor engine.
#pragma once

#include <hip/hip_runtime.h>

#include "pte_post.h"

namespace pte {

enum NodeKind { NODE_DENSE = 0, NODE_DELTA = 1 };
enum MpoOut { MPO_OUT_SVD_H = 0, MPO_OUT_SITE = 1, MPO_OUT_M = 2 };

struct GemmArgs {
  int M, N, K;
  const double2* A; long sai, sak;
  const double2* B; long sbk, sbj;
  double2* C; long sci, scj;
  int conjA, conjB;
  double2 alpha;
  int beta_zero;
};

struct MpoApplyArgs {
  const double2* G;   // GEMM result
  const double2* W;   // dense node [w][p][s][v]
  const double2* I;   // delta node weights [w][p]
  int kind, mode;
  int Dl, P, Dx, V, Wl, S;
  double2* out;
  long ldx;
};

// Summary of one truncated SVD, written by the device.
struct SvdInfo {
  int rank;        // kept singular values
  int overflow;    // rank above the bond capacity
  int sweeps;      // Jacobi sweeps (or -1 if not converged)
  int pad;
  double s0;       // largest singular value
  double discarded;  // 2-norm of the discarded singular values
  int rounds;      // rotation rounds logged (Gram Jacobi)
  int state;       // of a Gram Jacobi (see GramState)
};

// States of a Gram Jacobi (gram_svd_kernel). While it is not done, SvdInfo's
// `sweeps` counts the sweeps so far and `pad` is the rank.
enum GramState {
  kGramDone = 0,      // a freshly formed Gram matrix needed no rotation
  kGramFresh = 1,     // Y is there, no pass was made
  kGramRotated = 2    // a pass rotated: its log is to be replayed, then checked
};

struct JacobiArgs {
  double2* X; int m, n; long ldx;
  double2* V; long ldv;
  int nb;
  int slices;         // workgroups per block pair (row slices)
  int xrows_per;      // rows of X per slice (multiple of 32)
  int vrows_per;      // rows of V per slice (multiple of 32)
  double2* gpart;     // partial Grams [pair][slice][32*32] when slices > 1
  double tol, abs_tol_scale;
  int max_sweeps;
  int inner_sweeps;   // cyclic sweeps of the pair's 2JB x 2JB eigenproblem
  unsigned* bar;
  int* flags;
  double* fro2;
  int* info;
  // skipping of converged pairs (zeroed before the launch): skip[b], b < nb,
  // is 1 + the round in which block b was last rotated (0: never);
  // skip[nb + pair_index(bi, bj)] is 1 + the round in which that block pair
  // was last found to need no rotation (0: not since its last rotation)
  unsigned* skip;
};

struct EmitArgs {
  const double2* src; long lds;
  const int* perm;
  const SvdInfo* info;
  int A, B;
  long dj0, djk, da0, dak, db0, dbk;
  int conj;
  const int* rowmap;   // destination row of source row s (null: identity)
  double2* dst;
};

// Pivoted QR of a column-major matrix (see qrcp_kernel).
struct QrcpArgs {
  double2* A; int m, n; long lda;
  double drop;                // stop when the residual norm <= drop * ||A||_F
  double2* tau; double2* vscale; double* beta;
  int* piv;                   // [n] physical column of each step, then the rest
  int* done;                  // [n] scratch
  unsigned long long* cand;   // posts, zeroed before the launch: [2][gridDim.x][2] words
                              // 0 and 1, then [2][gridDim.x] words 2
  int* rank;                  // steps taken
  const int* max_steps;       // optional cap on the steps (device int)
  double* out;                // optional: [0] squared residual norm at the stop,
                              // [1] ||A||_F^2 (first run), [2] |beta_0|, [3] the
                              // first step count whose residual norm is at most
                              // mark_rel * |beta_0| (the steps taken if none)
  double mark_rel;            // 0: no mark
  int stop_at_mark;           // stop at the mark (adaptive cap)
  int start;                  // > 0: resume a factorisation stopped after `start`
                              // steps (done, piv, tau, vscale, beta kept)
  double drop_abs2;           // stop threshold on the squared residual when resuming
};

struct ApplyQArgs {
  const double2* A; int m; long lda;      // reflectors from qrcp_kernel
  const double2* tau; const double2* vscale; const int* piv; const int* qrank;
  const double2* W; long ldw;             // Jacobi unitary (qrank x qrank)
  const int* perm;
  const SvdInfo* info;
  int B;                                  // row i = a*B + b
  long dj0, djk, da0, dak, db0, dbk;      // strides d0 + dk * rank
  double2* dst;
};

constexpr int kQrcpMaxLocal = 64;         // columns per workgroup in qrcp_kernel

// One SVD's singular values, order and cut (batched post-processing).
struct SvdPostArgs {
  const double2* X; int m, n;               // orthogonalised X (ld = m)
  double* sigma; int* perm; double* sorted;
  SvdInfo* info;
  double epsrel; int max_rank; int pad;
};

// Y = R^H of one pivoted QR (batched).
struct RhArgs {
  const double2* A; long lda; int n; int pad;
  const int* piv; const double* beta; const int* rank;
  double2* Y;
};

// One small truncated SVD (small_svd_kernel): the pivoted QR's outputs
// (reflectors in A, tau, vscale, beta, piv, *qrank), Y = R^H in Y (n x r,
// ld n), info (info->pad = r) and, of ranks up to kGramSmallRank, the first
// pass of the Gram Jacobi with its rotation log.
struct SmallSvdArgs {
  double2* A; int m, n;
  double2* tau; double2* vscale; double* beta; int* piv; int* qrank;
  double2* Y;
  double* sigma; int* perm; double* sorted; SvdInfo* info;
  double epsrel; int max_rank; int max_sweeps;
  SvdInfo* copy;    // optional second copy of the summary (batched gather)
  double stop_rel;  // > 0: stop the QR at residual <= stop_rel * |beta_0|
  double* folded;   // optional: the squared residual of that stop
  long lds_bytes;   // dynamic LDS of the launch (Y goes through it when it fits)
  double* logc; double2* logs;
};

// One pass of the Jacobi SVD of Y (n x r, ld n; R^H of a pivoted QR, or that
// times the rotations so far) on its Gram matrix, in one workgroup
// (gram_svd_kernel): the rotation log (64 rotations per round), or, where none is
// needed, sigma, perm, sorted and the final info. With `expect` (a GramState),
// r is an upper bound: the rank is info->pad, and there is nothing to do unless
// info->state is `expect`.
struct GramSvdArgs {
  const double2* Y; int n, r;
  int expect;               // 0: the first pass, of rank r
  double* sigma; int* perm; double* sorted; SvdInfo* info;
  double epsrel; int max_rank; int max_sweeps;
  SvdInfo* copy;
  const double* extra2;     // optional squared weight counted in every tail
  double* logc; double2* logs;
};

// Y <- Y J in place and W <- W J (r x r, ld r, r = info->pad) with the rotations J
// of the last pass from its log; `first` sets W = J (also where no rotation was
// needed). Else nothing unless info->state is kGramRotated.
struct GramReplayArgs {
  double2* Y; int n;
  int first;
  double2* W;
  const SvdInfo* info;
  const double* logc; const double2* logs;
};

constexpr int kGramMaxRank = 126;           // G in LDS, two blocks of it per thread
constexpr int kGramMaxSweeps = 20;          // sweeps of a pass, all in the rotation log
constexpr int kGramMaxPasses = 6;           // passes, the last one rotating nothing
constexpr int kGramGridRank = 112;          // after the grid's QR: largest rank
constexpr int kGramGridRows = 512;          // and rows of Y (see gram_ok)
constexpr int kSmallMaxCols = kGramMaxRank; // columns of M in small_svd_kernel
constexpr int kSmallThreads = 512;          // its workgroup
constexpr int kGramThreads = 1024;          // workgroup of gram_svd_kernel
// Ranks whose first pass small_svd_kernel does itself: two blocks of G a thread hold
// no more. (A round takes 0.64 us with its 512 threads at rank 35, 0.68 with 1024;
// 0.96 and 0.92 at rank 74, where another launch would cost more than that gives.)
constexpr int kGramSmallRank = 88;
constexpr int kSmallRows = 38;              // rows of M a lane holds at most (no scratch)
constexpr size_t kSmallQrLds = 64 * kSmallRows * 16 + 2048;   // LDS of its QR
// lanes per column of small_svd_kernel's QR
__host__ __device__ constexpr int small_lanes(int n) {
  return n > 64 ? 4 : n > 32 ? 8 : n > 16 ? 16 : n > 8 ? 32 : 64;
}

struct ZeroItem {
  unsigned* p; int words; int pad;
};

__global__ void qrcp_kernel(QrcpArgs a);
__global__ void qrcp_batch_kernel(const QrcpArgs* probs, const int* starts,
                                  const int* block_prob);
__global__ void build_rh_kernel(const double2* A, long lda, int n, const int* piv,
                                const double* beta, const int* rank, double2* Y);
__global__ void build_rh_batch_kernel(const RhArgs* pa);
__global__ void column_norm_batch_kernel(const SvdPostArgs* pa);
__global__ void rank_sort_batch_kernel(const SvdPostArgs* pa);
__global__ void truncate_batch_kernel(const SvdPostArgs* pa, SvdInfo* out);
__global__ void zero_items_kernel(const ZeroItem* items);
__global__ void small_svd_kernel(SmallSvdArgs a);
__global__ void small_svd_batch_kernel(const SmallSvdArgs* probs);
template <int NT>                           // kSmallThreads (ranks up to kGramSmallRank)
__global__ void gram_svd_kernel(GramSvdArgs a);            // or kGramThreads
template <int NT>
__global__ void gram_svd_batch_kernel(const GramSvdArgs* probs);
__global__ void gram_replay_kernel(GramReplayArgs a);
__global__ void gram_replay_batch_kernel(const GramReplayArgs* probs);   // problem = blockIdx.y
__global__ void gather_qr_rank_kernel(const QrcpArgs* probs, int n, int* out);
__global__ void apply_q_kernel(ApplyQArgs a);
template <int RP>
__global__ void apply_q_wave_kernel(ApplyQArgs a);   // Q of at most kApplyQWaveRows rows
constexpr int kApplyQWaveRows = 1024;
__global__ void zgemm_kernel(GemmArgs a);
__global__ void zgemm_mfma_kernel(GemmArgs a);
__global__ void cgemm_mfma_kernel(GemmArgs a);
__global__ void mpo_apply_kernel(MpoApplyArgs a);
__global__ void mpo_apply_right_kernel(MpoApplyArgs a);
__global__ void jacobi_kernel(JacobiArgs a);
// the same with the slice held in an LDS tile of xrows_per + vrows_per rows
// (dynamic LDS: rows * kJacobiTileLd complex entries; at most kTileMaxRows rows)
__global__ void jacobi_tile_kernel(JacobiArgs a);
__global__ void jacobi_tile_batch_kernel(const JacobiArgs* probs, const int* starts,
                                         const int* block_prob);
__global__ void jacobi_batch_kernel(const JacobiArgs* probs, const int* starts,
                                    const int* block_prob);
__global__ void column_norm_kernel(const double2* X, int m, int n, long ldx, double* sigma);
__global__ void rank_sort_kernel(const double* sigma, int n, int* perm, double* sorted);
__global__ void truncate_kernel(const double* sorted, int n, double epsrel, SvdInfo* info,
                                int max_rank, const double* extra2);
__global__ void emit_kernel(EmitArgs a);
// *flag = 1 if a part of the `count` entries is not finite
__global__ void finite_check_kernel(const double2* x, long count, int* flag);
__global__ void conj_copy_kernel(const double2* src, long count, double2* dst);
__global__ void conj_transpose_kernel(const double2* src, int R, int C, double2* dst);
__global__ void transpose_kernel(const double2* src, int R, int C, double2* dst);
__global__ void leg_vector_kernel(const double2* T, int A, int P, int B, const double2* vec,
                                  double2* out);
__global__ void identity_carry_kernel(double2* dst, int R, int V);

constexpr int kJacobiBlock = 16;
constexpr int kJacobiTileLd = 2 * kJacobiBlock + 1;
constexpr int kTileMaxRows = 192;

}  // namespace pte
