// HIP kernels of the process-tensor engine for gfx950 (MI355X).
//
//  * zgemm_kernel      complex128 GEMM with arbitrary strides and optional
//                      conjugation (site x carry contractions, S V^H absorption)
//  * mpo_apply_kernel  applies one influence node W[w,p,s,v] to the GEMM result
//                      G[(l,p),(x,v)] and writes the SVD input matrix or a site
//  * jacobi_kernel     blocked one-sided Jacobi SVD (Hestenes) of a column-major
//                      matrix, one workgroup per row slice of a block pair and
//                      round; a pair waits for its two blocks' last rotation, the
//                      grid only between sweeps (cooperative launch)
//  * small_svd_kernel / gram_svd_kernel / gram_replay_kernel
//                      SVDs of ranks up to 126 by a Jacobi on the Gram matrix in
//                      one workgroup
//  * column_norm_kernel / rank_sort_kernel / truncate_kernel
//                      singular values, descending order, epsrel cut
//  * emit kernels      new sites, carries and S V^H rows from the Jacobi output
//
// Every kernel takes its sizes as arguments and bounds-checks its indices
// against them; the host checks that the sizes match the buffers.
#include "pte_device.h"
#include "pte_kernels.h"

namespace pte {

// Optional phase timers of the cooperative kernels (workgroup 0, thread 0,
// s_memrealtime ticks), compiled in with -DPTE_PHASE_TIMING only.
#ifdef PTE_PHASE_TIMING
__device__ unsigned long long g_phase[16];
#define PHASE_INIT() unsigned long long ph_t_ = wall_clock64()
#define PHASE(k)                                                       \
  do {                                                                 \
    if (blockIdx.x == 0 && threadIdx.x == 0) {                         \
      const unsigned long long t_ = wall_clock64();                    \
      g_phase[k] += t_ - ph_t_;                                        \
      ph_t_ = t_;                                                      \
    }                                                                  \
  } while (0)
// Segment cycle counts of the one-workgroup SVD (thread 0, s_memtime), with
// -DPTE_SEG_TIMING besides (their reads of the clock lengthen the steps): SEG_INIT() starts, SEG(k) adds the cycles since the last
// mark to slot k, SEG_FLUSH(k0, n) adds slots k0.. to g_phase.
#ifdef PTE_SEG_TIMING
#define SEG_INIT()                                 \
  unsigned long long sg_[6] = {0, 0, 0, 0, 0, 0}; \
  unsigned long long sg_t_ = clock64()
#define SEG(k)                                \
  do {                                        \
    const unsigned long long t_ = clock64(); \
    sg_[k] += t_ - sg_t_;                     \
    sg_t_ = t_;                               \
  } while (0)
#define SEG_FLUSH(k0, cnt)                                                 \
  do {                                                                     \
    if (threadIdx.x == 0)                                                  \
      for (int k_ = 0; k_ < (cnt); ++k_) atomicAdd(&g_phase[(k0) + k_], sg_[k_]); \
  } while (0)
#else
#define SEG_INIT() (void)0
#define SEG(k) (void)0
#define SEG_FLUSH(k0, cnt) (void)0
#endif
#else
#define PHASE_INIT() (void)0
#define PHASE(k) (void)0
#define SEG_INIT() (void)0
#define SEG(k) (void)0
#define SEG_FLUSH(k0, cnt) (void)0
#endif

// Optional per-round timestamps of the Jacobi (thread 0 of every workgroup,
// s_memrealtime ticks, for the first kRtRounds rounds and kRtBlocks
// workgroups), compiled in with -DPTE_ROUND_TRACE only.
#ifdef PTE_ROUND_TRACE
constexpr int kRtRounds = 1024, kRtBlocks = 512, kRtMarks = 8;
__device__ unsigned long long g_rtrace[(long)kRtRounds * kRtBlocks * kRtMarks];
#define RTRACE(k)                                                                     \
  do {                                                                                \
    if (threadIdx.x == 0 && rt_round_ < kRtRounds && bid < kRtBlocks)                 \
      g_rtrace[((long)rt_round_ * kRtBlocks + bid) * kRtMarks + (k)] = wall_clock64(); \
  } while (0)
#else
#define RTRACE(k) (void)0
#endif

// ---------------------------------------------------------------------------
// complex GEMM:  C(i,j) = alpha * sum_k opA(A)(i,k) * opB(B)(k,j) [+ C(i,j)]
// 64x64 output tile per 256-thread workgroup, 4x4 outputs per thread, K in
// slices of 16 staged through LDS.
// ---------------------------------------------------------------------------
constexpr int GB_M = 64, GB_N = 64, GB_K = 16;

__global__ void __launch_bounds__(256)
zgemm_kernel(GemmArgs a) {
  __shared__ double2 As[GB_K][GB_M + 1];
  __shared__ double2 Bs[GB_K][GB_N + 1];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;
  const int i0 = blockIdx.y * GB_M, j0 = blockIdx.x * GB_N;
  double2 acc[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[u][v] = make_double2(0.0, 0.0);

  const bool a_kfast = (a.sak == 1);
  const bool b_jfast = (a.sbj == 1);
  for (int k0 = 0; k0 < a.K; k0 += GB_K) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = tid + 256 * q;
      int row, kk;
      if (a_kfast) { row = e >> 4; kk = e & 15; } else { row = e & 63; kk = e >> 6; }
      const int gi = i0 + row, gk = k0 + kk;
      double2 val = make_double2(0.0, 0.0);
      if (gi < a.M && gk < a.K) {
        val = a.A[(long)gi * a.sai + (long)gk * a.sak];
        if (a.conjA) val.y = -val.y;
      }
      As[kk][row] = val;
      int col;
      if (b_jfast) { kk = e >> 6; col = e & 63; } else { kk = e & 15; col = e >> 4; }
      const int gj = j0 + col, gk2 = k0 + kk;
      double2 vb = make_double2(0.0, 0.0);
      if (gj < a.N && gk2 < a.K) {
        vb = a.B[(long)gk2 * a.sbk + (long)gj * a.sbj];
        if (a.conjB) vb.y = -vb.y;
      }
      Bs[kk][col] = vb;
    }
    __syncthreads();
#pragma unroll 4
    for (int kk = 0; kk < GB_K; ++kk) {
      double2 ra[4], rb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) ra[u] = As[kk][ty + 16 * u];
#pragma unroll
      for (int v = 0; v < 4; ++v) rb[v] = Bs[kk][tx + 16 * v];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) cfma(acc[u][v], ra[u], rb[v]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int gi = i0 + ty + 16 * u;
    if (gi >= a.M) continue;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int gj = j0 + tx + 16 * v;
      if (gj >= a.N) continue;
      double2 r = cmul(a.alpha, acc[u][v]);
      double2* c = a.C + (long)gi * a.sci + (long)gj * a.scj;
      if (!a.beta_zero) r = cadd(r, *c);
      *c = r;
    }
  }
}

// ---------------------------------------------------------------------------
// complex128 GEMM on the FP64 matrix cores (the plain form's contraction):
// C(i,j) = alpha * sum_k opA(A)(i,k) opB(B)(k,j) [+ C(i,j)], with a 3M split
// (three real products per complex product, Gauss):
//   P1 = Ar Br,  P2 = Ai Bi,  P3 = (Ar + Ai)(Br + Bi),
//   Re = P1 - P2,  Im = P3 - P1 - P2,
// accumulated in FP64 by v_mfma_f64_16x16x4_f64. 64x64 output tile per
// 256-thread workgroup, each wavefront a 32x32 quarter as 2x2 tiles of
// 16x16; K in slices of 16 staged through LDS as separate real and
// imaginary planes. Operand layout of the FP64 16x16x4 instruction (measured
// on gfx950): lane l supplies A[l%16][l/16] and B[l/16][l%16] and holds
// D[4*r + l/16][l%16] in its item r = 0..3 (rows interleaved by 4, unlike
// the FP32 16x16x4 instruction's D[4*(l/16)+r][l%16]).
// ---------------------------------------------------------------------------
typedef double doublex4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256)
zgemm_mfma_kernel(GemmArgs a) {
  __shared__ double Ar[GB_K][GB_M + 1], Ai[GB_K][GB_M + 1];
  __shared__ double Br[GB_K][GB_N + 1], Bi[GB_K][GB_N + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int i0 = blockIdx.y * GB_M, j0 = blockIdx.x * GB_N;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  doublex4 p1[2][2], p2[2][2], p3[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      p1[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
      p2[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
      p3[u][v] = doublex4{0.0, 0.0, 0.0, 0.0};
    }
  const bool a_kfast = (a.sak == 1);
  const bool b_jfast = (a.sbj == 1);
  for (int k0 = 0; k0 < a.K; k0 += GB_K) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = tid + 256 * q;
      int row, kk;
      if (a_kfast) { row = e >> 4; kk = e & 15; } else { row = e & 63; kk = e >> 6; }
      const int gi = i0 + row, gk = k0 + kk;
      double2 va = make_double2(0.0, 0.0);
      if (gi < a.M && gk < a.K) {
        va = a.A[(long)gi * a.sai + (long)gk * a.sak];
        if (a.conjA) va.y = -va.y;
      }
      Ar[kk][row] = va.x;
      Ai[kk][row] = va.y;
      int col;
      if (b_jfast) { kk = e >> 6; col = e & 63; } else { kk = e & 15; col = e >> 4; }
      const int gj = j0 + col, gk2 = k0 + kk;
      double2 vb = make_double2(0.0, 0.0);
      if (gj < a.N && gk2 < a.K) {
        vb = a.B[(long)gk2 * a.sbk + (long)gj * a.sbj];
        if (a.conjB) vb.y = -vb.y;
      }
      Br[kk][col] = vb.x;
      Bi[kk][col] = vb.y;
    }
    __syncthreads();
#pragma unroll
    for (int k4 = 0; k4 < GB_K; k4 += 4) {
      double ar[2], ai[2], br[2], bi[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        ar[u] = Ar[k4 + lk][wr + 16 * u + lr];
        ai[u] = Ai[k4 + lk][wr + 16 * u + lr];
      }
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        br[v] = Br[k4 + lk][wc + 16 * v + lr];
        bi[v] = Bi[k4 + lk][wc + 16 * v + lr];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          p1[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[u], br[v], p1[u][v], 0, 0, 0);
          p2[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[u], bi[v], p2[u][v], 0, 0, 0);
          p3[u][v] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[u] + ai[u], br[v] + bi[v],
                                                          p3[u][v], 0, 0, 0);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + 16 * u + 4 * r + lk;
        const int gj = j0 + wc + 16 * v + lr;
        if (gi < a.M && gj < a.N) {
          const double re = p1[u][v][r] - p2[u][v][r];
          const double im = p3[u][v][r] - p1[u][v][r] - p2[u][v][r];
          double2 c = cmul(a.alpha, make_double2(re, im));
          double2* dst = a.C + (long)gi * a.sci + (long)gj * a.scj;
          if (!a.beta_zero) c = cadd(c, *dst);
          *dst = c;
        }
      }
}

// ---------------------------------------------------------------------------
// complex GEMM in complex64 with FP32 accumulation on the matrix cores
// (precision form): C(i,j) = sum_k A(i,k) B(k,j), inputs and output stored
// as complex128 and rounded to complex64 when staged. 64x64 output tile per
// 256-thread workgroup; each wavefront owns a 32x32 quarter as 2x2 tiles of
// v_mfma_f32_16x16x4_f32, four real products per complex product:
//   Re += Ar Br - Ai Bi,   Im += Ar Bi + Ai Br.
// Operand layout of the 16x16x4 instruction: lane l supplies A[l%16][l/16]
// and B[l/16][l%16]; it holds D[4*(l/16)+r][l%16], r = 0..3.
// ---------------------------------------------------------------------------
typedef float floatx4 __attribute__((ext_vector_type(4)));

__global__ void __launch_bounds__(256)
cgemm_mfma_kernel(GemmArgs a) {
  __shared__ float2 As[GB_K][GB_M + 1];
  __shared__ float2 Bs[GB_K][GB_N + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int i0 = blockIdx.y * GB_M, j0 = blockIdx.x * GB_N;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  floatx4 accr[2][2], acci[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      accr[u][v] = floatx4{0.f, 0.f, 0.f, 0.f};
      acci[u][v] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
  const bool a_kfast = (a.sak == 1);
  const bool b_jfast = (a.sbj == 1);
  for (int k0 = 0; k0 < a.K; k0 += GB_K) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int e = tid + 256 * q;
      int row, kk;
      if (a_kfast) { row = e >> 4; kk = e & 15; } else { row = e & 63; kk = e >> 6; }
      const int gi = i0 + row, gk = k0 + kk;
      float2 va = make_float2(0.f, 0.f);
      if (gi < a.M && gk < a.K) {
        const double2 v = a.A[(long)gi * a.sai + (long)gk * a.sak];
        va = make_float2((float)v.x, a.conjA ? -(float)v.y : (float)v.y);
      }
      As[kk][row] = va;
      int col;
      if (b_jfast) { kk = e >> 6; col = e & 63; } else { kk = e & 15; col = e >> 4; }
      const int gj = j0 + col, gk2 = k0 + kk;
      float2 vb = make_float2(0.f, 0.f);
      if (gj < a.N && gk2 < a.K) {
        const double2 v = a.B[(long)gk2 * a.sbk + (long)gj * a.sbj];
        vb = make_float2((float)v.x, a.conjB ? -(float)v.y : (float)v.y);
      }
      Bs[kk][col] = vb;
    }
    __syncthreads();
#pragma unroll
    for (int k4 = 0; k4 < GB_K; k4 += 4) {
      float2 av[2], bv[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) av[u] = As[k4 + lk][wr + 16 * u + lr];
#pragma unroll
      for (int v = 0; v < 2; ++v) bv[v] = Bs[k4 + lk][wc + 16 * v + lr];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          accr[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].x, bv[v].x, accr[u][v], 0, 0, 0);
          accr[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(-av[u].y, bv[v].y, accr[u][v], 0, 0, 0);
          acci[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].x, bv[v].y, acci[u][v], 0, 0, 0);
          acci[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u].y, bv[v].x, acci[u][v], 0, 0, 0);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gi = i0 + wr + 16 * u + 4 * lk + r;
        const int gj = j0 + wc + 16 * v + lr;
        if (gi < a.M && gj < a.N) {
          double2 c = make_double2((double)accr[u][v][r], (double)acci[u][v][r]);
          if (!a.beta_zero) c = cadd(c, a.C[(long)gi * a.sci + (long)gj * a.scj]);
          a.C[(long)gi * a.sci + (long)gj * a.scj] = c;
        }
      }
}

// ---------------------------------------------------------------------------
// T[x,s,l,w] = sum_{p,v} W[w,p,s,v] * G[(l,p),(x,v)]
//   mode MPO_OUT_SVD_H : X[(l*Wl+w) + (x*S+s)*ldx] = conj(T)   (X = M^H)
//   mode MPO_OUT_SITE  : out[(l*S+s)*Dx + x] = T   (requires Wl == 1)
//   mode MPO_OUT_M     : out[(x*S+s) + (l*Wl+w)*ldx] = T     (M column-major)
// node_kind DELTA: W[w,p,s,v] = delta(w,v) delta(p,s) I[w,p] (I is Wl x P).
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
mpo_apply_kernel(MpoApplyArgs a) {
  const long total = (long)a.Dx * a.S * a.Dl * a.Wl;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total;
       e += (long)gridDim.x * blockDim.x) {
    // e enumerates (x, s, l, w) with w fastest
    long t = e;
    const int w = t % a.Wl; t /= a.Wl;
    const int l = t % a.Dl; t /= a.Dl;
    const int s = t % a.S;  t /= a.S;
    const int x = (int)t;
    const long gcols = (long)a.Dx * a.V;
    double2 acc = make_double2(0.0, 0.0);
    if (a.kind == NODE_DELTA) {
      // p = s, v = w
      const double2 g = a.G[((long)l * a.P + s) * gcols + (long)x * a.V + w];
      acc = cmul(a.I[(long)w * a.P + s], g);
    } else {
      for (int p = 0; p < a.P; ++p) {
        const double2* grow = a.G + ((long)l * a.P + p) * gcols + (long)x * a.V;
        const double2* wrow = a.W + (((long)w * a.P + p) * a.S + s) * a.V;
        for (int v = 0; v < a.V; ++v) cfma(acc, wrow[v], grow[v]);
      }
    }
    if (a.mode == MPO_OUT_SVD_H) {
      a.out[((long)l * a.Wl + w) + ((long)x * a.S + s) * a.ldx] = cconj(acc);
    } else if (a.mode == MPO_OUT_M) {
      a.out[((long)x * a.S + s) + ((long)l * a.Wl + w) * a.ldx] = acc;
    } else {
      a.out[((long)l * a.S + s) * a.Dx + x] = acc;
    }
  }
}

// ---------------------------------------------------------------------------
// TEMPO zip (left to right):
// T[x,s,r,e] = sum_{p,w} W[w,p,s,e] * G[(x,w),(p,r)]
//   mode MPO_OUT_SVD_H : X[(r*E+e) + (x*S+s)*ldx] = conj(T)
//   mode MPO_OUT_M     : out[(x*S+s) + (r*E+e)*ldx] = T   (M column-major)
//   mode MPO_OUT_SITE  : out[(x*S+s)*E + e] = T (requires Dr == 1)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
mpo_apply_right_kernel(MpoApplyArgs a) {
  // reuse of fields: Dl <- Dr (right bond of the site), Wl <- E (east leg),
  // V <- W (west leg of the node)
  const int Dr = a.Dl, E = a.Wl, Wn = a.V;
  const long total = (long)a.Dx * a.S * Dr * E;
  for (long e_ = blockIdx.x * (long)blockDim.x + threadIdx.x; e_ < total;
       e_ += (long)gridDim.x * blockDim.x) {
    long t = e_;
    const int e = t % E; t /= E;
    const int r = t % Dr; t /= Dr;
    const int s = t % a.S; t /= a.S;
    const int x = (int)t;
    const long gcols = (long)a.P * Dr;
    double2 acc = make_double2(0.0, 0.0);
    if (a.kind == NODE_DELTA) {
      // W[w,p,s,e] = delta(w,e) delta(p,s) I[w,p]  ->  w = e, p = s
      const double2 g = a.G[((long)x * Wn + e) * gcols + (long)s * Dr + r];
      acc = cmul(a.I[(long)e * a.P + s], g);
    } else {
      for (int w = 0; w < Wn; ++w) {
        const double2* grow = a.G + ((long)x * Wn + w) * gcols;
        for (int p = 0; p < a.P; ++p) {
          const double2 wv = a.W[(((long)w * a.P + p) * a.S + s) * E + e];
          cfma(acc, wv, grow[(long)p * Dr + r]);
        }
      }
    }
    if (a.mode == MPO_OUT_SVD_H) {
      a.out[((long)r * E + e) + ((long)x * a.S + s) * a.ldx] = cconj(acc);
    } else if (a.mode == MPO_OUT_M) {
      a.out[((long)x * a.S + s) + ((long)r * E + e) * a.ldx] = acc;
    } else {
      a.out[((long)x * a.S + s) * E + e] = acc;
    }
  }
}

// ---------------------------------------------------------------------------
// Blocked one-sided Jacobi SVD.
// X (m x n, column-major, leading dimension ldx) is orthogonalised column-wise:
// X <- X Q with Q unitary accumulated in V (n x n, column-major). Columns are
// grouped into blocks of JB; in every round each block pair of the
// round-robin tournament over nb blocks is handled by `slices` workgroups,
// each owning a slice of the rows of X and of V. The pair's 2JB x 2JB Gram
// matrix is summed from the slices' partial Grams, diagonalised (cyclic
// two-sided Jacobi in LDS, at most inner_sweeps sweeps, identically in every
// workgroup of the pair) and the resulting unitary applied to the slice's rows
// of X and V. A sweep is nb-1 rounds; the iteration stops after a sweep in
// which no pair needed a rotation. Rounds are not separated by grid barriers:
// every block carries a version (rounds completed on it), a pair starts a
// round once both of its blocks have reached it and, when all of its slices
// are done, releases them for the next round; the slices of a pair exchange
// partial Grams through a pair-local barrier (double-buffered by round
// parity); a grid barrier closes each sweep. A pair needs one when some
// |g_ij| > tol*sqrt(g_ii g_jj) and |g_ij| > abs_tol*sqrt(max(g_ii, g_jj)).
// ---------------------------------------------------------------------------
constexpr int JB = 16;          // block width
constexpr int JP = 2 * JB;      // columns per block pair
constexpr int JR = 32;          // rows per streamed chunk
constexpr int JT = 256;         // threads per workgroup
#ifndef PTE_JACOBI_SUM_BATCH
#define PTE_JACOBI_SUM_BATCH 4
#endif
// slices of partial Grams whose loads are in flight together
constexpr int kJacobiSumBatch = PTE_JACOBI_SUM_BATCH;

__device__ __forceinline__ void tournament_pair(int nplayers, int round, int slot,
                                                int& a, int& b) {
  if (slot == 0) {
    a = nplayers - 1;
    b = round % (nplayers - 1);
  } else {
    a = (round + slot) % (nplayers - 1);
    b = (round - slot + nplayers - 1) % (nplayers - 1);
  }
}

// Does the Hermitian 2x2 block [[app, apq], [conj(apq), aqq]] need a rotation:
// |apq| > tol * sqrt(|app aqq|) and |apq| > abs_tol * sqrt(max(app, aqq)),
// compared in squares.
__device__ __forceinline__ bool needs_rotation(double app, double aqq, double mag2,
                                               double tol2, double abs_tol2) {
  return mag2 > tol2 * fabs(app * aqq) && mag2 > abs_tol2 * fmax(fmax(app, aqq), 0.0) &&
         mag2 > 0.0;
}

// 1/sqrt(x) for normal positive x: the hardware estimate (measured relative
// error 2^-24) refined by one cubic step to full double precision.
__device__ __forceinline__ double rsqrt_nr(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Rotation of the 2 x 2 block [[app, apq], [conj(apq), aqq]]: with
// d = aqq - app and h = sqrt(d^2 + 4 |apq|^2), c = cos(theta) =
// sqrt((h + |d|) / 2h) and s = sign(d) apq / (h c) (theta = pi/4 for d = 0); no
// sum in it cancels, and the phase of apq stays in s, so its modulus is not
// needed. The identity where no rotation is needed. The Gram matrices are
// scaled to a trace near one, so the squares stay in range.
// Returns whether one is; the rotated diagonal is app - shift, aqq + shift.
__device__ __forceinline__ bool gram_rotation(bool valid, double app, double aqq, double2 apq,
                                              double tol2, double abs_tol2, double& c,
                                              double2& s, double& shift) {
  const double mag2 = cabs2(apq);
  const bool need = valid & (mag2 > tol2 * fabs(app * aqq)) & (mag2 > abs_tol2 * app) &
                    (mag2 > abs_tol2 * aqq) & (mag2 > 0.0);
  const double d = aqq - app;
  const double h2 = need ? fma(d, d, 4.0 * mag2) : 1.0;
  const double rh = rsqrt_nr(h2);
  const double cos2 = fma(0.5 * fabs(d), rh, 0.5);
  const double rc = rsqrt_nr(cos2);
  const double f = copysign(rh * rc, d < 0.0 ? -1.0 : 1.0);
  c = need ? cos2 * rc : 1.0;
  s = make_double2(need ? apq.x * f : 0.0, need ? apq.y * f : 0.0);
  shift = need ? f * rc * mag2 : 0.0;
  return need;
}
__device__ __forceinline__ bool gram_rotation(bool valid, double app, double aqq, double2 apq,
                                              double tol2, double abs_tol2, double& c,
                                              double2& s) {
  double shift;
  return gram_rotation(valid, app, aqq, apq, tol2, abs_tol2, c, s, shift);
}

// Places of a Hermitian matrix kept by round-robin position (gram_jacobi and
// the pair sweeps below): position 2q holds the first column a_q of pair q,
// position 2q + 1 its second, b_q; position 0 keeps its column and the others
// move on by one position a round (gram_next), so that after 2P - 1 rounds (P
// pairs) every two columns have met and all are back. The matrix is stored as
// the P (P + 1) / 2 blocks (q1, q2), q1 <= q2, of 2 x 2 entries, entry e of every
// block in a plane of its own.
__device__ __forceinline__ int gram_block(int q1, int q2) { return q2 * (q2 + 1) / 2 + q1; }

// The cosine that belongs to the rounded s: c + (1 - c^2 - |s|^2) / 2c. The root of
// cos2, which near one is rounded to twice the spacing above than below, makes c too
// small on average, and the columns' norms shrank by 6e-15 over the 600 rotations
// of an 88 x 83 matrix, which set the error of the factorisation (1.5e-14 of the
// largest singular value; 3.3e-15 so). 1.5% of that SVD's time.
__device__ __forceinline__ double unit_c(double c, double2 s) {
  return fma(0.5 * __builtin_amdgcn_rcp(c), fma(-c, c, 1.0) - cabs2(s), c);
}

// position of column c in round 0 (P pairs) and a position's next one
__device__ __forceinline__ int gram_pos(int c, int P) {
  const int L = 2 * P - 1;
  return c == L ? 0 : c == 0 ? 1 : c < P ? 2 * c : 2 * (L - c) + 1;
}
__device__ __forceinline__ int gram_next(int x, int P) {
  if (x == 0 || P == 1) return x;
  if (x == 2) return 1;
  if ((x & 1) == 0) return x - 2;
  return x == 2 * P - 1 ? x - 1 : x + 2;
}

// where the entry of positions (x, y) is kept (T: entries of a plane), and
// whether conjugated
__device__ __forceinline__ int gram_place(int x, int y, int T, bool& conj) {
  const int qx = x >> 1, qy = y >> 1;
  conj = qx > qy || (qx == qy && x > y);
  if (conj) return (2 * (y & 1) + (x & 1)) * T + gram_block(qy, qx);
  return (2 * (x & 1) + (y & 1)) * T + gram_block(qx, qy);
}

// ---- cyclic two-sided Jacobi sweeps on a block pair's 2JB x 2JB Gram matrix,
// by 256 threads ----
// The matrix is kept by position (PT blocks, four planes) in two buffers: a
// round reads one and writes the other with the entries where their columns are
// in the next round. What a round takes is the chain from one round's rotations
// to the next's, so wavefront 0 does nothing else: lane q has pair q's diagonal
// in registers, transforms the one entry of another block that will be its
// next pair's off-diagonal one, and computes the next rotation while wavefronts
// 1 and 2 rotate the 120 off-diagonal blocks from both sides (a thread each) and
// 1 to 3 accumulate the rotations in W, whose rows are in registers: lane q (mod
// 16) of a row of lanes has the entries of columns a_q and b_q, which move on by
// one lane a round. One barrier a round (11 cycles with four wavefronts).
// A round takes 0.39 us; 0.75 us with every wavefront computing the rotations
// from a column-indexed matrix and W in LDS, and 0.65 us with the matrix by
// position but the rotations and the updates one after the other.
constexpr int PP = JB;                      // pairs of a block pair's columns
constexpr int PT = PP * (PP + 1) / 2;       // blocks of its Gram matrix
constexpr int kPairOwners = PT - PP;        // off-diagonal ones, a thread each
static_assert(PP == 16 && kPairOwners <= 128, "a DPP row of pairs; owners in wavefronts 1 and 2");
constexpr int kDppRowShl1 = 0x101, kDppRowShr1 = 0x111;

// A thread's constants: its block (wavefront 0: pair lane % 16's diagonal one),
// the places of the entries in the next round (as in gram_jacobi) and the places
// at which it stores the Gram matrix.
struct PairThread {
  int q1, q2;
  unsigned dst[2];
  int store[4];       // -1: not stored (lower triangle); bit 30: conjugated
};

__device__ __forceinline__ PairThread pair_thread(int slices) {
  PairThread t;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int b = min(max(tid - 64, 0), kPairOwners - 1);
  int c = 1;
  while (c * (c + 1) / 2 <= b) ++c;
  t.q2 = wave == 0 ? lane & 15 : c;
  t.q1 = wave == 0 ? lane & 15 : b - c * (c - 1) / 2;
  t.dst[0] = t.dst[1] = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    bool conj = false;
    const int at = gram_place(gram_next(2 * t.q1 + (e >> 1), PP),
                              gram_next(2 * t.q2 + (e & 1), PP), PT, conj);
    t.dst[e >> 1] |= ((unsigned)at | (conj ? 0x8000u : 0u)) << (16 * (e & 1));
    // entries of a thread: the MFMA tile of its wavefront (one slice), or
    // entry tid + 256 e of the summed partial Grams
    const int i = slices == 1 ? 16 * (wave >> 1) + 4 * e + (lane >> 4) : (tid + JT * e) / JP;
    const int j = slices == 1 ? 16 * (wave & 1) + (lane & 15) : (tid + JT * e) % JP;
    bool cs = false;
    const int place = gram_place(gram_pos(i, PP), gram_pos(j, PP), PT, cs);
    t.store[e] = i > j ? -1 : place | (cs ? 1 << 30 : 0) | (i == j ? 1 << 29 : 0);
  }
  return t;
}

// entry e of a thread's Gram entries (scaled by sc)
__device__ __forceinline__ void pair_store(double2* Gp, const PairThread& t, int e, double2 v,
                                           double sc) {
  const int s = t.store[e];
  if (s < 0) return;
  const double y = (s & (1 << 29)) ? 0.0 : ((s & (1 << 30)) ? -v.y : v.y);
  Gp[s & 0xffff] = make_double2(v.x * sc, y * sc);
}

// does some pair of the block pair need a rotation (the workgroup's answer)
__device__ __forceinline__ bool pair_needs(const double2* Gp, const PairThread& t, double tol2,
                                           double abs_tol2) {
  const int b = gram_block(t.q1, t.q2);
  const int b1 = gram_block(t.q1, t.q1), b2 = gram_block(t.q2, t.q2);
  const double da1 = Gp[b1].x, db1 = Gp[3 * PT + b1].x;
  const double da2 = Gp[b2].x, db2 = Gp[3 * PT + b2].x;
  bool any = needs_rotation(da1, db2, cabs2(Gp[PT + b]), tol2, abs_tol2);
  if (threadIdx.x >= 64) {
    any |= needs_rotation(da1, da2, cabs2(Gp[b]), tol2, abs_tol2);
    any |= needs_rotation(db1, da2, cabs2(Gp[2 * PT + b]), tol2, abs_tol2);
    any |= needs_rotation(db1, db2, cabs2(Gp[3 * PT + b]), tol2, abs_tol2);
  }
  return __builtin_amdgcn_readfirstlane(__syncthreads_or((int)any)) != 0;
}

// lane move; a lane without a source keeps `old`
template <int CTRL>
__device__ __forceinline__ double dpp_keep_d(double old, double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, 0xf, 0xf, false),
      __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, 0xf, 0xf, false));
}
// The sweeps; W (row-major, by column) goes to Ws, whose memory is the second
// buffer until then. rc and rs have two buffers of PP entries.
__device__ __forceinline__ void pair_sweeps(double2* Gp, double* rc, double2* rs,
                                            double2 (*Ws)[JP + 2], const PairThread& t,
                                            double tol2, double abs_tol2, int inner_sweeps) {
  static_assert(4 * PT <= JP * (JP + 2), "the second buffer fits into Ws");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q = lane & 15;
  const bool first = q == 0, last = q == PP - 1;
  const int rounds = inner_sweeps * (JP - 1);
  double2* from = Gp;
  double2* to = &Ws[0][0];
  auto put = [&](unsigned place, double2 v) {   // place in the upper 16 bits
    v.y = __hiloint2double(__double2hiint(v.y) ^ (int)(place & 0x80000000u),
                           __double2loint(v.y));
    to[(place >> 16) & 0x7fffu] = v;
  };
  if (wave == 0) {
    // Pair q's next columns come from pairs q + 1 (its a) and q - 1 (its b); at
    // the ends a_0 stays, b_0 was a_1, and a_last was b_last. Lane 0 has its two
    // columns the other way round (its apq is the conjugate, its s -conj(s)):
    // what enters at the ends of the lanes is then the value that a lane
    // without a source keeps, but for one selection. Of the block (q1, q2) of
    // those two pairs the entry (x, y) is wanted, x, y = b, a in the middle, a, a
    // at the first and b, b at the last: with the columns' c it is rotated to
    // c1 (c2 E_cc + z2 E_cs) + z1 (c2 E_sc + z2 E_ss), where E_c. is the column's
    // own entry, E_s. the other column's, and z = -s (row) or -conj(s) (column)
    // for an a, conj(s) (row) or s (column) for a b.
    const int q1 = first ? 0 : last ? PP - 2 : q - 1, q2 = first ? 1 : last ? PP - 1 : q + 1;
    const int row = first ? 0 : 1, col = last ? 1 : 0;
    const int blk = gram_block(q1, q2);
    const int cc = (2 * row + col) * PT + blk, cs = (2 * row + (col ^ 1)) * PT + blk;
    const int sc = (2 * (row ^ 1) + col) * PT + blk;
    const int ss = (2 * (row ^ 1) + (col ^ 1)) * PT + blk;
    const double z1x = first ? -1.0 : 1.0, z2x = last ? 1.0 : -1.0, sx = first ? -1.0 : 1.0;
    const unsigned dst = t.dst[0] ^ (first ? 0x80000000u : 0u);
    const int dq = gram_block(q, q);
    double app = Gp[(first ? 3 : 0) * PT + dq].x, aqq = Gp[(first ? 0 : 3) * PT + dq].x;
    double c, shift;
    double2 apq = Gp[PT + dq], s;
    if (first) apq.y = -apq.y;
    bool need = gram_rotation(true, app, aqq, apq, tol2, abs_tol2, c, s, shift);
    rc[q] = c;       // (the four rows of lanes are alike)
    rs[q] = make_double2(sx * s.x, s.y);
    __syncthreads();
    for (int round = 0; round < rounds; ++round) {
      const double* const c_ = rc + (round & 1) * PP;
      const double2* const s_ = rs + (round & 1) * PP;
      const double2 ecc = from[cc], ecs = from[cs], esc = from[sc], ess = from[ss];
      const double c1 = c_[q1], c2 = c_[q2];
      const double2 s1 = s_[q1], s2 = s_[q2];
      put(dst, need ? make_double2(0.0, 0.0) : apq);
      const double na = app - shift, nb = aqq + shift;
      const double x = first ? na : nb;
      aqq = dpp_keep_d<kDppRowShr1>(nb, x);
      app = dpp_keep_d<kDppRowShl1>(x, na);
      const double2 z1 = make_double2(z1x * s1.x, -s1.y);
      const double2 z2 = make_double2(z2x * s2.x, s2.y);
      const double2 n0 = cadd(cscale(ecc, c2), cmul(z2, ecs));
      const double2 n1 = cadd(cscale(esc, c2), cmul(z2, ess));
      apq = cconj(cadd(cscale(n0, c1), cmul(z1, n1)));
      need = gram_rotation(true, app, aqq, apq, tol2, abs_tol2, c, s, shift);
      const int at = ((round + 1) & 1) * PP + q;
      rc[at] = c;
      rs[at] = make_double2(sx * s.x, s.y);
      double2* const y = from;
      from = to;
      to = y;
      __syncthreads();
    }
    __syncthreads();
  } else {
    // rows of W, four at a time: 0 to 23 wavefront 3, 24 to 27 wavefront 1, 28 to
    // 31 wavefront 2
    const int row0 = (wave == 3 ? 0 : 20 + 4 * wave) + (lane >> 4);
    const int ca = q, cb = JP - 1 - q;    // (lane 0 the other way round, as above)
    const double sx = first ? -1.0 : 1.0;
    const bool own = tid - 64 < kPairOwners;
    const int b = gram_block(t.q1, t.q2);
    constexpr int kRows = 6;
    double2 wa[kRows], wb[kRows];
#pragma unroll
    for (int h = 0; h < kRows; ++h) {
      wa[h] = make_double2(row0 + 4 * h == ca ? 1.0 : 0.0, 0.0);
      wb[h] = make_double2(row0 + 4 * h == cb ? 1.0 : 0.0, 0.0);
    }
    __syncthreads();
    for (int round = 0; round < rounds; ++round) {
      const double* const c_ = rc + (round & 1) * PP;
      const double2* const s_ = rs + (round & 1) * PP;
      const double c = c_[q];
      const double2 s = make_double2(sx * s_[q].x, s_[q].y);
      auto rows = [&](int h) __attribute__((always_inline)) {
        const double2 ya = csub(cscale(wa[h], c), cmul(cconj(s), wb[h]));
        const double2 yb = cadd(cmul(s, wa[h]), cscale(wb[h], c));
        const double2 x = make_double2(first ? ya.x : yb.x, first ? ya.y : yb.y);
        wb[h] = make_double2(dpp_keep_d<kDppRowShr1>(yb.x, x.x), dpp_keep_d<kDppRowShr1>(yb.y, x.y));
        wa[h] = make_double2(dpp_keep_d<kDppRowShl1>(x.x, ya.x), dpp_keep_d<kDppRowShl1>(x.y, ya.y));
      };
      if (wave == 3) {
#pragma unroll
        for (int h = 1; h < kRows; ++h) rows(h);
      } else if (own) {
        const double2 b00 = from[b], b01 = from[PT + b];
        const double2 b10 = from[2 * PT + b], b11 = from[3 * PT + b];
        const double c1 = c_[t.q1], c2 = c_[t.q2];
        const double2 s1 = s_[t.q1], s2 = s_[t.q2];
        const double2 s1c = cconj(s1), s2c = cconj(s2);
        const double2 n00 = csub(cscale(b00, c2), cmul(s2c, b01));
        const double2 n01 = cadd(cmul(s2, b00), cscale(b01, c2));
        const double2 n10 = csub(cscale(b10, c2), cmul(s2c, b11));
        const double2 n11 = cadd(cmul(s2, b10), cscale(b11, c2));
        put(t.dst[0] << 16, csub(cscale(n00, c1), cmul(s1, n10)));
        put(t.dst[0], csub(cscale(n01, c1), cmul(s1, n11)));
        put(t.dst[1] << 16, cadd(cmul(s1c, n00), cscale(n10, c1)));
        put(t.dst[1], cadd(cmul(s1c, n01), cscale(n11, c1)));
      }
      rows(0);
      double2* const y = from;
      from = to;
      to = y;
      __syncthreads();
    }
    __syncthreads();   // (wavefront 0 has left the buffers too)
#pragma unroll
    for (int h = 0; h < kRows; ++h) {
      if (h >= 1 && wave != 3) break;
      Ws[row0 + 4 * h][ca] = wa[h];
      Ws[row0 + 4 * h][cb] = wb[h];
    }
  }
  __syncthreads();
}

// power of two that brings ||X||_F^2 to [1, 4) (1 where that is not a number)
__device__ __forceinline__ double gram_scaling(double fro2) {
  return (fro2 > 0.0 && fro2 < 1.7e308) ? ldexp(1.0, -2 * (ilogb(fro2) >> 1)) : 1.0;
}

// One 32-row chunk of the pair's 32 columns (rows r0.., below hi), four
// entries per thread (entry e = tid + 256 q: row e % 32, column e / 32), read
// with agent-scope loads; PF chunks are issued before any is consumed so
// that their latencies overlap.
constexpr int PF = 4;

__device__ __forceinline__ void load_chunk(double2 (&out)[4], const double2* base, long ld,
                                           int r0, int hi, const int* cols) {
  // 16-byte agent-coherent loads within the first 2^31 bytes of the
  // matrix (the buffer offset range), the pair of 8-byte loads beyond
  const __amdgpu_buffer_rsrc_t rs = agent_rsrc(base, 0x7fffffffu);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = threadIdx.x + JT * q;
    const int rr = e % JR, cc = e / JR;
    const int gr = r0 + rr, gc = cols[cc];
    const long off = gr + (long)gc * ld;
    out[q] = (gr < hi && gc >= 0)
                 ? (off < kBufMaxEntries ? ld_agent16(rs, (unsigned)off * 16u) : ld_agent(base + off))
                 : make_double2(0.0, 0.0);
  }
}

__device__ __forceinline__ void put_chunk(double2 (*Xs)[JP + 1], const double2 (&in)[4]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int e = threadIdx.x + JT * q;
    Xs[e % JR][e / JR] = in[q];
  }
}

__device__ __forceinline__ void jacobi_body(const JacobiArgs& a, const int bid,
                                            const unsigned nblk) {
  __shared__ double2 Xs[JR][JP + 1];
  __shared__ double2 Gp[4 * PT];              // the pair's Gram matrix, by position
  __shared__ double2 Ws[JP][JP + 2];
  __shared__ double2 rot_s[2 * PP];
  __shared__ double rot_c[2 * PP];
  __shared__ int cols[JP];
  __shared__ bool skip_pair;
  __shared__ double red[JT];

  const int tid = threadIdx.x;
  const int R = a.slices;
  const int pair = bid / R, slice = bid % R;
  const int x_lo = min(a.m, slice * a.xrows_per), x_hi = min(a.m, x_lo + a.xrows_per);
  const int v_lo = min(a.n, slice * a.vrows_per), v_hi = min(a.n, v_lo + a.vrows_per);
  unsigned epoch = 0;
  const PairThread pt = pair_thread(R);

  // V = identity, Frobenius norm of X
  for (long e = bid * (long)JT + tid; e < (long)a.n * a.n;
       e += (long)nblk * JT) {
    const long i = e % a.n, j = e / a.n;
    st_agent(a.V + (i + j * a.ldv), make_double2(i == j ? 1.0 : 0.0, 0.0));
  }
  double part = 0.0;
  for (long e = bid * (long)JT + tid; e < (long)a.m * a.n;
       e += (long)nblk * JT) {
    const long i = e % a.m, j = e / a.m;
    part += cabs2(a.X[i + j * a.ldx]);
  }
  red[tid] = part;
  __syncthreads();
  for (int s = JT / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) atomicAdd(a.fro2, red[0]);
  grid_barrier_all(a.bar, nblk, bid, epoch);
  // the pairs' Gram matrices are scaled with ||X||_F^2 (gram_scaling)
  const double fro2 = ld_agent(a.fro2);
  const double gsc = gram_scaling(fro2);
  const double tol2 = a.tol * a.tol;
  const double abs_tol2 = a.abs_tol_scale * a.abs_tol_scale * (fro2 * gsc);
  const int ti = tid >> 4, tj = tid & 15;        // 2x2 Gram blocking
  const int npairs = a.nb / 2;
  unsigned* pair_bar = a.bar + kBarrierWords;
  unsigned* pair_done = pair_bar + npairs;
  unsigned* blockver = pair_done + npairs;
  unsigned gen = 0, pair_epoch = 0;

  int sweep = 0;
  bool converged = false;
  PHASE_INIT();
  for (; sweep < a.max_sweeps; ++sweep) {
    for (int round = 0; round < a.nb - 1; ++round) {
      PHASE(7);
#ifdef PTE_ROUND_TRACE
      const int rt_round_ = sweep * (a.nb - 1) + round;
#endif
      RTRACE(0);
      int bi, bj;
      tournament_pair(a.nb, round, pair, bi, bj);
      if (tid < JP) {
        const int c = (tid < JB) ? bi * JB + tid : bj * JB + (tid - JB);
        cols[tid] = (c < a.n) ? c : -1;
      }
      // both blocks released by the pairs that held them in the previous round
      const int plo = min(bi, bj), phi = max(bi, bj);
      unsigned* const pair_ok = a.skip + a.nb + ((long)phi * (phi - 1)) / 2 + plo;
      if (tid == 0) {
        while (ld_agent(blockver + bi) < gen || ld_agent(blockver + bj) < gen)
          __builtin_amdgcn_s_sleep(1);
        // a pair found converged whose blocks have not been rotated since has
        // the same Gram matrix: it needs no rotation and no pass over X
        const unsigned ok = ld_agent(pair_ok);
        skip_pair = ok != 0u && ld_agent(a.skip + bi) < ok && ld_agent(a.skip + bj) < ok;
      }
      __syncthreads();
      RTRACE(1);
      if (__builtin_amdgcn_readfirstlane((int)skip_pair)) {
        // the pair barrier is kept in a skipped round: without it a slice
        // could finish the next round before a slower slice of its pair
        // finished this one, and the arrival count on pair_done, which
        // releases the blocks, would then never reach this round's total
        if (R > 1) grid_barrier(pair_bar + pair, R, pair_epoch);
      } else {
      // ---- partial Gram of the pair's columns over this slice's rows ----
      double2 g[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) g[u][v] = make_double2(0.0, 0.0);
      for (int gbase = x_lo; gbase < x_hi; gbase += PF * JR) {
        double2 pre[PF][4];
#pragma unroll
        for (int c = 0; c < PF; ++c) load_chunk(pre[c], a.X, a.ldx, gbase + c * JR, x_hi, cols);
#pragma unroll
        for (int c = 0; c < PF; ++c) {
          if (gbase + c * JR >= x_hi) break;
          put_chunk(Xs, pre[c]);
          __syncthreads();
#pragma unroll 4
          for (int rr = 0; rr < JR; ++rr) {
            const double2 a0 = Xs[rr][ti], a1 = Xs[rr][ti + 16];
            const double2 b0 = Xs[rr][tj], b1 = Xs[rr][tj + 16];
            cfmac(g[0][0], a0, b0);
            cfmac(g[0][1], a0, b1);
            cfmac(g[1][0], a1, b0);
            cfmac(g[1][1], a1, b1);
          }
          __syncthreads();
        }
      }
      if (R == 1) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int v = 0; v < 2; ++v) {
            const int i = ti + 16 * u, j = tj + 16 * v;
            bool conj;
            const int at = gram_place(gram_pos(i, PP), gram_pos(j, PP), PT, conj);
            const double y = i == j ? 0.0 : (conj ? -g[u][v].y : g[u][v].y);
            if (i <= j) Gp[at] = make_double2(g[u][v].x * gsc, y * gsc);
          }
      } else {
        // double-buffered by round parity (every round of a pair, skipped or
        // not, passes its pair barrier)
        double2* gbuf = a.gpart + (long)(pair_epoch & 1) * npairs * R * (JP * JP);
        double2* mine = gbuf + ((long)pair * R + slice) * (JP * JP);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int v = 0; v < 2; ++v) st_agent(mine + ((ti + 16 * u) * JP + tj + 16 * v), g[u][v]);
        PHASE(0);
        RTRACE(2);
        grid_barrier(pair_bar + pair, R, pair_epoch);
        PHASE(1);
        RTRACE(3);
        // identical summation order (slice 0, 1, ...) in every workgroup of
        // the pair; loads of kJacobiSumBatch slices are in flight together
        constexpr int SB = kJacobiSumBatch;
        double2 acc[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = make_double2(0.0, 0.0);
        const double2* gp = gbuf + (long)pair * R * (JP * JP);
        for (int sl0 = 0; sl0 < R; sl0 += SB) {
          double2 v[SB][4];
#pragma unroll
          for (int t = 0; t < SB; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              v[t][q] = (sl0 + t < R) ? ld_agent(gp + (long)(sl0 + t) * (JP * JP) + tid + JT * q)
                                      : make_double2(0.0, 0.0);
#pragma unroll
          for (int t = 0; t < SB; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (sl0 + t < R) acc[q] = cadd(acc[q], v[t][q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) pair_store(Gp, pt, q, acc[q], gsc);
      }
      __syncthreads();
      const bool need = pair_needs(Gp, pt, tol2, abs_tol2);
      PHASE(2);
      RTRACE(4);
      // record the outcome for later rounds: a rotated pair's blocks change,
      // an unrotated pair is converged as long as they do not
      if (slice == 0 && tid == 0) {
        if (need) {
          st_agent(a.skip + bi, gen + 1);
          st_agent(a.skip + bj, gen + 1);
          st_agent(pair_ok, 0u);
        } else {
          st_agent(pair_ok, gen + 1);
        }
      }
      if (need) {
        pair_sweeps(Gp, rot_c, rot_s, Ws, pt, tol2, abs_tol2, a.inner_sweeps);
        PHASE(3);
        RTRACE(5);
        // ---- X_pair <- X_pair Ws, V_pair <- V_pair Ws over this slice ----
        const int rr = tid >> 3, c0 = (tid & 7) * 4;
        const int nx = (x_hi - x_lo + JR - 1) / JR, nv = (v_hi - v_lo + JR - 1) / JR;
        for (int t0 = 0; t0 < nx + nv; t0 += PF) {
          double2 pre[PF][4];
#pragma unroll
          for (int c = 0; c < PF; ++c) {
            const int t = t0 + c;
            if (t < nx) load_chunk(pre[c], a.X, a.ldx, x_lo + t * JR, x_hi, cols);
            else if (t < nx + nv) load_chunk(pre[c], a.V, a.ldv, v_lo + (t - nx) * JR, v_hi, cols);
          }
#pragma unroll
          for (int c = 0; c < PF; ++c) {
            const int t = t0 + c;
            if (t >= nx + nv) break;
            const bool isx = t < nx;
            double2* base = isx ? a.X : a.V;
            const long ld = isx ? a.ldx : a.ldv;
            const int r0 = isx ? x_lo + t * JR : v_lo + (t - nx) * JR;
            const int hi = isx ? x_hi : v_hi;
            put_chunk(Xs, pre[c]);
            __syncthreads();
            double2 o[4];
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) o[cc] = make_double2(0.0, 0.0);
#pragma unroll 8
            for (int i = 0; i < JP; ++i) {
              const double2 xv = Xs[rr][i];
#pragma unroll
              for (int cc = 0; cc < 4; ++cc) cfma(o[cc], xv, Ws[i][c0 + cc]);
            }
            __syncthreads();
            // through LDS, so that each store covers 32 consecutive rows of
            // one column (512 contiguous bytes) instead of scattered entries
#pragma unroll
            for (int cc = 0; cc < 4; ++cc) Xs[rr][c0 + cc] = o[cc];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int e = tid + JT * q;
              const int row = e % JR, col = e / JR;
              const int gr = r0 + row, gc = cols[col];
              const long off = gr + (long)gc * ld;
              if (gr < hi && gc >= 0) {
                if (off < kBufMaxEntries)
                  st_agent16(agent_rsrc(base, 0x7fffffffu), (unsigned)off * 16u, Xs[row][col]);
                else
                  st_agent(base + off, Xs[row][col]);
              }
            }
            __syncthreads();
          }
        }
        if (tid == 0) st_agent(a.flags + sweep, 1);
        PHASE(4);
        RTRACE(6);
      }
      }   // skip_pair
      // the last slice of the pair to finish releases both blocks
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(pair_done + pair, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        if (old == (gen + 1) * (unsigned)R - 1) {
          st_agent(blockver + bi, gen + 1);
          st_agent(blockver + bj, gen + 1);
        }
      }
      ++gen;
      PHASE(5);
      RTRACE(7);
    }
    grid_barrier_all(a.bar, nblk, bid, epoch);
    if (__hip_atomic_load(&a.flags[sweep], __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT) == 0) {
      converged = true;
      break;
    }
  }
  if (bid == 0 && tid == 0) *a.info = converged ? sweep + 1 : -1;
}

// Two workgroups a CU: the row slices of a pair are split over twice as many
// (2652 x 2364: 265 ms; 451 ms with one).
__global__ void __launch_bounds__(JT, 2)
jacobi_kernel(JacobiArgs a) {
  jacobi_body(a, blockIdx.x, gridDim.x);
}

// Several independent SVDs in one cooperative launch: workgroup b works on
// problem block_prob[b] as its (b - starts[p])-th workgroup of
// starts[p+1] - starts[p]; every problem has its own barrier counter.
__global__ void __launch_bounds__(JT, 2)
jacobi_batch_kernel(const JacobiArgs* probs, const int* starts, const int* block_prob) {
  const int p = block_prob[blockIdx.x];
  const int s0 = starts[p];
  const JacobiArgs a = probs[p];
  jacobi_body(a, blockIdx.x - s0, starts[p + 1] - s0);
}

// The same Jacobi with the slice kept in LDS for the round (one workgroup
// per compute unit): each round loads the slice's rows of X and of V in the
// pair's 32 columns into an LDS tile with one batch of coalesced loads,
// computes the partial Gram from it and, after the pair's inner sweeps, the
// rotation X <- X W, V <- V W in place on the FP64 matrix cores
// (v_mfma_f64_16x16x4_f64, 3M split), and writes the tile back with coalesced
// stores. The round protocol (block versions, converged-pair skipping, pair
// barrier, release count) is the one of jacobi_body. The tile has
// a.xrows_per + a.vrows_per rows of JP + 1 entries (dynamic LDS).
constexpr int kTileLd = kJacobiTileLd;
static_assert(kTileLd == JP + 1, "tile row stride");

__device__ __forceinline__ void jacobi_tile_body(const JacobiArgs& a, const int bid,
                                                 const unsigned nblk) {
  extern __shared__ double2 tile[];
  __shared__ double2 Gp[4 * PT];              // the pair's Gram matrix, by position
  __shared__ double2 Ws[JP][JP + 2];
  __shared__ double2 rot_s[2 * PP];
  __shared__ double rot_c[2 * PP];
  __shared__ int cols[JP];
  __shared__ bool skip_pair;
  __shared__ double red[JT];

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int R = a.slices;
  const int pair = bid / R, slice = bid % R;
  const int xr = a.xrows_per, vr = a.vrows_per, tr = xr + vr;
  const int x_lo = min(a.m, slice * xr), x_hi = min(a.m, x_lo + xr);
  const int v_lo = min(a.n, slice * vr), v_hi = min(a.n, v_lo + vr);
  // 16-byte agent-coherent accesses to X, V and the partial Grams (every
  // offset of the tile path fits 31 bits: at most 16 slices of 192 rows and
  // 8192 columns)
  const __amdgpu_buffer_rsrc_t xrs =
      agent_rsrc(a.X, (unsigned)min((long)a.ldx * a.n * 16, 0x7fffffffL));
  const __amdgpu_buffer_rsrc_t vrs =
      agent_rsrc(a.V, (unsigned)min((long)a.ldv * a.n * 16, 0x7fffffffL));
  const __amdgpu_buffer_rsrc_t grs =
      agent_rsrc(a.gpart, (unsigned)min(2L * (a.nb / 2) * a.slices * (JP * JP) * 16, 0x7fffffffL));
  unsigned epoch = 0;
  const PairThread pt = pair_thread(R);

  // V = identity, Frobenius norm of X
  for (long e = bid * (long)JT + tid; e < (long)a.n * a.n; e += (long)nblk * JT) {
    const long i = e % a.n, j = e / a.n;
    st_agent(a.V + (i + j * a.ldv), make_double2(i == j ? 1.0 : 0.0, 0.0));
  }
  double part = 0.0;
  for (long e = bid * (long)JT + tid; e < (long)a.m * a.n; e += (long)nblk * JT) {
    const long i = e % a.m, j = e / a.m;
    part += cabs2(a.X[i + j * a.ldx]);
  }
  red[tid] = part;
  __syncthreads();
  for (int s = JT / 2; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) atomicAdd(a.fro2, red[0]);
  grid_barrier_all(a.bar, nblk, bid, epoch);
  // the pairs' Gram matrices are scaled with ||X||_F^2 (gram_scaling)
  const double fro2 = ld_agent(a.fro2);
  const double gsc = gram_scaling(fro2);
  const double tol2 = a.tol * a.tol;
  const double abs_tol2 = a.abs_tol_scale * a.abs_tol_scale * (fro2 * gsc);
  const int npairs = a.nb / 2;
  unsigned* pair_bar = a.bar + kBarrierWords;
  unsigned* pair_done = pair_bar + npairs;
  unsigned* blockver = pair_done + npairs;
  unsigned gen = 0, pair_epoch = 0;
  const int ntile = tr * JP;          // entries of the tile

  int sweep = 0;
  bool converged = false;
  for (; sweep < a.max_sweeps; ++sweep) {
    for (int round = 0; round < a.nb - 1; ++round) {
#ifdef PTE_ROUND_TRACE
      const int rt_round_ = sweep * (a.nb - 1) + round;
#endif
      RTRACE(0);
      int bi, bj;
      tournament_pair(a.nb, round, pair, bi, bj);
      if (tid < JP) {
        const int c = (tid < JB) ? bi * JB + tid : bj * JB + (tid - JB);
        cols[tid] = (c < a.n) ? c : -1;
      }
      // both blocks released by the pairs that held them in the previous round
      const int plo = min(bi, bj), phi = max(bi, bj);
      unsigned* const pair_ok = a.skip + a.nb + ((long)phi * (phi - 1)) / 2 + plo;
      if (tid == 0) {
        while (ld_agent(blockver + bi) < gen || ld_agent(blockver + bj) < gen)
          __builtin_amdgcn_s_sleep(1);
        const unsigned ok = ld_agent(pair_ok);
        skip_pair = ok != 0u && ld_agent(a.skip + bi) < ok && ld_agent(a.skip + bj) < ok;
      }
      __syncthreads();
      RTRACE(1);
      if (__builtin_amdgcn_readfirstlane((int)skip_pair)) {
        // the pair barrier is kept in a skipped round (see jacobi_body)
        if (R > 1) grid_barrier(pair_bar + pair, R, pair_epoch);
      } else {
        // ---- the slice's rows of X and V into the tile: entry e is row
        // e % tr of column e / tr, so that a wavefront reads runs of
        // consecutive rows of one column; every load of the tile is in
        // flight at once (at most kTileMaxRows * JP / JT per thread) ----
        {
          constexpr int kLoads = kTileMaxRows * JP / JT;
          double2 v[kLoads];
#pragma unroll
          for (int q = 0; q < kLoads; ++q) {
            const int e = tid + JT * q;
            const int row = e % tr, col = e / tr;
            v[q] = make_double2(0.0, 0.0);
            if (e < ntile && cols[col] >= 0) {
              if (row < xr) {
                if (x_lo + row < x_hi)
                  v[q] = ld_agent16(xrs, (unsigned)(x_lo + row + (long)cols[col] * a.ldx) * 16u);
              } else if (v_lo + row - xr < v_hi) {
                v[q] = ld_agent16(vrs, (unsigned)(v_lo + row - xr + (long)cols[col] * a.ldv) * 16u);
              }
            }
          }
#pragma unroll
          for (int q = 0; q < kLoads; ++q) {
            const int e = tid + JT * q;
            if (e < ntile) tile[(e % tr) * kTileLd + e / tr] = v[q];
          }
        }
        __syncthreads();
        // partial Grams are double-buffered by the parity of the pair
        // barrier's epoch before this round's barrier
        const double2* const gbuf =
            a.gpart + (long)(pair_epoch & 1) * npairs * R * (JP * JP) + (long)pair * R * (JP * JP);
        {
          const int I = wave >> 1, J = wave & 1;
          doublex4 p1 = {0.0, 0.0, 0.0, 0.0}, p2 = p1, p3 = p1;
          for (int k4 = 0; k4 < xr; k4 += 4) {
            const double2 x = tile[(k4 + lk) * kTileLd + 16 * I + lr];
            const double2 y = tile[(k4 + lk) * kTileLd + 16 * J + lr];
            const double ar = x.x, ai = -x.y;
            p1 = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, y.x, p1, 0, 0, 0);
            p2 = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, y.y, p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f64_16x16x4f64(ar + ai, y.x + y.y, p3, 0, 0, 0);
          }
          double2* mine = const_cast<double2*>(gbuf) + (long)slice * (JP * JP);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int gi = 16 * I + 4 * r + lk, gj = 16 * J + lr;
            const double2 g = make_double2(p1[r] - p2[r], p3[r] - p1[r] - p2[r]);
            if (R == 1) pair_store(Gp, pt, r, g, gsc);
            else st_agent16(grs, (unsigned)((mine - a.gpart) + gi * JP + gj) * 16u, g);
          }
        }
        if (R > 1) {
          RTRACE(2);
          grid_barrier(pair_bar + pair, R, pair_epoch);
          RTRACE(3);
          // identical summation order (slice 0, 1, ...) in every workgroup
          // of the pair; the loads of all slices (at most 16) in flight
          // together
          constexpr int SB = 16;
          double2 acc[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] = make_double2(0.0, 0.0);
          const double2* gp = gbuf;
          for (int sl0 = 0; sl0 < R; sl0 += SB) {
            double2 v[SB][4];
#pragma unroll
            for (int t = 0; t < SB; ++t)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                v[t][q] = (sl0 + t < R)
                              ? ld_agent16(grs, (unsigned)((gp - a.gpart) + (long)(sl0 + t) * (JP * JP) +
                                                           tid + JT * q) * 16u)
                              : make_double2(0.0, 0.0);
#pragma unroll
            for (int t = 0; t < SB; ++t)
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (sl0 + t < R) acc[q] = cadd(acc[q], v[t][q]);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) pair_store(Gp, pt, q, acc[q], gsc);
        }
        __syncthreads();
        const bool need = pair_needs(Gp, pt, tol2, abs_tol2);
        RTRACE(4);
        // record the outcome for later rounds: a rotated pair's blocks change,
        // an unrotated pair is converged as long as they do not
        if (slice == 0 && tid == 0) {
          if (need) {
            st_agent(a.skip + bi, gen + 1);
            st_agent(a.skip + bj, gen + 1);
            st_agent(pair_ok, 0u);
          } else {
            st_agent(pair_ok, gen + 1);
          }
        }
        if (need) {
          pair_sweeps(Gp, rot_c, rot_s, Ws, pt, tol2, abs_tol2, a.inner_sweeps);
          RTRACE(5);
          // ---- tile <- tile W on the matrix cores: B = W (lane: k = 4 k4 +
          // lk, column lr of the 16-column half v), A = 16 tile rows ----
          double wr[8][2], wi[8][2];
#pragma unroll
          for (int k4 = 0; k4 < 8; ++k4)
#pragma unroll
            for (int v = 0; v < 2; ++v) {
              const double2 w = Ws[4 * k4 + lk][16 * v + lr];
              wr[k4][v] = w.x;
              wi[k4][v] = w.y;
            }
          for (int t = wave; t < tr / 16; t += 4) {
            doublex4 p1[2], p2[2], p3[2];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
              p1[v] = doublex4{0.0, 0.0, 0.0, 0.0};
              p2[v] = p1[v];
              p3[v] = p1[v];
            }
#pragma unroll
            for (int k4 = 0; k4 < 8; ++k4) {
              const double2 x = tile[(16 * t + lr) * kTileLd + 4 * k4 + lk];
#pragma unroll
              for (int v = 0; v < 2; ++v) {
                p1[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x, wr[k4][v], p1[v], 0, 0, 0);
                p2[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.y, wi[k4][v], p2[v], 0, 0, 0);
                p3[v] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.x + x.y, wr[k4][v] + wi[k4][v],
                                                             p3[v], 0, 0, 0);
              }
            }
            // the wavefront's reads of these 16 rows are complete (in-order
            // LDS operations of one wavefront) before it overwrites them
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                tile[(16 * t + 4 * r + lk) * kTileLd + 16 * v + lr] =
                    make_double2(p1[v][r] - p2[v][r], p3[v][r] - p1[v][r] - p2[v][r]);
          }
          __syncthreads();
          // ---- the tile back, entry e as in the load ----
          for (int e = tid; e < ntile; e += JT) {
            const int row = e % tr, col = e / tr;
            const int gc = cols[col];
            if (gc < 0) continue;
            const double2 val = tile[row * kTileLd + col];
            if (row < xr) {
              if (x_lo + row < x_hi)
                st_agent16(xrs, (unsigned)(x_lo + row + (long)gc * a.ldx) * 16u, val);
            } else if (v_lo + row - xr < v_hi) {
              st_agent16(vrs, (unsigned)(v_lo + row - xr + (long)gc * a.ldv) * 16u, val);
            }
          }
          if (tid == 0) st_agent(a.flags + sweep, 1);
          RTRACE(6);
        }
      }   // skip_pair
      // the last slice of the pair to finish releases both blocks
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(pair_done + pair, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        if (old == (gen + 1) * (unsigned)R - 1) {
          st_agent(blockver + bi, gen + 1);
          st_agent(blockver + bj, gen + 1);
        }
      }
      ++gen;
      RTRACE(7);
    }
    grid_barrier_all(a.bar, nblk, bid, epoch);
    if (__hip_atomic_load(&a.flags[sweep], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
      converged = true;
      break;
    }
  }
  if (bid == 0 && tid == 0) *a.info = converged ? sweep + 1 : -1;
}

__global__ void __launch_bounds__(JT)
jacobi_tile_kernel(JacobiArgs a) {
  jacobi_tile_body(a, blockIdx.x, gridDim.x);
}

// Several independent SVDs in one cooperative launch of the LDS-tile
// Jacobi (problem map as in jacobi_batch_kernel; the dynamic LDS holds the
// largest problem's tile).
__global__ void __launch_bounds__(JT)
jacobi_tile_batch_kernel(const JacobiArgs* probs, const int* starts, const int* block_prob) {
  const int p = block_prob[blockIdx.x];
  const int s0 = starts[p];
  const JacobiArgs a = probs[p];
  jacobi_tile_body(a, blockIdx.x - s0, starts[p + 1] - s0);
}

// sigma_j = || X[:, j] ||  (one workgroup per column)
__device__ __forceinline__ void column_norm_body(const double2* X, int m, int n, long ldx,
                                                 double* sigma, int j) {
  __shared__ double red[256];
  if (j >= n) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < m; i += 256) s += cabs2(X[i + (long)j * ldx]);
  red[threadIdx.x] = s;
  __syncthreads();
  for (int t = 128; t > 0; t >>= 1) {
    if (threadIdx.x < t) red[threadIdx.x] += red[threadIdx.x + t];
    __syncthreads();
  }
  if (threadIdx.x == 0) sigma[j] = sqrt(red[0]);
}

__global__ void __launch_bounds__(256)
column_norm_kernel(const double2* X, int m, int n, long ldx, double* sigma) {
  column_norm_body(X, m, n, ldx, sigma, blockIdx.x);
}

// descending order, ties by index: perm[rank] = j, sorted[rank] = sigma[j]
__device__ __forceinline__ void rank_sort_body(const double* sigma, int n, int* perm,
                                               double* sorted, int j) {
  if (j >= n) return;
  const double sj = sigma[j];
  int rank = 0;
  for (int i = 0; i < n; ++i) {
    const double si = sigma[i];
    rank += (si > sj) || (si == sj && i < j);
  }
  perm[rank] = j;
  sorted[rank] = sj;
}

__global__ void __launch_bounds__(256)
rank_sort_kernel(const double* sigma, int n, int* perm, double* sorted) {
  rank_sort_body(sigma, n, perm, sorted, blockIdx.x * 256 + threadIdx.x);
}

// extra2: squared norm of a part of the matrix left out of `sorted` (the
// residual of a pivoted QR stopped at a rank cap), counted in every tail
__device__ __forceinline__ void truncate_body(const double* sorted, int n, double epsrel,
                                              SvdInfo* info, int max_rank, SvdInfo* copy,
                                              const double* extra2 = nullptr) {
  __shared__ double part[1024];
  __shared__ int cnt[1024];
  const int tid = threadIdx.x;
  const double base2 = extra2 ? *extra2 : 0.0;
  const int per = (n + 1023) / 1024;
  const int lo = min(n, tid * per), hi = min(n, lo + per);
  double s = 0.0;
  for (int i = lo; i < hi; ++i) s += sorted[i] * sorted[i];
  part[tid] = s;
  __syncthreads();
  // suffix sums of the per-thread partials (serial over 1024 values by thread 0)
  if (tid == 0) {
    double acc = base2;
    for (int t = 1023; t >= 0; --t) {
      const double v = part[t];
      part[t] = acc;        // sum of everything after thread t's segment
      acc += v;
    }
  }
  __syncthreads();
  const double s0 = (n > 0) ? sorted[0] : 0.0;
  const double thr = epsrel * s0;
  double tail = part[tid];
  int c = 0;
  for (int i = hi - 1; i >= lo; --i) {
    tail += sorted[i] * sorted[i];
    if (sqrt(tail) > thr) ++c;
  }
  cnt[tid] = c;
  __syncthreads();
  for (int t = 512; t > 0; t >>= 1) {
    if (tid < t) cnt[tid] += cnt[tid + t];
    __syncthreads();
  }
  if (tid == 0) {
    int k = cnt[0];
    info->rank = k;
    info->s0 = s0;
    info->overflow = (k > max_rank) ? 1 : 0;
    // discarded 2-norm
    double d = base2;
    for (int i = n - 1; i >= k; --i) d += sorted[i] * sorted[i];
    info->discarded = sqrt(d);
    if (copy) *copy = *info;
  }
}

__global__ void __launch_bounds__(1024)
truncate_kernel(const double* sorted, int n, double epsrel, SvdInfo* info,
                int max_rank, const double* extra2) {
  truncate_body(sorted, n, epsrel, info, max_rank, nullptr, extra2);
}

// ---- the same post-processing for many SVDs at once (problem = blockIdx.y,
// or blockIdx.x for the truncation); see SvdPostArgs ----
__global__ void __launch_bounds__(256)
column_norm_batch_kernel(const SvdPostArgs* pa) {
  const SvdPostArgs a = pa[blockIdx.y];
  column_norm_body(a.X, a.m, a.n, a.m, a.sigma, blockIdx.x);
}

__global__ void __launch_bounds__(256)
rank_sort_batch_kernel(const SvdPostArgs* pa) {
  const SvdPostArgs a = pa[blockIdx.y];
  rank_sort_body(a.sigma, a.n, a.perm, a.sorted, blockIdx.x * 256 + threadIdx.x);
}

// also gathers every SvdInfo into `out` for a single copy to the host
__global__ void __launch_bounds__(1024)
truncate_batch_kernel(const SvdPostArgs* pa, SvdInfo* out) {
  const SvdPostArgs a = pa[blockIdx.x];
  truncate_body(a.sorted, a.n, a.epsrel, a.info, a.max_rank, out + blockIdx.x);
}

// zero a list of device words (barrier counters, sweep flags): item = blockIdx.x
__global__ void __launch_bounds__(256)
zero_items_kernel(const ZeroItem* items) {
  const ZeroItem it = items[blockIdx.x];
  for (int i = threadIdx.x; i < it.words; i += 256) it.p[i] = 0u;
}

// out[i] = *probs[i].rank (pivoted-QR ranks for a single copy to the host)
__global__ void __launch_bounds__(256)
gather_qr_rank_kernel(const QrcpArgs* probs, int n, int* out) {
  for (int i = threadIdx.x; i < n; i += 256) out[i] = *probs[i].rank;
}



// ---------------------------------------------------------------------------
// Emission of the truncated factors. After the Jacobi on X = M^H (m' x n'):
// M = V Sigma (Z/Sigma)^H with Z the orthogonalised X. Left singular vector j
// of M is V[:, perm[j]]; Sigma * right^H row j is conj(Z[:, perm[j]]).
// ---------------------------------------------------------------------------
// dst[j*dj + a*da + b*db] = src[(a*B + b) + perm[j]*lds]     (conj if right)
// for a < A, b < B, j < k, with each stride d = d0 + dk * k. Left factors
// read V (no conjugation), Sigma*right^H rows read Z (conjugated).
__global__ void __launch_bounds__(256)
emit_kernel(EmitArgs a) {
  const int k = a.info->rank;
  const long dj = a.dj0 + a.djk * (long)k;
  const long da = a.da0 + a.dak * (long)k;
  const long db = a.db0 + a.dbk * (long)k;
  const int rows = a.A * a.B;
  const long total = (long)rows * k;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int s = e % rows;
    const int j = e / rows;
    const int c = a.rowmap ? a.rowmap[s] : s;
    const int aa = c / a.B, b = c % a.B;
    double2 v = a.src[s + (long)a.perm[j] * a.lds];
    if (a.conj) v.y = -v.y;
    a.dst[j * dj + aa * da + b * db] = v;
  }
}

// ---------------------------------------------------------------------------
// Householder QR with column pivoting (preconditioner of the Jacobi SVD).
// A (m x n, column-major, lda) -> A P = Q R with P the column permutation
// piv (piv[t] = physical column of step t), Q = H_0 ... H_{r-1},
// H_t = I - tau_t v_t v_t^H, v_t[t] = 1 and v_t[i] = A[i + piv[t]*lda] *
// vscale[t] for i > t (the pivot column keeps its unscaled entries),
// R[t][piv[t]] = beta[t] and R[t][c] = A[t + c*lda] for t above the diagonal.
// The reflector convention is LAPACK's zlarfg, the column-norm downdate with
// its cancellation guard is zlaqp2's. The factorisation stops at step r when
// the Frobenius norm of the unfactored block is at most drop * ||A||_F; the
// rows below r of R are dropped (a perturbation of that size).
// Column c belongs to workgroup c % gridDim.x; every workgroup forms the
// step's reflector from the pivot column itself, so workgroups wait for each
// other once per step: each posts its candidate (largest residual norm) and
// every one waits for all posts of the step and reduces them identically.
// A post is of 8-byte words that each carry the step's tag, so reading the
// posts is the waiting: no arrival counter stands between them (two dependent
// atomics and a separate read of the candidates less). A step at 380 x 108 takes
// 7.2 us on 27 workgroups (8.8 with the counters; 1.5 forming the reflector, 1.3
// updating the columns, 2.3 until their stores are acknowledged, 1.7 waiting for
// the posts), at 996 x 860 9.0 us on 215 (9.9). The posts are double-buffered by step parity: a workgroup
// posts step j + 2 after reading all posts of step j + 1, which were made after
// their workgroups had read step j's. They are zeroed before the launch (no
// step has tag 0).
// ---------------------------------------------------------------------------
// (value, column) maximum with ties to the smaller column; -1 = none
__device__ __forceinline__ void better(double& v, int& c, double ov, int oc) {
  if (oc >= 0 && (c < 0 || ov > v || (ov == v && oc < c))) { v = ov; c = oc; }
}

// Posts the workgroup's candidate of step j (see QrcpPost; wcol: number of the
// column among its own). Every wavefront waits for its own column stores first.
__device__ __forceinline__ void qrcp_post(const QrcpArgs& a, int blk, int nblk, int j, double wmax,
                                          int wcol, double wsum, double* cw_max, int* cw_col,
                                          double* cw_sum) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) { cw_max[wave] = wmax; cw_col[wave] = wcol; cw_sum[wave] = wsum; }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = -1.0, sm = 0.0;
    int c = -1;
    for (int w = 0; w < 4; ++w) {
      sm += cw_sum[w];
      better(v, c, cw_max[w], cw_col[w]);
    }
    QrcpPost post;
    post.norm = c >= 0 ? (unsigned long long)__double_as_longlong(v) : 0ull;
    post.sum = (unsigned long long)__double_as_longlong(sm);
    post.local = c >= 0 ? (unsigned)c : kQrNoColumn;
    const unsigned long long tag = qrcp_tag(j);
    const long at = (long)(j & 1) * nblk + blk;
    st_agent(a.cand + 2 * at, qrcp_word(post, 0, tag));
    st_agent(a.cand + 2 * at + 1, qrcp_word(post, 1, tag));
    st_agent(a.cand + 4 * nblk + at, qrcp_word(post, 2, tag));
  }
}

// Waits for the posts of step j and reduces them: the column of the largest
// norm (ties to the smaller column; -1: none) and the residual total, the same
// bits in every thread of the grid. The waits poll by atomic loads (the compiler
// may take a buffer load out of the loop).
__device__ __forceinline__ void qrcp_reduce(const QrcpArgs& a, int nblk, int j,
                                            double (*slot)[4], unsigned (*slotk)[4],
                                            unsigned (*slotc)[4], int (*slotn)[4], int& parity,
                                            int* bestc, double* total) {
  const unsigned long long tag = qrcp_tag(j);
  const long at = (long)(j & 1) * nblk + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr unsigned kNone = ~0u;
  // a workgroup without columns left has norm 0
  QrcpPost post{0ull, 0ull, kQrNoColumn};
  if ((int)threadIdx.x < nblk) {
    unsigned long long w0, w1;
    for (;;) {
      w0 = ld_agent(a.cand + 2 * at);
      w1 = ld_agent(a.cand + 2 * at + 1);
      if (qrcp_tagged(w0, tag) && qrcp_tagged(w1, tag)) break;
      __builtin_amdgcn_s_sleep(1);
    }
    post = qrcp_unpack(w0, w1);
  }
  const unsigned key = (unsigned)(post.norm >> 32);
  const unsigned col = post.local == kQrNoColumn ? kNone : threadIdx.x + post.local * nblk;
  const unsigned wkey = wave_max(key);
  const unsigned wcol = wave_min(key == wkey ? col : kNone);
  const int tied = __popcll(__ballot(key == wkey && col != kNone));
  if (lane == 0) {
    slotk[parity][wave] = wkey;
    slotc[parity][wave] = wcol;
    slotn[parity][wave] = tied;
  }
  // block_sum256 synchronises before reading, which also publishes the slots
  *total = block_sum256(__longlong_as_double((long long)post.sum), slot, parity);
  const int par = parity ^ 1;
  unsigned k = 0, c = kNone;
  int count = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const unsigned ok = slotk[par][w], oc = slotc[par][w];
    const int on = slotn[par][w];
    if (on > 0 && (count == 0 || ok > k)) { k = ok; c = oc; count = on; }
    else if (on > 0 && ok == k) { c = min(c, oc); count += on; }
  }
  if (__builtin_amdgcn_readfirstlane(count) > 1) {
    // upper halves tie: the lower ones of the tied workgroups
    unsigned low = 0;
    const bool mine = key == k && col != kNone;
    if (mine) {
      unsigned long long w2;
      for (;;) {
        w2 = ld_agent(a.cand + 4 * nblk + at);
        if (qrcp_tagged(w2, tag)) break;
        __builtin_amdgcn_s_sleep(1);
      }
      low = qrcp_norm_low(w2);
    }
    const unsigned wlow = wave_max(low);
    const unsigned wc = wave_min(mine && low == wlow ? col : kNone);
    __syncthreads();   // the slots above are read
    if (lane == 0) {
      slotk[par][wave] = wlow;
      slotc[par][wave] = wc;
    }
    __syncthreads();
    k = 0;
    c = kNone;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const unsigned ok = slotk[par][w], oc = slotc[par][w];
      if (oc != kNone && (c == kNone || ok > k || (ok == k && oc < c))) { k = ok; c = oc; }
    }
  }
  *bestc = __builtin_amdgcn_readfirstlane((int)c);
}

// loads of the pivoted QR issued together (per thread), and the rows of a
// column (per lane, times 64) kept in registers between its dot product and
// its update
constexpr int kQrBatch = 8;
constexpr int kQrCache = 16;

__device__ __forceinline__ void qrcp_body(const QrcpArgs& a, const int blk, const int nblk) {
  extern __shared__ double2 vcol[];            // reflector of the step (m)
  __shared__ double slot[2][4];
  __shared__ unsigned slotk[2][4], slotc[2][4];
  __shared__ int slotn[2][4];
  __shared__ double vn1[kQrcpMaxLocal], vn2[kQrcpMaxLocal];
  __shared__ int done[kQrcpMaxLocal];
  __shared__ double cw_max[4], cw_sum[4];
  __shared__ int cw_col[4];
  int parity = 0;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int m = a.m, n = a.n;
  const long lda = a.lda;
  const int kmax = m < n ? m : n;
  const int nloc = (n - blk + nblk - 1) / nblk;   // own columns blk, blk+nblk, ...

  // initial column norms (one wavefront per column); when resuming, the
  // norms of the unfactored rows start..m-1 of the columns not yet pivoted
  const int j0 = a.start;
  double wmax = -1.0, wsum = 0.0;
  int wcol = -1;
  // each wavefront keeps its first own column (q = wave) in registers for the
  // whole factorisation, rows lane + 64 u (u < kQrCache) at absolute row
  // indices (rows below the current step are left as they are); its
  // updates are still stored every step, for the pivot reads and the
  // factors. It stays resident until it is pivoted.
  double2 res[kQrCache];
  bool resident = false;
#pragma unroll
  for (int u = 0; u < kQrCache; ++u) res[u] = make_double2(0.0, 0.0);
  if (wave < nloc && !(j0 > 0 && ld_agent(a.done + blk + wave * nblk))) {
    const double2* col = a.A + (long)(blk + wave * nblk) * lda;
    const __amdgpu_buffer_rsrc_t crs = agent_rsrc(col, (unsigned)m * 16u);
#pragma unroll
    for (int u = 0; u < kQrCache; ++u) {
      const int i = lane + 64 * u;
      if (i >= j0 && i < m) res[u] = ld_agent16(crs, (unsigned)(i) * 16u);
    }
    resident = true;
  }
  for (int q = wave; q < nloc; q += 4) {
    const int c = blk + q * nblk;
    if (j0 > 0 && ld_agent(a.done + c)) {
      if (lane == 0) done[q] = 1;
      continue;
    }
    const double2* col = a.A + (long)c * lda;
    const __amdgpu_buffer_rsrc_t crs = agent_rsrc(col, (unsigned)m * 16u);
    double part = 0.0;
    for (int base = j0 + lane; base < m; base += 64 * kQrBatch) {
      double2 t[kQrBatch];
#pragma unroll
      for (int u = 0; u < kQrBatch; ++u) {
        const int i = base + 64 * u;
        t[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
      }
#pragma unroll
      for (int u = 0; u < kQrBatch; ++u) part += cabs2(t[u]);
    }
    const double nrm = sqrt(wave_sum(part));
    if (lane == 0) {
      vn1[q] = nrm; vn2[q] = nrm; done[q] = 0;
      if (j0 == 0) st_agent(a.done + c, 0);
    }
    wsum += nrm * nrm;
    better(wmax, wcol, nrm, q);   // (the workgroup's columns ascend with q)
  }
  qrcp_post(a, blk, nblk, j0, wmax, wcol, wsum, cw_max, cw_col, cw_sum);
  double total;
  int p;
  qrcp_reduce(a, nblk, j0, slot, slotk, slotc, slotn, parity, &p, &total);
  const double total0 = total;
  const double drop2 = j0 > 0 ? a.drop_abs2 : a.drop * a.drop * total;
  const double tol3z = 1.4901161193847656e-08;   // sqrt(eps), zlaqp2
  const int jmax =
      __builtin_amdgcn_readfirstlane(a.max_steps ? min(kmax, max(1, *a.max_steps)) : kmax);
  int j = j0;
  // mark: the first step count with residual^2 <= (mark_rel |beta_0|)^2;
  // every workgroup reduces the same candidates in the same order, so the
  // test (and a stop on it) is uniform over the grid
  int mark = -1;
  double mark2 = -1.0;
  if (a.mark_rel > 0.0 && j0 > 0) {
    const double b0 = a.mark_rel * fabs(a.beta[0]);
    mark2 = b0 * b0;
  }
  PHASE_INIT();
  // p, the step and the exit are the same in every lane, and scalar for the
  // compiler by the readfirstlanes (else the buffer descriptors of the columns
  // would be assembled lane by lane)
  while (j < jmax && p >= 0 && __builtin_amdgcn_readfirstlane((int)(total > drop2))) {
    // reflector j from the pivot column p (rows j..m-1), whole workgroup: the
    // column is read once into vcol (loads issued in batches, so that their
    // latencies overlap), then scaled in LDS
    const double2* pc = a.A + (long)p * lda;
    const __amdgpu_buffer_rsrc_t prs = agent_rsrc(pc, (unsigned)m * 16u);
    double part = 0.0;
    for (int base = j + tid; base < m; base += 256 * kQrBatch) {
      double2 t[kQrBatch];
#pragma unroll
      for (int q = 0; q < kQrBatch; ++q) {
        const int i = base + 256 * q;
        t[q] = (i < m) ? ld_agent16(prs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
      }
#pragma unroll
      for (int q = 0; q < kQrBatch; ++q) {
        const int i = base + 256 * q;
        if (i < m) {
          vcol[i] = t[q];
          if (i > j) part += cabs2(t[q]);
        }
      }
    }
    const double xnorm2 = block_sum256(part, slot, parity);
    const double2 alpha = vcol[j];
    double2 tau, scale;
    double beta;
    if (xnorm2 == 0.0 && alpha.y == 0.0) {
      tau = make_double2(0.0, 0.0);
      scale = make_double2(0.0, 0.0);
      beta = alpha.x;
    } else {
      beta = -copysign(sqrt(alpha.x * alpha.x + alpha.y * alpha.y + xnorm2), alpha.x);
      const double dr = alpha.x - beta, di = alpha.y;
      const double den = dr * dr + di * di;
      scale = make_double2(dr / den, -di / den);
      tau = make_double2((beta - alpha.x) / beta, -alpha.y / beta);
    }
    __syncthreads();   // every thread has read alpha = vcol[j]
    for (int i = j + tid; i < m; i += 256)
      vcol[i] = (i == j) ? make_double2(1.0, 0.0) : cmul(vcol[i], scale);
    if (blk == 0 && tid == 0) {
      a.piv[j] = p;
      a.tau[j] = tau;
      a.vscale[j] = scale;
      a.beta[j] = beta;
    }
    if (p % nblk == blk && tid == 0) {
      done[p / nblk] = 1;
      st_agent(a.done + p, 1);
    }
    if (p % nblk == blk && p / nblk == wave) resident = false;
    __syncthreads();
    PHASE(8);
    // apply H_j^H to the own remaining columns, downdate their norms
    const double2 tc = make_double2(tau.x, -tau.y);
    const bool reflect = (tau.x != 0.0 || tau.y != 0.0);
    wmax = -1.0; wsum = 0.0; wcol = -1;
    for (int q = wave; q < nloc; q += 4) {
      if (done[q]) continue;
      const int c = blk + q * nblk;
      double2* col = a.A + (long)c * lda;
      const __amdgpu_buffer_rsrc_t crs = agent_rsrc(col, (unsigned)m * 16u);
      if (q == wave && resident) {
        // the resident column: rows below 64 kQrCache from registers, the
        // rest (if any) streamed. The register rows are processed without
        // branches: rows outside [j, m) take a zero reflector entry (their
        // update is then exact: x - 0 = x); only the stores are predicated,
        // after all the arithmetic.
        const int beyond = max(j, 64 * kQrCache);
        if (reflect) {
          double2 vr[kQrCache];
          double2 w = make_double2(0.0, 0.0);
#pragma unroll
          for (int u = 0; u < kQrCache; ++u) {
            const int i = lane + 64 * u;
            const double2 vi = vcol[min(i, m - 1)];
            vr[u] = (i >= j && i < m) ? vi : make_double2(0.0, 0.0);
            cfmac(w, vr[u], res[u]);
          }
          for (int base = beyond + lane; base < m; base += 64 * kQrBatch) {
            double2 t[kQrBatch];
#pragma unroll
            for (int u = 0; u < kQrBatch; ++u) {
              const int i = base + 64 * u;
              t[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int u = 0; u < kQrBatch; ++u) {
              const int i = base + 64 * u;
              if (i < m) cfmac(w, vcol[i], t[u]);
            }
          }
          w.x = wave_sum(w.x);
          w.y = wave_sum(w.y);
          const double2 tw = cmul(tc, w);
#pragma unroll
          for (int u = 0; u < kQrCache; ++u) res[u] = csub(res[u], cmul(vr[u], tw));
#pragma unroll
          for (int u = 0; u < kQrCache; ++u) {
            const int i = lane + 64 * u;
            if (i >= j && i < m) st_agent16(crs, (unsigned)(i) * 16u, res[u]);
          }
          for (int base = beyond + lane; base < m; base += 64 * kQrBatch) {
            double2 t[kQrBatch];
#pragma unroll
            for (int u = 0; u < kQrBatch; ++u) {
              const int i = base + 64 * u;
              t[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
            }
#pragma unroll
            for (int u = 0; u < kQrBatch; ++u) {
              const int i = base + 64 * u;
              if (i < m) st_agent16(crs, (unsigned)(i) * 16u, csub(t[u], cmul(vcol[i], tw)));
            }
          }
        }
        // row j of the updated column: register j / 64 of lane j % 64 (or
        // memory beyond the registers)
        double2 rj2 = make_double2(0.0, 0.0);
        if (j < 64 * kQrCache) {
#pragma unroll
          for (int u = 0; u < kQrCache; ++u)
            if (u == (j >> 6)) rj2 = res[u];
          rj2.x = __shfl(rj2.x, j & 63, 64);
          rj2.y = __shfl(rj2.y, j & 63, 64);
        } else {
          __threadfence_block();
          rj2 = ld_agent16(crs, (unsigned)(j) * 16u);
        }
        double nv = vn1[q];
        if (nv != 0.0) {
          const double rj = sqrt(cabs2(rj2));
          double temp = 1.0 - (rj / nv) * (rj / nv);
          temp = temp > 0.0 ? temp : 0.0;
          const double ratio = nv / vn2[q];
          const double temp2 = temp * ratio * ratio;
          if (temp2 <= tol3z) {
            // recompute the norm of rows j+1.. from the registers and, beyond
            // them, from memory (this lane's own stores: complete them before
            // reading back)
            __threadfence_block();
            double pp = 0.0;
#pragma unroll
            for (int u = 0; u < kQrCache; ++u) {
              const int i = lane + 64 * u;
              if (i > j && i < m) pp += cabs2(res[u]);
            }
            for (int i = max(j + 1, 64 * kQrCache) + lane; i < m; i += 64)
              pp += cabs2(ld_agent16(crs, (unsigned)(i) * 16u));
            nv = (j + 1 < m) ? sqrt(wave_sum(pp)) : 0.0;
            if (lane == 0) { vn1[q] = nv; vn2[q] = nv; }
          } else {
            nv = nv * sqrt(temp);
            if (lane == 0) vn1[q] = nv;
          }
        }
        wsum += nv * nv;
        better(wmax, wcol, nv, q);
        continue;
      }
      // rows j .. j + 64 kQrCache - 1 stay in registers between the dot
      // product and the update; all loads are issued in batches
      double2 cache[kQrCache];
#pragma unroll
      for (int u = 0; u < kQrCache; ++u) {
        const int i = j + lane + 64 * u;
        cache[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
      }
      if (reflect) {
        double2 w = make_double2(0.0, 0.0);
#pragma unroll
        for (int u = 0; u < kQrCache; ++u) {
          const int i = j + lane + 64 * u;
          if (i < m) cfmac(w, vcol[i], cache[u]);
        }
        for (int base = j + lane + 64 * kQrCache; base < m; base += 64 * kQrBatch) {
          double2 t[kQrBatch];
#pragma unroll
          for (int u = 0; u < kQrBatch; ++u) {
            const int i = base + 64 * u;
            t[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
          }
#pragma unroll
          for (int u = 0; u < kQrBatch; ++u) {
            const int i = base + 64 * u;
            if (i < m) cfmac(w, vcol[i], t[u]);
          }
        }
        w.x = wave_sum(w.x);
        w.y = wave_sum(w.y);
        const double2 tw = cmul(tc, w);
#pragma unroll
        for (int u = 0; u < kQrCache; ++u) {
          const int i = j + lane + 64 * u;
          if (i < m) {
            cache[u] = csub(cache[u], cmul(vcol[i], tw));
            st_agent16(crs, (unsigned)(i) * 16u, cache[u]);
          }
        }
        for (int base = j + lane + 64 * kQrCache; base < m; base += 64 * kQrBatch) {
          double2 t[kQrBatch];
#pragma unroll
          for (int u = 0; u < kQrBatch; ++u) {
            const int i = base + 64 * u;
            t[u] = (i < m) ? ld_agent16(crs, (unsigned)(i) * 16u) : make_double2(0.0, 0.0);
          }
#pragma unroll
          for (int u = 0; u < kQrBatch; ++u) {
            const int i = base + 64 * u;
            if (i < m) st_agent16(crs, (unsigned)(i) * 16u, csub(t[u], cmul(vcol[i], tw)));
          }
        }
      }
      // row j of the updated column sits in lane 0's first cached entry
      double2 rj2 = cache[0];
      rj2.x = __shfl(rj2.x, 0, 64);
      rj2.y = __shfl(rj2.y, 0, 64);
      double nv = vn1[q];
      if (nv != 0.0) {
        const double rj = sqrt(cabs2(rj2));
        double temp = 1.0 - (rj / nv) * (rj / nv);
        temp = temp > 0.0 ? temp : 0.0;
        const double ratio = nv / vn2[q];
        const double temp2 = temp * ratio * ratio;
        if (temp2 <= tol3z) {
          // recompute the norm of rows j+1.. from the cached entries and,
          // beyond them, from memory (this lane's own stores: complete them
          // before reading back)
          __threadfence_block();
          double pp = 0.0;
#pragma unroll
          for (int u = 0; u < kQrCache; ++u) {
            const int i = j + lane + 64 * u;
            if (i > j && i < m) pp += cabs2(cache[u]);
          }
          for (int i = j + lane + 64 * kQrCache; i < m; i += 64) pp += cabs2(ld_agent16(crs, (unsigned)(i) * 16u));
          nv = (j + 1 < m) ? sqrt(wave_sum(pp)) : 0.0;
          if (lane == 0) { vn1[q] = nv; vn2[q] = nv; }
        } else {
          nv = nv * sqrt(temp);
          if (lane == 0) vn1[q] = nv;
        }
      }
      wsum += nv * nv;
      better(wmax, wcol, nv, q);
    }
    PHASE(9);
    ++j;
    qrcp_post(a, blk, nblk, j, wmax, wcol, wsum, cw_max, cw_col, cw_sum);
    PHASE(10);
    qrcp_reduce(a, nblk, j, slot, slotk, slotc, slotn, parity, &p, &total);
    PHASE(12);
    if (a.mark_rel > 0.0) {
      if (j == 1) {
        const double b0 = a.mark_rel * fabs(beta);
        mark2 = b0 * b0;
      }
      if (mark < 0 && __builtin_amdgcn_readfirstlane((int)(total <= mark2))) {
        mark = j;
        if (a.stop_at_mark) break;
      }
    }
  }
  // remaining columns in ascending order after the pivots
  if (blk == 0 && tid == 0) {
    int t = j;
    for (int c = 0; c < n; ++c)
      if (!ld_agent(a.done + c)) a.piv[t++] = c;
    *a.rank = j;
    if (a.out) {
      a.out[0] = (p >= 0 && j < kmax) ? total : 0.0;
      if (j0 == 0) a.out[1] = total0;
      a.out[2] = j > 0 ? fabs(a.beta[0]) : 0.0;
      a.out[3] = (double)(mark >= 0 ? mark : j);
    }
  }
}

__global__ void __launch_bounds__(256)
qrcp_kernel(QrcpArgs a) {
  qrcp_body(a, blockIdx.x, gridDim.x);
}

// Several pivoted QRs in one cooperative launch (see jacobi_batch_kernel).
__global__ void __launch_bounds__(256)
qrcp_batch_kernel(const QrcpArgs* probs, const int* starts, const int* block_prob) {
  const int p = block_prob[blockIdx.x];
  const int s0 = starts[p];
  const QrcpArgs a = probs[p];
  qrcp_body(a, blockIdx.x - s0, starts[p + 1] - s0);
}

// Y = R^H (n x r, column-major, ld = n) in the pivoted column order:
// Y[s + t*n] = conj(R[t][piv[s]])
__device__ __forceinline__ void build_rh_body(const double2* A, long lda, int n,
                                              const int* piv, const double* beta,
                                              const int* rank, double2* Y, int bid,
                                              int nblocks) {
  const int r = *rank;
  const long total = (long)n * r;
  for (long e = bid * 256L + threadIdx.x; e < total; e += (long)nblocks * 256) {
    const int s = e % n;
    const int t = e / n;
    double2 v = make_double2(0.0, 0.0);
    if (t < s) v = cconj(A[t + (long)piv[s] * lda]);
    else if (t == s) v = make_double2(beta[s], 0.0);
    Y[e] = v;
  }
}

__global__ void __launch_bounds__(256)
build_rh_kernel(const double2* A, long lda, int n, const int* piv, const double* beta,
                const int* rank, double2* Y) {
  build_rh_body(A, lda, n, piv, beta, rank, Y, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(256)
build_rh_batch_kernel(const RhArgs* pa) {
  const RhArgs a = pa[blockIdx.y];
  build_rh_body(a.A, a.lda, a.n, a.piv, a.beta, a.rank, a.Y, blockIdx.x, gridDim.x);
}

// ---------------------------------------------------------------------------
// Small truncated SVD in one workgroup (M with at most kSmallMaxCols columns and
// kSmallRows rows per lane of a column, see small_lanes): the pivoted QR with
// M in registers (small_qr), then the Jacobi of Y = R^H (n x r) on its Gram
// matrix in LDS (below), singular values, order and cut.
// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// Jacobi SVD of Y = R^H (n x r, r <= kGramMaxRank) of a pivoted QR in one
// workgroup, on the Gram matrix.
//
// One-sided Jacobi rotates columns of Y, and of the accumulated W, and takes
// three inner products of length n per pair and round to find each rotation.
// Here a pass finds the rotations on G = Y^H Y (formed on the FP64 matrix
// cores) by two-sided rotations in LDS: a pair's three entries are read, not
// summed. They are applied to the rows of Y and of W afterwards, by as many
// wavefronts as there are rows (gram_replay_kernel), from a log of every round's
// rotations. Then the next pass forms G anew, from the rotated Y. The SVD is done
// when such a fresh G needs no rotation: that is the stopping rule of
// jacobi_kernel on the inner products of Y's own columns, and the singular
// values are their norms.
//
// The rows of R fall off with the pivots, G = D A D with D their norms. Where A
// is well conditioned, Jacobi keeps the small entries of such a matrix to high
// relative accuracy (Demmel and Veselic, 1992), and the second pass only checks.
// A pivoted QR does not guarantee that: on Kahan's matrix of 100 columns (A of
// condition 1e12) the roots of the first pass's diagonal are off by 2e-11 of the
// largest. Its Y is nearly orthogonal all the same, so that one sweep of a second
// pass settles the pairs that are left (2 to 7 of thousands, as of some matrices
// with a flat spectrum), and its columns' norms are right to rounding.
//
// The order is the round-robin of P = ceil(r / 2) pairs: position 2q holds the
// pair's first column a_q, position 2q + 1 its second, b_q; position 0 keeps
// its column and the others move on by one position a round (gram_next), so
// that after re - 1 rounds (re = 2P) every two columns have met and all are
// back. G is kept by positions, as the P (P + 1) / 2 blocks (q1, q2), q1 <= q2,
// of 2 x 2 entries (the Hermitian half; 129 KB of LDS at r = 126), entry e of
// every block in a plane of its own. A round is
//   (1) every thread reads the blocks it owns; wavefront 0, one pair per lane,
//       computes the rotations from the diagonal blocks, to LDS and to the log;
//   (2) every thread rotates its blocks from both sides, J_q1^H B J_q2, and
//       writes each entry where its columns are in the next round,
// with a barrier after each. Reads and writes go to addresses that are the same
// in every round: no index arithmetic, and reads without bank conflicts. (By
// columns, with the packed triangle's indices computed every round, that
// arithmetic alone took longer than the rotations: 1.5 us a round at r = 83.)
// The padding column of an odd r is zero and stays so. A sweep starts with a
// test of all pairs; a pass without a sweep is the check.
// Rotation: (x_a, x_b) <- (c x_a - conj(s) x_b, s x_a + c x_b), s carrying the
// phase of g_ab.
// Bound by the chain of a round in one compute unit: LDS reads, about 60
// dependent FP64 operations of a rotation, the blocks' 48 each, LDS writes.
// 88 x 83 matrix in small_svd_kernel, QR included: 0.78 ms, the replay 0.06, the
// check 0.025, against 1.83 ms with one-sided sweeps in LDS. (Against
// jacobi_tile_kernel after the grid's QR: the host's rule has both sides.)
// ---------------------------------------------------------------------------
// 16 x 16 tile t of the upper triangle of Y^H Y (list (0,0), (0,1), (1,1),
// (0,2), ...) by one wavefront, 3M on the FP64 matrix cores; Y is n x r with
// leading dimension ld. Lane l gets rows 4 q + l / 16 of column l % 16.
__device__ __forceinline__ void gram_tile_index(int t, int& I, int& J) {
  J = 0;
  while ((J + 1) * (J + 2) / 2 <= t) ++J;
  I = t - J * (J + 1) / 2;
}

__device__ __forceinline__ void gram_tile(const double2* Y, long ld, int n, int r, int t,
                                          double2 (&g)[4]) {
  const int lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  int I, J;
  gram_tile_index(t, I, J);
  const int ci = 16 * I + lr, cj = 16 * J + lr;
  const double2* yi = Y + (long)min(ci, r - 1) * ld;
  const double2* yj = Y + (long)min(cj, r - 1) * ld;
  doublex4 p1 = {0.0, 0.0, 0.0, 0.0}, p2 = p1, p3 = p1;
  // four slices of four rows loaded together
  for (int k4 = 0; k4 < n; k4 += 16) {
    double2 x[4], y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = k4 + 4 * q + lk;
      x[q] = yi[min(k, n - 1)];
      y[q] = yj[min(k, n - 1)];
      if (k >= n || ci >= r) x[q] = make_double2(0.0, 0.0);
      if (k >= n || cj >= r) y[q] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      p1 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q].x, y[q].x, p1, 0, 0, 0);
      p2 = __builtin_amdgcn_mfma_f64_16x16x4f64(-x[q].y, y[q].y, p2, 0, 0, 0);
      p3 = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q].x - x[q].y, y[q].x + y[q].y, p3, 0, 0, 0);
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) g[q] = make_double2(p1[q] - p2[q], p3[q] - p1[q] - p2[q]);
}

// that tile into G (zeroed before: the padding column has no entries)
__device__ __forceinline__ void gram_store(double2* G, int r, int t, const double2 (&g)[4]) {
  const int lane = threadIdx.x & 63;
  const int lr = lane & 15, lk = lane >> 4;
  const int P = (r + 1) / 2, T = P * (P + 1) / 2;
  int I, J;
  gram_tile_index(t, I, J);
  const int j = 16 * J + lr;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = 16 * I + 4 * q + lk;
    if (i > j || j >= r) continue;
    bool conj;
    const int at = gram_place(gram_pos(i, P), gram_pos(j, P), T, conj);
    const double im = i == j ? 0.0 : g[q].y;
    G[at] = make_double2(g[q].x, conj ? -im : im);
  }
}

// Two-sided Jacobi sweeps on G (rank r) in LDS; rc, rs: LDS scratch of 64
// rotations; NB: blocks per thread, at least T / NT. Returns the sweeps done: none if no
// pair needs a rotation, max_sweeps also where some pair still does.
template <int NT, int NB>
__device__ __forceinline__ int gram_jacobi(double2* G, int r, double tol2, double abs_tol2,
                                           int max_sweeps, double* rc, double2* rs,
                                           double* logc, double2* logs) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int P = (r + 1) / 2, L = 2 * P - 1;
  const int T = P * (P + 1) / 2;
  int q1[NB], q2[NB];      // own blocks tid, tid + NT, ... (q1 = -1: none)
  // places of the entries in the next round, 15 bits each, and in bit 15 the
  // conjugation: entries 0 and 1 in dst[u][0], 2 and 3 in dst[u][1]
  unsigned dst[NB][2];
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int b = tid + u * NT;
    int c = 0;
    if (b < T) {
      c = (int)((sqrtf(8.0f * (float)b + 1.0f) - 1.0f) * 0.5f);
      while ((c + 1) * (c + 2) / 2 <= b) ++c;
      while (c * (c + 1) / 2 > b) --c;
    }
    q2[u] = c;
    q1[u] = b < T ? b - c * (c + 1) / 2 : -1;
    dst[u][0] = dst[u][1] = 0;
    if (q1[u] >= 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bool conj = false;
        const int at = gram_place(gram_next(2 * q1[u] + (e >> 1), P),
                                  gram_next(2 * q2[u] + (e & 1), P), T, conj);
        dst[u][e >> 1] |= ((unsigned)at | (conj ? 0x8000u : 0u)) << (16 * (e & 1));
      }
    }
  }
  auto put = [&](unsigned place, double2 v) {   // place in the upper 16 bits
    v.y = __hiloint2double(__double2hiint(v.y) ^ (int)(place & 0x80000000u),
                           __double2loint(v.y));
    G[(place >> 16) & 0x7fffu] = v;
  };
  int sweeps = 0;
  for (;;) {
    int mine = 0;
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if (q1[u] < 0) continue;
      const int b = tid + u * NT, b1 = gram_block(q1[u], q1[u]), b2 = gram_block(q2[u], q2[u]);
      const double da1 = G[b1].x, db1 = G[3 * T + b1].x;
      const double da2 = G[b2].x, db2 = G[3 * T + b2].x;
      bool any = needs_rotation(da1, db2, cabs2(G[T + b]), tol2, abs_tol2);
      if (q1[u] != q2[u]) {
        any |= needs_rotation(da1, da2, cabs2(G[b]), tol2, abs_tol2);
        any |= needs_rotation(db1, da2, cabs2(G[2 * T + b]), tol2, abs_tol2);
        any |= needs_rotation(db1, db2, cabs2(G[3 * T + b]), tol2, abs_tol2);
      }
      if (any) mine = 1;
    }
    if (!__syncthreads_or(mine) || sweeps == max_sweeps) break;
    for (int t = 0; t < L; ++t) {
      double2 b00[NB], b01[NB], b10[NB], b11[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int b = q1[u] >= 0 ? tid + u * NT : 0;
        b00[u] = G[b];
        b01[u] = G[T + b];
        b10[u] = G[2 * T + b];
        b11[u] = G[3 * T + b];
      }
      if (wave == 0) {
        const bool valid = lane < P;
        const int d = gram_block(min(lane, P - 1), min(lane, P - 1));
        double c;
        double2 sn;
        gram_rotation(valid, G[d].x, G[3 * T + d].x, G[T + d], tol2, abs_tol2, c, sn);
        c = unit_c(c, sn);
        if (valid) {
          rc[lane] = c;
          rs[lane] = sn;
          const long e = (long)(sweeps * L + t) * 64 + lane;
          logc[e] = c;
          logs[e] = sn;
        }
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (q1[u] >= 0) {
          const double c1 = rc[q1[u]], c2 = rc[q2[u]];
          const double2 s1 = rs[q1[u]], s2 = rs[q2[u]];
          const double2 s1c = cconj(s1), s2c = cconj(s2);
          const bool diag = q1[u] == q2[u];
          if (diag) b10[u] = cconj(b01[u]);
          const double2 n00 = csub(cscale(b00[u], c2), cmul(s2c, b01[u]));
          const double2 n01 = cadd(cmul(s2, b00[u]), cscale(b01[u], c2));
          const double2 n10 = csub(cscale(b10[u], c2), cmul(s2c, b11[u]));
          const double2 n11 = cadd(cmul(s2, b10[u]), cscale(b11[u], c2));
          double2 m00 = csub(cscale(n00, c1), cmul(s1, n10));
          double2 m01 = csub(cscale(n01, c1), cmul(s1, n11));
          const double2 m10 = cadd(cmul(s1c, n00), cscale(n10, c1));
          double2 m11 = cadd(cmul(s1c, n01), cscale(n11, c1));
          if (diag) {
            m00.y = 0.0;
            m11.y = 0.0;
            // a rotated pair is diagonal
            if (s1.x != 0.0 || s1.y != 0.0) m01 = make_double2(0.0, 0.0);
          } else {
            put(dst[u][1] << 16, m10);
          }
          put(dst[u][0] << 16, m00);
          put(dst[u][0], m01);
          put(dst[u][1], m11);
        }
      }
      __syncthreads();
    }
    ++sweeps;
  }
  return sweeps;
}

// squared norm of column c (after whole sweeps)
__device__ __forceinline__ double gram_diag(const double2* G, int c, int r) {
  const int P = (r + 1) / 2, T = P * (P + 1) / 2;
  const int x = gram_pos(c, P), q = x >> 1;
  return G[((x & 1) ? 3 * T : 0) + gram_block(q, q)].x;
}

// Scales G by an even power of two that brings its trace to [1, 4), so that
// the squares of its entries in the rotations' tests stay in range; returns the
// scaled trace, and in *half half the exponent taken out (sigma = sqrt(g_cc)
// 2^half). Called by the whole workgroup after a barrier; ends with one.
template <int NT>
__device__ __forceinline__ double gram_scale(double2* G, int r, int* half) {
  double tr = 0.0;
  for (int i = threadIdx.x & 63; i < r; i += 64) tr += gram_diag(G, i, r);
  tr = wave_sum(tr);          // the same bits in every wavefront
  *half = 0;
  if (!(tr > 0.0 && tr < 1.7e308)) return tr;
  *half = ilogb(tr) >> 1;
  const int P = (r + 1) / 2;
  __syncthreads();
  for (int e = threadIdx.x; e < 2 * P * (P + 1); e += NT) {
    const double2 v = G[e];
    G[e] = make_double2(ldexp(v.x, -2 * *half), ldexp(v.y, -2 * *half));
  }
  __syncthreads();
  return ldexp(tr, -2 * *half);
}

// LDS of the Gram Jacobi: G, 64 rotations, three r-vectors
__device__ __host__ constexpr int gram_entries(int r) {
  return 4 * (((r + 1) / 2) * ((r + 1) / 2 + 1) / 2);
}

// Singular values (roots of G's diagonal), descending order and cut, by the
// whole workgroup; s_sig, s_sorted, s_tail: LDS, r entries each, outside G.
// extra2: squared weight left out of G, counted in every tail (valid in every
// thread of wavefront 0).
template <int NT>
__device__ __forceinline__ void gram_finish(const double2* G, int r, double epsrel,
                                            int max_rank, double extra2, int sweeps, int half,
                                            double* s_sig,
                                            double* s_sorted, double* s_tail, double* sigma,
                                            int* perm, double* sorted, SvdInfo* info,
                                            SvdInfo* copy) {
  const int tid = threadIdx.x, lane = tid & 63;
  int bad = 0;
  if (tid < r) {
    const double d = gram_diag(G, tid, r);
    bad = !(d < 1.7e308);                     // not a number, or overflowed
    const double sg = ldexp(sqrt(fmax(d, 0.0)), half);
    s_sig[tid] = sg;
    sigma[tid] = sg;
  }
  bad = __syncthreads_or(bad);
  if (tid < r && !bad) {
    const double sj = s_sig[tid];
    int rank = 0;
    for (int i = 0; i < r; ++i) {
      const double si = s_sig[i];
      rank += (si > sj) || (si == sj && i < tid);
    }
    perm[rank] = tid;
    sorted[rank] = sj;
    s_sorted[rank] = sj;
  }
  __syncthreads();
  if (tid >= 64) return;
  // tails sum_{i >= j} s_i^2 of the two values of each lane: suffix scan of
  // the lane sums; k = #{j: sqrt(tail_j) > epsrel s_0}
  const int i0 = 2 * lane, i1 = i0 + 1;
  const double v0 = i0 < r && !bad ? s_sorted[i0] * s_sorted[i0] : 0.0;
  const double v1 = i1 < r && !bad ? s_sorted[i1] * s_sorted[i1] : 0.0;
  double x = v0 + v1;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_down(x, off, 64);
    if (lane + off < 64) x += o;
  }
  double after = __shfl_down(x, 1, 64);
  if (lane == 63) after = 0.0;
  const double t1 = after + v1 + extra2, t0 = after + (v0 + v1) + extra2;
  const double s0 = bad ? 0.0 : s_sorted[0];
  const double thr = epsrel * s0;
  const int k = bad ? 0 : __popcll(__ballot(i0 < r && sqrt(t0) > thr)) +
                          __popcll(__ballot(i1 < r && sqrt(t1) > thr));
  if (i0 < r) s_tail[i0] = t0;
  if (i1 < r) s_tail[i1] = t1;
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    SvdInfo inf;
    inf.rank = k;
    inf.overflow = k > max_rank ? 1 : 0;
    inf.sweeps = sweeps + 1;
    inf.pad = r;
    inf.s0 = s0;
    inf.discarded = sqrt(k < r ? s_tail[k] : extra2);
    inf.rounds = 0;
    inf.state = kGramDone;
    *info = inf;
    if (copy) *copy = inf;
  }
}

// Rest of a pass after the Gram matrix, `before` sweeps after the start: the
// whole workgroup of NT threads, NB blocks of G per thread at most.
template <int NT, int NB, class Args>
__device__ __forceinline__ void gram_run(const Args& a, double2* G, int n, int r,
                                         double extra2, int before) {
  double2* rs = G + gram_entries(r);
  double* rc = reinterpret_cast<double*>(rs + 64);
  double* s_sig = rc + 64;
  int half;
  const double tr = gram_scale<NT>(G, r, &half);
  const double eps = 2.220446049250313e-16;
  const double tol = (n > 16 ? n : 16) * eps;
  const int sweeps = gram_jacobi<NT, NB>(G, r, tol * tol, eps * eps * tr, a.max_sweeps, rc, rs,
                                         a.logc, a.logs);
  if (sweeps > 0) {
    if (threadIdx.x == 0) {
      SvdInfo inf = {};
      inf.sweeps = before + sweeps;
      inf.pad = r;
      inf.rounds = sweeps * (max(2, r + (r & 1)) - 1);
      inf.state = kGramRotated;
      *a.info = inf;
      if (a.copy) *a.copy = inf;
    }
    return;
  }
  gram_finish<NT>(G, r, a.epsrel, a.max_rank, extra2, before, half, s_sig, s_sig + r,
                  s_sig + 2 * r, a.sigma, a.perm, a.sorted, a.info, a.copy);
}

// 1024 threads at ranks above kGramSmallRank: there the rotations' FP64 issue and
// the LDS traffic of G set the time of a round, not its barriers (112: 1.35 us a
// round, 1.7 us with 512 threads; 74: 0.92 us and 0.96; 35: 0.68 us and 0.64).
template <int NT>
__device__ __forceinline__ void gram_svd_body(const GramSvdArgs& a) {
  extern __shared__ double2 lds_gram[];
  int rank = a.r, before = 0;
  if (a.expect) {
    const SvdInfo inf = *a.info;
    if (inf.state != a.expect) return;
    rank = inf.pad;
    before = inf.sweeps;
  }
  const int r = __builtin_amdgcn_readfirstlane(rank);
  double2* G = lds_gram;
  for (int e = threadIdx.x; e < gram_entries(r); e += NT) G[e] = make_double2(0.0, 0.0);
  __syncthreads();
  const int nb = (r + 15) / 16;
  for (int t = threadIdx.x >> 6; t < nb * (nb + 1) / 2; t += NT / 64) {
    double2 g[4];
    gram_tile(a.Y, a.n, a.n, r, t, g);
    gram_store(G, r, t, g);
  }
  __syncthreads();
  // 990 blocks at rank 88, 2016 at rank 126
  gram_run<NT, 2>(a, G, a.n, r, a.extra2 ? *a.extra2 : 0.0, before);
}

template <int NT>
__global__ void __launch_bounds__(NT)
gram_svd_kernel(GramSvdArgs a) {
  gram_svd_body<NT>(a);
}
template __global__ void gram_svd_kernel<kSmallThreads>(GramSvdArgs);
template __global__ void gram_svd_kernel<kGramThreads>(GramSvdArgs);

template <int NT>
__global__ void __launch_bounds__(NT)
gram_svd_batch_kernel(const GramSvdArgs* probs) {
  const GramSvdArgs a = probs[blockIdx.x];
  gram_svd_body<NT>(a);
}
template __global__ void gram_svd_batch_kernel<kSmallThreads>(const GramSvdArgs*);
template __global__ void gram_svd_batch_kernel<kGramThreads>(const GramSvdArgs*);

// wavefront shifts by one lane: lane i reads lane i + 1 (down) or i - 1 (up)
constexpr int kDppWaveShl1 = 0x130, kDppWaveShr1 = 0x138;
template <int CTRL>
__device__ __forceinline__ double2 dpp_d2(double2 v) {
  return make_double2(dpp_d<CTRL>(v.x), dpp_d<CTRL>(v.y));
}

// Applies the logged rotations to the rows of Y (in place) and of W (r x r, the
// identity in the first pass), one wavefront per row. Lane q holds the entries of
// the row in columns a_q and b_q; going to the next round of the round-robin
// moves every a one lane down and every b one lane up (a_0 stays, b of the
// last lane turns into its a, a_1 into b_0), so that a round is 12 FMAs and
// register moves, with no LDS, no barrier and no column index; after whole
// sweeps every entry is back in its column. The rounds' rotations are the
// same for all rows (L2) and are loaded four rounds ahead. 0.05 us a round.
__device__ __forceinline__ void gram_replay_body(const GramReplayArgs& a, int row) {
  const SvdInfo inf = *a.info;
  const int r = inf.pad, n = a.n;
  if (inf.state != kGramRotated && !(a.first && inf.state == kGramDone)) return;
  if (r < 1 || row >= n + r) return;
  const int lane = threadIdx.x & 63;
  const int re = max(2, r + (r & 1)), P = re / 2, L = re - 1;
  const double2 zero = make_double2(0.0, 0.0);
  const int ca = lane == 0 ? L : lane, cb = lane == 0 ? 0 : L - lane;
  const bool oa = lane < P && ca < r, ob = lane < P && cb < r;
  const bool isy = row < n;
  double2 xa = zero, xb = zero;
  if (isy) {
    if (oa) xa = a.Y[row + (long)ca * n];
    if (ob) xb = a.Y[row + (long)cb * n];
  } else if (a.first) {
    if (oa && ca == row - n) xa.x = 1.0;
    if (ob && cb == row - n) xb.x = 1.0;
  } else {
    if (oa) xa = a.W[row - n + (long)ca * r];
    if (ob) xb = a.W[row - n + (long)cb * r];
  }
  const int rounds = inf.rounds;
  const int le = min(lane, P - 1);
  constexpr int PFR = 4;
  double nc[PFR];
  double2 ns[PFR];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int u = 0; u < PFR; ++u) {
      const long e = (long)min(t0 + u, rounds - 1) * 64 + le;
      nc[u] = a.logc[e];
      ns[u] = a.logs[e];
    }
  };
  if (rounds > 0) fetch(0);
  for (int t0 = 0; t0 < rounds; t0 += PFR) {
    double c[PFR];
    double2 s[PFR];
#pragma unroll
    for (int u = 0; u < PFR; ++u) { c[u] = nc[u]; s[u] = ns[u]; }
    if (t0 + PFR < rounds) fetch(t0 + PFR);
#pragma unroll
    for (int u = 0; u < PFR; ++u) {
      if (t0 + u < rounds) {
        // the small term first, so that a component is rounded once at its own
        // size: fma(c, x, s y) in place of fma(s, y, c x)
        const double2 ta = cmul(make_double2(-s[u].x, s[u].y), xb), tb = cmul(s[u], xa);
        const double2 ya = make_double2(fma(c[u], xa.x, ta.x), fma(c[u], xa.y, ta.y));
        const double2 yb = make_double2(fma(c[u], xb.x, tb.x), fma(c[u], xb.y, tb.y));
        if (P > 1) {
          const double2 down = dpp_d2<kDppWaveShl1>(ya), up = dpp_d2<kDppWaveShr1>(yb);
          xa = lane == 0 ? ya : (lane == P - 1 ? yb : down);
          xb = lane == 0 ? down : up;
        } else {
          xa = ya;
          xb = yb;
        }
      }
    }
  }
  if (isy) {
    if (oa) a.Y[row + (long)ca * n] = xa;
    if (ob) a.Y[row + (long)cb * n] = xb;
  } else {
    if (oa) a.W[row - n + (long)ca * r] = xa;
    if (ob) a.W[row - n + (long)cb * r] = xb;
  }
}

__global__ void __launch_bounds__(256)
gram_replay_kernel(GramReplayArgs a) {
  gram_replay_body(a, blockIdx.x * 4 + (threadIdx.x >> 6));
}

__global__ void __launch_bounds__(256)
gram_replay_batch_kernel(const GramReplayArgs* probs) {
  const GramReplayArgs a = probs[blockIdx.y];
  gram_replay_body(a, blockIdx.x * 4 + (threadIdx.x >> 6));
}

// ---------------------------------------------------------------------------
// Pivoted Householder QR of M (m x n) with M in registers: G = 2^lg lanes per
// column (small_lanes), lane g of a group holding rows g + G u, u < RP. The
// reflectors (zlarfg) and the eps-rank stop are qrcp_kernel's; the residual
// norms are summed anew in every step (two FMAs a row, in place of the
// downdate's square root and division and of a pass over the pivot column), and
// the pivot is the first column with the largest one. A step:
//   (1) each group has the norm, first entry and reflector scalars of its
//       remaining rows; each wavefront posts its largest column to LDS; barrier;
//   (2) every wavefront picks the winner of the posts; the winner's group
//       writes its column to LDS; barrier;
//   (3) every group applies the reflector to its column.
// Row j (row u = j / G of lane j % G) is taken out of the registers before step
// j and stored as R's when the step is done, so registers of finished rows are
// zero: the inner product, the update and the norm run over all RP rows without
// masks or branches, and the pivot column is copied to LDS whole, as
// [u][64 lanes]. (Skipping the finished rows took 1550 instructions a step at
// 12 rows a lane, two thirds of them branches, masks and register copies.) The
// reflector is used unscaled, its scale (vscale, as in the factors of
// qrcp_kernel) folded into the scalars. All of it fits 256 VGPRs up to 38 rows a
// lane, with no scratch, as the reflector's rows are read eight at a time and the
// scalars of the whole factorisation lie in LDS (with 40 rows, and a branch after
// those reads, which let the compiler gather them all before it, 448 bytes a lane
// were spilled and a step at 160 x 126 took 12 us).
// 512 threads: a workgroup barrier costs 86 cycles with 8 wavefronts, 326 with
// 16 and 11 with 4, and 256 threads would not hold M.
// Bound by the chain of a step (two barriers, two passes through LDS, the
// reductions and the reflector's scalars): 1.7 us a step at 24 x 24, 1.9 at
// 40 x 44, 2.8 at 88 x 83, where M in LDS took 3.0, 3.2 and 4.4.
// ---------------------------------------------------------------------------
struct SmallCand {
  double2 tau, scale;
  double sum, beta;
  double norm2;      // squared norm
  int col;
  int pad;
};
constexpr int kSmallWaves = kSmallThreads / 64;
static_assert(kSmallWaves == 8, "the posts are reduced over groups of 8 lanes");
static_assert(64 * kSmallRows * 16 + kSmallWaves * (int)sizeof(SmallCand) +
                  2 * 128 * (int)sizeof(int) + 2 * (int)sizeof(double) <=
                  (int)kSmallQrLds, "LDS of the QR");

__device__ __forceinline__ double larger(double a, double b) { return b > a ? b : a; }
template <int HALF>
__device__ __forceinline__ double swap_larger(double v) {
  double lo, hi;
  swap_d<HALF>(v, lo, hi);
  return larger(lo, hi);
}

template <int RP>
__device__ __forceinline__ int small_qr(const SmallSvdArgs& a, const int lg, double2* vcol,
                                        SmallCand* cand, int* s_piv, int* s_done,
                                        double* s_stop, double& folded2) {
  // up to 24 rows the reflector's rows stay in registers between the inner
  // product and the update, else they are read again
  constexpr bool kKeep = RP <= 24;
  const int m = a.m, n = a.n, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int G = 1 << lg;
  const int myc = tid >> lg, g = tid & (G - 1);
  const double eps = 2.220446049250313e-16;
  const int kmax = min(m, n);
  bool alive = myc < n;
  double2 col[RP];
#pragma unroll
  for (int u = 0; u < RP; ++u) {
    const int i = g + G * u;
    col[u] = make_double2(0.0, 0.0);
    if (alive && i < m) col[u] = a.A[i + (long)myc * m];
  }
  for (int c = tid; c < n; c += kSmallThreads) s_done[c] = 0;
  // takes row jn out (cj: its entry, in the lane that held it), then the norm,
  // reflector scalars and post of step jn
  double2 cj = make_double2(0.0, 0.0);
  auto post = [&](int jn) __attribute__((always_inline)) {
    const int uj = jn >> lg;
    const bool here = alive && g == (jn & (G - 1));
    cj = make_double2(0.0, 0.0);
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      if (u == uj) {
        cj = make_double2(here ? col[u].x : 0.0, here ? col[u].y : 0.0);
        col[u] = make_double2(here ? 0.0 : col[u].x, here ? 0.0 : col[u].y);
      }
    }
    double tail = 0.0, tail1 = 0.0, ax = cj.x, ay = cj.y;
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      tail = fma(col[u].x, col[u].x, tail);
      tail1 = fma(col[u].y, col[u].y, tail1);
    }
    tail += tail1;
    double z = 0.0;
    group_sum4(tail, ax, ay, z, G);
    const double norm2 = alive ? tail + fma(ax, ax, ay * ay) : 0.0;
    // largest column of the wavefront: its norms are the same bits in all lanes
    // of a group, so the first lane with the largest one is lane 0 of a group
    double big = norm2, sv = norm2;
    if (G <= 4) { big = larger(big, dpp_d<kDppHalfMirror>(big)); sv += dpp_d<kDppHalfMirror>(sv); }
    if (G <= 8) { big = larger(big, dpp_d<kDppMirror>(big)); sv += dpp_d<kDppMirror>(sv); }
    if (G <= 16) { big = swap_larger<16>(big); sv = swap_sum<16>(sv); }
    if (G <= 32) { big = swap_larger<32>(big); sv = swap_sum<32>(sv); }
    const unsigned long long at = __ballot(alive && norm2 == big);
    double beta = ax;
    double2 tau = make_double2(0.0, 0.0), scale = make_double2(0.0, 0.0);
    if (tail != 0.0 || ay != 0.0) {
      beta = -copysign(sqrt(norm2), ax);
      const double dr = ax - beta;
      const double den = fma(dr, dr, ay * ay);
      scale = make_double2(dr / den, -ay / den);
      tau = make_double2(-dr / beta, -ay / beta);
    }
    if (lane == (at ? __ffsll(at) - 1 : 0)) {
      SmallCand* cd = cand + wave;
      cd->tau = tau;
      cd->scale = scale;
      cd->sum = sv;
      cd->beta = beta;
      cd->norm2 = big;
      cd->col = at ? myc : -1;
    }
  };
  post(0);
  SEG_INIT();
  bool folded = false;
  double total;
  int j = 0;
  for (;;) {
    __syncthreads();
    SEG(0);
    // the posts, replicated in every group of 8 lanes; ties go to the first
    // wavefront, whose columns are the smaller ones
    const SmallCand* cl = cand + (lane & (kSmallWaves - 1));
    const int mcol = cl->col;
    const double wnorm2 = cl->norm2;
    total = cl->sum;
    double big = wnorm2;
    big = larger(big, dpp_d<kDppXor1>(big));
    total += dpp_d<kDppXor1>(total);
    big = larger(big, dpp_d<kDppXor2>(big));
    total += dpp_d<kDppXor2>(total);
    big = larger(big, dpp_d<kDppHalfMirror>(big));
    total += dpp_d<kDppHalfMirror>(total);
    const unsigned long long at = __ballot(mcol >= 0 && wnorm2 == big);
    const int ws = at ? __ffsll(at) - 1 : 0;          // wavefront of the winner
    const int p = at ? __builtin_amdgcn_readlane(mcol, ws) : -1;
    // residual test; an adaptive stop (stop_rel > 0) ends at a residual of
    // stop_rel * |beta_0| and counts it in the cut
    // (both thresholds are kept in LDS, from step 0 on)
    const double drop2 = j == 0 ? eps * eps * total : s_stop[0];
    bool go = j < kmax && p >= 0 && total > drop2;
    folded = a.stop_rel > 0.0 && j >= 1 && total <= s_stop[1];
    if (folded) {
      folded = p >= 0 && j < kmax;
      go = false;
    }
    // (the same in every lane; said so, so that the loop, its step and all that
    // hangs on them stay in scalar registers and scalar branches)
    if (!__builtin_amdgcn_readfirstlane((int)go)) break;
    const SmallCand* cw = cand + ws;
    const double2 tau = cw->tau, scale = cw->scale;
    if (j == 0 && tid == 0) {
      s_stop[0] = drop2;
      s_stop[1] = (a.stop_rel * cw->beta) * (a.stop_rel * cw->beta);
    }
    if (alive && myc == p) {
#pragma unroll
      for (int u = 0; u < RP; ++u) vcol[64 * u + g] = col[u];
      alive = false;
      if (g == 0) {
        s_piv[j] = p;
        s_done[p] = j + 1;
        a.tau[j] = tau;
        a.vscale[j] = scale;
        a.beta[j] = cw->beta;
      }
    }
    SEG(1);
    __syncthreads();
    SEG(2);
    if (alive) {
      double2 pv[kKeep ? RP : 1];
      double2 S = make_double2(0.0, 0.0);
#pragma unroll
      for (int u = 0; u < RP; ++u) {
        const double2 v = vcol[64 * u + g];
        if constexpr (kKeep) pv[u] = v;
        cfmac(S, v, col[u]);
        // at most eight rows of the reflector in flight beside M's registers
        if (!kKeep && u % 8 == 7) __builtin_amdgcn_sched_barrier(0);
      }
      double2 w = cadd(cj, cmulc(scale, S));
      double z0 = 0.0, z1 = 0.0;
      group_sum4(w.x, w.y, z0, z1, G);
      const double2 tw = cmulc(tau, w);
      const double2 sv2 = cmul(scale, tw);
      SEG(3);
      if (g == (j & (G - 1))) a.A[j + (long)myc * m] = csub(cj, tw);
      if (!kKeep) asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < RP; ++u) {
        double2 v;
        if constexpr (kKeep) v = pv[u];
        else v = vcol[64 * u + g];
        cfma(col[u], make_double2(-v.x, -v.y), sv2);
        if (!kKeep && u % 8 == 7) __builtin_amdgcn_sched_barrier(0);
      }
    }
    ++j;
    SEG(4);
    post(j);
    SEG(5);
  }
  folded2 = folded ? total : 0.0;
  SEG_FLUSH(0, 6);
  // reflectors to global memory (apply_q_kernel reads them)
  const int myt = myc < n ? s_done[myc] - 1 : -1;    // step that took the own column
  if (myt >= 0) {
    // (opaque copy: the indices and masks of the loads above would otherwise be
    // kept in registers through the loop for reuse here)
    int g2 = g;
    asm volatile("" : "+v"(g2));
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      const int i = g2 + G * u;
      if (i > myt && i < m) a.A[i + (long)myc * m] = col[u];
    }
  }
  // remaining columns in ascending order after the pivots
  if (wave == 0) {
    const bool r0 = lane < n && !s_done[lane], r1 = lane + 64 < n && !s_done[lane + 64];
    const unsigned long long b0 = __ballot(r0), b1 = __ballot(r1);
    const unsigned long long below = (1ull << lane) - 1ull;
    if (r0) s_piv[j + __popcll(b0 & below)] = lane;
    if (r1) s_piv[j + __popcll(b0) + __popcll(b1 & below)] = lane + 64;
  }
  if (tid == 0) *a.qrank = j;
  __syncthreads();
  for (int t = tid; t < n; t += kSmallThreads) a.piv[t] = s_piv[t];
  return j;
}

__device__ __forceinline__ void small_svd_body(const SmallSvdArgs& a) {
  constexpr int NT = kSmallThreads;
  extern __shared__ double2 lds_small[];
  const int m = a.m, n = a.n, tid = threadIdx.x, wave = tid >> 6;
  // QR phase: the pivot column, the posts, pivots and done flags
  double2* vcol = lds_small;
  SmallCand* cand = reinterpret_cast<SmallCand*>(vcol + 64 * kSmallRows);
  int* s_piv = reinterpret_cast<int*>(cand + kSmallWaves);
  int* s_done = s_piv + 128;
  double* s_stop = reinterpret_cast<double*>(s_done + 128);
  PHASE_INIT();
  const int lg = __builtin_amdgcn_readfirstlane(31 - __clz(small_lanes(n)));
  const int rows = (m + (1 << lg) - 1) >> lg;
  double folded2;
  const int steps = rows <= 4 ? small_qr<4>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2)
                : rows <= 8  ? small_qr<8>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2)
                : rows <= 16 ? small_qr<16>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2)
                : rows <= 24 ? small_qr<24>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2)
                : rows <= 32 ? small_qr<32>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2)
                             : small_qr<kSmallRows>(a, lg, vcol, cand, s_piv, s_done, s_stop, folded2);
  PHASE(13);
  const int r = __builtin_amdgcn_readfirstlane(steps);
  if (r == 0) {
    if (tid == 0) {
      SvdInfo inf;
      inf.rank = 0; inf.overflow = 0; inf.sweeps = 1; inf.pad = 0;
      inf.s0 = 0.0; inf.discarded = 0.0;
      inf.rounds = 0; inf.state = kGramDone;
      *a.info = inf;
      if (a.copy) *a.copy = inf;
    }
    return;
  }
  // ---- Y = R^H (n x r) to global memory; G from it on the matrix cores, by
  // way of LDS where Y fits it (odd leading dimension: the tile loads step
  // over columns), else from global memory; G replaces Y in LDS ----
  for (long e = tid; e < (long)n * r; e += NT) {
    const int sidx = e % n, t = e / n;
    double2 v = make_double2(0.0, 0.0);
    if (t < sidx) v = cconj(a.A[t + (long)s_piv[sidx] * m]);
    else if (t == sidx) v = make_double2(a.beta[sidx], 0.0);
    a.Y[e] = v;
  }
  __syncthreads();
  if (tid == 0 && a.folded) *a.folded = folded2;
  if (r > kGramSmallRank) {
    // gram_svd_kernel goes on from Y
    if (tid == 0) {
      a.info->sweeps = 0;
      a.info->pad = r;
      a.info->state = kGramFresh;
    }
    return;
  }
  double2* Gm = lds_small;
  const int nb = (r + 15) / 16, tiles = nb * (nb + 1) / 2;
  const int ldy = n | 1;
  if ((long)ldy * r * (long)sizeof(double2) <= a.lds_bytes) {
    double2* Ys = lds_small;
    for (long e = tid; e < (long)n * r; e += NT) Ys[e % n + (e / n) * ldy] = a.Y[e];
    __syncthreads();
    constexpr int kTiles = 3;                 // of the 21 at rank 88, 8 wavefronts
    double2 g[kTiles][4];
#pragma unroll
    for (int u = 0; u < kTiles; ++u)
      if (wave + u * (NT / 64) < tiles) gram_tile(Ys, ldy, n, r, wave + u * (NT / 64), g[u]);
    __syncthreads();
    for (int e = tid; e < gram_entries(r); e += NT) Gm[e] = make_double2(0.0, 0.0);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kTiles; ++u)
      if (wave + u * (NT / 64) < tiles) gram_store(Gm, r, wave + u * (NT / 64), g[u]);
  } else {
    for (int e = tid; e < gram_entries(r); e += NT) Gm[e] = make_double2(0.0, 0.0);
    __syncthreads();
    for (int t = wave; t < tiles; t += NT / 64) {
      double2 g[4];
      gram_tile(a.Y, n, n, r, t, g);
      gram_store(Gm, r, t, g);
    }
  }
  __syncthreads();
  // one block per thread up to rank 62 (496 blocks), two at 88 (990)
  if (r <= 62) gram_run<NT, 1>(a, Gm, n, r, folded2, 0);
  else gram_run<NT, 2>(a, Gm, n, r, folded2, 0);
  PHASE(14);
}

__global__ void __launch_bounds__(kSmallThreads)
small_svd_kernel(SmallSvdArgs a) {
  small_svd_body(a);
}

__global__ void __launch_bounds__(kSmallThreads)
small_svd_batch_kernel(const SmallSvdArgs* probs) {
  const SmallSvdArgs a = probs[blockIdx.x];
  small_svd_body(a);
}

// Left singular vectors Q W[:, perm[j]] (j < k) of the pivoted QR, the
// reflectors applied from the last to the first to a column held in LDS;
// row i = a*B + b goes to dst[j*dj + a*da + b*db].
// One column per workgroup, the reflector entries of each step loaded into
// registers in one batch (rows t + tid + 256 u, u < kApplyQRegs; rows beyond
// on demand) and those of the next step issued before this step's
// reduction, so that their latency overlaps the work.
constexpr int kApplyQRegs = 8;

__global__ void __launch_bounds__(256)
apply_q_kernel(ApplyQArgs a) {
  extern __shared__ double2 cvec[];
  __shared__ double slot[2][4], sloti[2][4];
  int parity = 0;
  const int tid = threadIdx.x;
  const int k = a.info->rank;
  const int r = *a.qrank;
  const int m = a.m;
  const long dj = a.dj0 + a.djk * (long)k;
  const long da = a.da0 + a.dak * (long)k;
  const long db = a.db0 + a.dbk * (long)k;
  for (int j = blockIdx.x; j < k; j += gridDim.x) {
    const double2* w = a.W + (long)a.perm[j] * a.ldw;
    for (int i = tid; i < m; i += blockDim.x)
      cvec[i] = (i < r) ? w[i] : make_double2(0.0, 0.0);
    __syncthreads();
    // reflector t's entries (unscaled) for rows t + tid + 256 u
    double2 vn[kApplyQRegs];
    auto fetch = [&](int t) {
      const double2* v = a.A + (long)a.piv[t] * a.lda;
#pragma unroll
      for (int u = 0; u < kApplyQRegs; ++u) {
        const int i = t + tid + 256 * u;
        vn[u] = (i < m) ? v[i] : make_double2(0.0, 0.0);
      }
    };
    if (r > 0) fetch(r - 1);
    for (int t = r - 1; t >= 0; --t) {
      double2 vc[kApplyQRegs];
#pragma unroll
      for (int u = 0; u < kApplyQRegs; ++u) vc[u] = vn[u];
      const double2 tau = a.tau[t];
      const double2 sc = a.vscale[t];
      const double2* v = a.A + (long)a.piv[t] * a.lda;
      if (t > 0) fetch(t - 1);
      if (tau.x == 0.0 && tau.y == 0.0) continue;
      double2 acc = make_double2(0.0, 0.0);
#pragma unroll
      for (int u = 0; u < kApplyQRegs; ++u) {
        const int i = t + tid + 256 * u;
        if (i < m) {
          vc[u] = (i == t) ? make_double2(1.0, 0.0) : cmul(vc[u], sc);
          cfmac(acc, vc[u], cvec[i]);
        }
      }
      for (int i = t + tid + 256 * kApplyQRegs; i < m; i += blockDim.x) {
        const double2 vi = cmul(v[i], sc);
        cfmac(acc, vi, cvec[i]);
      }
      const double2 tw = cmul(tau, block_sum256c(acc, slot, sloti, parity));
#pragma unroll
      for (int u = 0; u < kApplyQRegs; ++u) {
        const int i = t + tid + 256 * u;
        if (i < m) cvec[i] = csub(cvec[i], cmul(vc[u], tw));
      }
      for (int i = t + tid + 256 * kApplyQRegs; i < m; i += blockDim.x) {
        const double2 vi = cmul(v[i], sc);
        cvec[i] = csub(cvec[i], cmul(vi, tw));
      }
      __syncthreads();
    }
    for (int i = tid; i < m; i += blockDim.x) {
      const int aa = i / a.B, b = i % a.B;
      a.dst[(long)j * dj + (long)aa * da + (long)b * db] = cvec[i];
    }
    __syncthreads();
  }
}

// The same for Q of at most 64 RP rows: one wavefront per column, rows lane +
// 64 u (u < RP) in registers, wavefront reductions only (no barrier, no LDS);
// a reflector is loaded two steps ahead (one at RP = 16), and the batches of rows
// above the reflector are passed over. Against a workgroup per column: all of a
// TEMPO run's with 200 to 500 rows 23.5 -> 15.7 ms, 996 x 860 1.24 -> 1.13 ms; the
// registers (and the gain) end at 1024 rows.
template <int RP>
__global__ void __launch_bounds__(256)
apply_q_wave_kernel(ApplyQArgs a) {
  const int lane = threadIdx.x & 63;
  const int j = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int k = a.info->rank;
  if (j >= k) return;   // a whole wavefront; the kernel has no barrier
  const int r = __builtin_amdgcn_readfirstlane(*a.qrank);
  const int m = a.m;
  const double2* w = a.W + (long)a.perm[j] * a.ldw;
  double2 x[RP], next[2][RP];
#pragma unroll
  for (int u = 0; u < RP; ++u) {
    const int i = lane + 64 * u;
    const double2 wi = w[max(min(i, r - 1), 0)];
    x[u] = make_double2(i < r ? wi.x : 0.0, i < r ? wi.y : 0.0);
    next[0][u] = next[1][u] = make_double2(0.0, 0.0);
  }
  // are rows 64 u .. 64 u + 63 above row t (a batch that reflector t leaves)
  auto above = [&](int u, int t) __attribute__((always_inline)) {
    return RP > 2 && 64 * (u + 1) <= t;
  };
  // row m - 1 of the reflector in place of rows beyond m (not used)
  auto fetch = [&](int t, int p, double2 (&to)[RP]) __attribute__((always_inline)) {
    const double2* v = a.A + (long)p * a.lda;
#pragma unroll
    for (int u = 0; u < RP; ++u)
      if (!above(u, t)) to[u] = v[min(lane + 64 * u, m - 1)];
  };
  constexpr int D = RP <= 8 ? 2 : 1;   // steps from a load to its use
  int piv = 0;                         // of reflector t - D
  double2 tau = make_double2(0.0, 0.0), sc = tau;
  auto step = [&](int t, double2 (&buf)[RP]) __attribute__((always_inline)) {
    double2 v[RP];
#pragma unroll
    for (int u = 0; u < RP; ++u) v[u] = buf[u];
    const double2 tau_t = tau, sc_t = sc;
    if (t >= D) fetch(t - D, piv, buf);
    tau = a.tau[max(t - 1, 0)];
    sc = a.vscale[max(t - 1, 0)];
    piv = a.piv[max(t - D - 1, 0)];
    if (tau_t.x == 0.0 && tau_t.y == 0.0) return;
    double2 acc = make_double2(0.0, 0.0), acc2 = acc;
#pragma unroll
    for (int u = 0; u < RP; ++u) {
      if (above(u, t)) continue;
      const int i = lane + 64 * u;
      const double2 y = cmul(v[u], sc_t);
      const bool in = i > t && i < m;
      v[u] = make_double2(i == t ? 1.0 : (in ? y.x : 0.0), in ? y.y : 0.0);
      if (u & 1) cfmac(acc2, v[u], x[u]);
      else cfmac(acc, v[u], x[u]);
    }
    double re = acc.x + acc2.x, im = acc.y + acc2.y, z0 = 0.0, z1 = 0.0;
    group_sum4(re, im, z0, z1, 64);
    const double2 tw = cmul(tau_t, make_double2(re, im));
#pragma unroll
    for (int u = 0; u < RP; ++u)
      if (!above(u, t)) x[u] = csub(x[u], cmul(v[u], tw));
  };
  if (r > 0) {
    fetch(r - 1, a.piv[r - 1], next[0]);
    if (D == 2 && r > 1) fetch(r - 2, a.piv[r - 2], next[1]);
    tau = a.tau[r - 1];
    sc = a.vscale[r - 1];
    piv = a.piv[max(r - 1 - D, 0)];
  }
  int t = r - 1;
  if (D == 2)
    for (; t >= 1; t -= 2) {
      step(t, next[0]);
      step(t - 1, next[1]);
    }
  for (; t >= 0; --t) step(t, next[0]);
  const long dj = a.dj0 + a.djk * (long)k;
  const long da = a.da0 + a.dak * (long)k;
  const long db = a.db0 + a.dbk * (long)k;
#pragma unroll
  for (int u = 0; u < RP; ++u) {
    const int i = lane + 64 * u;
    if (i < m) a.dst[(long)j * dj + (long)(i / a.B) * da + (long)(i % a.B) * db] = x[u];
  }
}
template __global__ void apply_q_wave_kernel<2>(ApplyQArgs);
template __global__ void apply_q_wave_kernel<4>(ApplyQArgs);
template __global__ void apply_q_wave_kernel<8>(ApplyQArgs);
template __global__ void apply_q_wave_kernel<16>(ApplyQArgs);

__global__ void __launch_bounds__(256)
finite_check_kernel(const double2* x, long count, int* flag) {
  bool bad = false;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < count; e += (long)gridDim.x * 256) {
    const double2 v = x[e];
    bad |= !(isfinite(v.x) && isfinite(v.y));
  }
  if (bad) *flag = 1;
}

// X (rows x cols, column-major, ld = rows) = conj(src) with src row-major
// (cols x rows): X[r + c*rows] = conj(src[c*rows + r]) -- a plain conjugate
__global__ void __launch_bounds__(256)
conj_copy_kernel(const double2* src, long count, double2* dst) {
  for (long e = blockIdx.x * 256L + threadIdx.x; e < count; e += (long)gridDim.x * 256)
    dst[e] = cconj(src[e]);
}

// X[r + c*R] = conj(src[r*C + c])  (src row-major R x C)
__global__ void __launch_bounds__(256)
conj_transpose_kernel(const double2* src, int R, int C, double2* dst) {
  const long total = (long)R * C;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int r = e % R;
    const long c = e / R;
    dst[e] = cconj(src[(long)r * C + c]);
  }
}

// X[r + c*R] = src[r*C + c]: row-major R x C to column-major
__global__ void __launch_bounds__(256)
transpose_kernel(const double2* src, int R, int C, double2* dst) {
  const long total = (long)R * C;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int r = e % R;
    const long c = e / R;
    dst[e] = src[(long)r * C + c];
  }
}

// out[i] = sum_j in[j*stride_j ... ] : contract one leg of a tensor [a][p][b]
// with a vector: out[a][b] = sum_p T[a][p][b] * vec[p]
__global__ void __launch_bounds__(256)
leg_vector_kernel(const double2* T, int A, int P, int B, const double2* vec,
                  double2* out) {
  const long total = (long)A * B;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int b = e % B;
    const long aa = e / B;
    double2 acc = make_double2(0.0, 0.0);
    for (int p = 0; p < P; ++p) cfma(acc, T[(aa * P + p) * B + b], vec[p]);
    out[e] = acc;
  }
}

__global__ void __launch_bounds__(256)
identity_carry_kernel(double2* dst, int R, int V) {
  // dst[(r*X + x)*V + v] = delta(x, r*V + v), X = R*V
  const int X = R * V;
  const long total = (long)R * X * V;
  for (long e = blockIdx.x * 256L + threadIdx.x; e < total; e += (long)gridDim.x * 256) {
    const int v = e % V;
    const long t = e / V;
    const int x = t % X;
    const int r = t / X;
    dst[e] = make_double2(x == r * V + v ? 1.0 : 0.0, 0.0);
  }
}

}  // namespace pte

#ifdef PTE_ROUND_TRACE
// per-round timestamp readout (n entries at most); clears the buffer
extern "C" int pte_debug_round_trace(unsigned long long* out, long n) {
  const long total = (long)pte::kRtRounds * pte::kRtBlocks * pte::kRtMarks;
  if (n > total) n = total;
  if (hipDeviceSynchronize() != hipSuccess) return -3;
  if (hipMemcpyFromSymbol(out, HIP_SYMBOL(pte::g_rtrace), sizeof(unsigned long long) * n) !=
      hipSuccess)
    return -3;
  void* dev = nullptr;
  if (hipGetSymbolAddress(&dev, HIP_SYMBOL(pte::g_rtrace)) != hipSuccess) return -3;
  if (hipMemset(dev, 0, sizeof(unsigned long long) * total) != hipSuccess) return -3;
  if (hipDeviceSynchronize() != hipSuccess) return -3;
  return 0;
}
#endif

#ifdef PTE_PHASE_TIMING
// phase timer readout (s_memrealtime ticks); resets the timers
extern "C" int pte_debug_phases(unsigned long long* out) {
  if (hipDeviceSynchronize() != hipSuccess) return -3;
  if (hipMemcpyFromSymbol(out, HIP_SYMBOL(pte::g_phase), sizeof(unsigned long long) * 16) !=
      hipSuccess)
    return -3;
  unsigned long long z[16] = {0};
  if (hipMemcpyToSymbol(HIP_SYMBOL(pte::g_phase), z, sizeof(z)) != hipSuccess) return -3;
  return 0;
}
#endif
