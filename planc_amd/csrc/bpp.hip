// Batched block-principal-pivoting NNLS in FP64: min ||A x - b||, x >= 0,
// given the normal equations G = A^T A (k x k, k <= 64) and right-hand sides
// b = A^T a (one per column).  Restates BPPNNLS::solveNNLSMultipleRHS
// (nnls/bppnnls.hpp:67-191) column by column: each column's pivoting
// (P, Ninf, exchange rules Cols1 / Cols2 / backup rule, 1e-12 clamps) is
// independent of the other columns, so the reference's chunk-wide loop and
// its grouping of equal passive sets (:204-259, a factorisation-sharing
// device) give the same per-column iterates.  MAX_ITERATIONS = 5k per
// column; a column that exceeds it reports -1 (the reference exits).
//
// One wavefront per right-hand side: lane i owns variable i, the passive set
// is a 64-bit wave-uniform mask (ballots).  Two forms:
//  * bpp_pair_kernel: with H = G^-1 formed once for all columns, a pivot step
//    solves the smaller of the passive and the complementary system (at most
//    k / 2 variables, compacted).  Bound by FP64 arithmetic and the lane
//    broadcasts of the elimination (two v_readlane per FMA).  Taken where G's
//    1-norm condition is at most BPP_COND.
//  * bpp_kernel: a masked k x k elimination of the passive system per step,
//    for any other G and for columns the first form gives up.
// One ANLS-BPP iteration at 65536 x 16384, k = 64 (81920 columns, BF16
// products): 70.8 ms with the masked elimination of all k columns alone, 2.57
// ms with the pair (the products are 0.8 ms of it).
#include <algorithm>

#include "common.h"

namespace planc {

namespace {

__device__ inline double bcast(double v, int lane) {
  int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}

__device__ inline unsigned long long ballot64(bool p) { return __ballot(p); }

// The inverse of the Gram, shared by all columns of a solve.
struct BppInfo {
  double hnorm;  // 1-norm of H
  int ok;        // H may be used
};

// Passive set and exchange rules (nnls/bppnnls.hpp:93-145): full exchanges
// while the number of infeasible variables falls (or up to three times while
// it does not), else the largest infeasible index alone.
struct Exchange {
  unsigned long long P;
  int pcnt, ninf;
  __device__ Exchange(int k) : P(0ull), pcnt(3), ninf(k + 1) {}
  __device__ void step(unsigned long long nonopt, unsigned long long infea) {
    const int notgood = __popcll(nonopt) + __popcll(infea);
    if (notgood < ninf) {
      pcnt = 3;
      ninf = notgood;
      P = (P | nonopt) & ~infea;
    } else if (pcnt >= 1) {
      pcnt -= 1;
      P = (P | nonopt) & ~infea;
    } else {
      const int r = 63 - __clzll(nonopt | infea);
      P ^= (1ull << r);
    }
  }
};

// General form: any G.  Takes every column when the shared inverse is not
// usable (info->ok == 0), else only the columns that bpp_pair_kernel gave up
// (iters < 0).  Columns of the tableau left of the pivot are already unit
// vectors, so an elimination step only touches the columns right of it.
template <int KM>
__global__ __launch_bounds__(256) void bpp_kernel(const double *G, int k, const float *B, long b_cs,
                                                  long b_rs, long nrhs, float *X, long x_cs, long x_rs,
                                                  int maxit, const BppInfo *info, const int *iters, int *failed_out) {
  __shared__ double Gs[KM][KM + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const bool all = info->ok == 0;
  const long stride = (long)gridDim.x * nw;
  const long col0 = (long)blockIdx.x * nw + wave;
  if (!all) {
    int any = 0;
    for (long c = (long)blockIdx.x * nw + threadIdx.x % nw + (threadIdx.x / nw) * stride; c < nrhs;
         c += (blockDim.x / nw) * stride)
      any |= iters[c] < 0;  // the block's columns, spread over its threads
    if (!__syncthreads_or(any)) return;
  }
  for (int e = threadIdx.x; e < KM * KM; e += blockDim.x) {
    int r = e % KM, c = e / KM;
    Gs[r][c] = (r < k && c < k) ? G[r + (size_t)k * c] : 0.0;
  }
  __syncthreads();
  const bool live = lane < k;
  for (long col = col0; col < nrhs; col += stride) {
    if (!all && iters[col] >= 0) continue;
    const double b = live ? (double)B[col * b_cs + lane * b_rs] : 0.0;
    double x = 0.0, y = -b;
    Exchange ex(k);
    unsigned long long nonopt = ballot64(live && y < 0.0);
    unsigned long long infea = 0ull;
    int iter = 0;
    bool failed = false;
    while (nonopt | infea) {
      if (++iter > maxit) {
        failed = true;
        break;
      }
      ex.step(nonopt, infea);
      const unsigned long long P = ex.P;
      // Masked system [G(P,P) 0; 0 I] x = [b_P; 0], lane = row.
      const bool pi = (P >> lane) & 1ull;
      double a[KM];
#pragma unroll
      for (int t = 0; t < KM; ++t) {
        bool pt = (P >> t) & 1ull;
        a[t] = (pi && pt) ? Gs[lane < KM ? lane : 0][t] : (lane == t ? 1.0 : 0.0);
      }
      double rhs = pi ? b : 0.0;
      double diag = 1.0;
#pragma unroll
      for (int j = 0; j < KM; ++j) {
        if ((P >> j) & 1ull) {
          const double piv = bcast(a[j], j);
          const double rj = bcast(rhs, j);
          const double f = (lane != j) ? a[j] / piv : 0.0;
          diag = lane == j ? piv : diag;
#pragma unroll
          for (int t = j + 1; t < KM; ++t) a[t] = fma(-f, bcast(a[t], j), a[t]);
          rhs = fma(-f, rj, rhs);
        }
      }
      x = pi ? rhs / diag : 0.0;
      // Y = G x - b with the full Gram.
      double gx = 0.0;
#pragma unroll
      for (int t = 0; t < KM; ++t) {
        double xt = bcast(x, t);
        if (live) gx = fma(Gs[lane][t], xt, gx);
      }
      y = live ? gx - b : 0.0;
      if (fabs(x) < 1e-12) x = 0.0;
      if (fabs(y) < 1e-12) y = 0.0;
      nonopt = ballot64(live && y < 0.0 && !pi);
      infea = ballot64(live && x < 0.0 && pi);
    }
    if (live) X[col * x_cs + lane * x_rs] = (float)x;
    if (failed && lane == 0 && failed_out) *failed_out = 1;
  }
}

// ---------------------------------------------------------------------------
// H = G^-1 once for all columns (in-place Gauss-Jordan of the SPD Gram in
// LDS, one block), its 1-norm, and whether bpp_pair_kernel may use it: G
// positive definite with a 1-norm condition of at most BPP_COND, so that a
// solution formed from H is good to about eps cond^2 <= 2e-6 before its
// refinement (which squares that).
constexpr double BPP_COND = 1e5;
constexpr int BPP_INV_THR = 1024;

__global__ __launch_bounds__(BPP_INV_THR) void bpp_invert_kernel(const double *G, int k, double *H, BppInfo *info) {
  __shared__ double S[64][65];
  __shared__ double nrm[2][64];
  const int tid = threadIdx.x;
  const int kk = k * k;
  constexpr int U = 4096 / BPP_INV_THR;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = tid + u * BPP_INV_THR;
    if (e < kk) S[e % k][e / k] = G[e];
  }
  __syncthreads();
  auto col_norm = [&](int which) {
    if (tid < k) {
      double t = 0.0;
      for (int i = 0; i < k; ++i) t += fabs(S[i][tid]);
      nrm[which][tid] = t;
    }
  };
  col_norm(0);
  __syncthreads();
  bool pos = true;
  for (int j = 0; j < k; ++j) {
    const double d = S[j][j];
    pos = pos && d > 0.0;
    const double p = 1.0 / d;
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = tid + u * BPP_INV_THR, i = e % k, t = e / k;
      if (e >= kk) continue;
      const double aij = S[i][j], ajt = S[j][t];
      if (i != j && t != j) v[u] = fma(-aij * p, ajt, S[i][t]);
      else if (i == j && t == j) v[u] = p;
      else v[u] = i == j ? ajt * p : -aij * p;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int e = tid + u * BPP_INV_THR;
      if (e < kk) S[e % k][e / k] = v[u];
    }
    __syncthreads();
  }
  col_norm(1);
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = tid + u * BPP_INV_THR;
    if (e < kk) H[e] = 0.5 * (S[e % k][e / k] + S[e / k][e % k]);
  }
  if (tid == 0) {
    double g = 0.0, h = 0.0;
    bool fin = true;
    for (int i = 0; i < k; ++i) {
      fin = fin && nrm[0][i] < 1e300 && nrm[1][i] < 1e300;  // NaN fails too
      g = fmax(g, nrm[0][i]);
      h = fmax(h, nrm[1][i]);
    }
    info->hnorm = h;
    info->ok = pos && fin && g * h <= BPP_COND;
  }
}

// Solution of the compact q x q SPD system whose row `lane` is a (zero rows
// past q), lane = row: Gauss-Jordan, the pivot row broadcast with v_readlane.
// Elimination steps touch only the columns right of the pivot.
template <int QM>
__device__ inline double solve_compact(double (&a)[QM], double rhs, int q, int lane) {
  double dinv = 0.0;
#pragma unroll
  for (int j = 0; j < QM; ++j) {
    if (j < q) {
      const double rp = 1.0 / bcast(a[j], j);
      const double rj = bcast(rhs, j);
      const double f = (lane != j) ? a[j] * rp : 0.0;
      dinv = lane == j ? rp : dinv;
#pragma unroll
      for (int t = j + 1; t < QM; ++t) a[t] = fma(-f, bcast(a[t], j), a[t]);
      rhs = fma(-f, rj, rhs);
    }
  }
  return rhs * dinv;
}

// Gathers rows and columns `sel` (compact lane -> variable) of the symmetric
// M (LDS, row pitch LD) and solves for the right-hand side rhs.
template <int QM, int LD>
__device__ inline double gather_solve(const double *M, int sel, double rhs, int q, int lane) {
  double a[QM];
#pragma unroll
  for (int t = 0; t < QM; ++t) {
    const int st = __builtin_amdgcn_readlane(sel, t);
    a[t] = (lane < q && t < q) ? M[sel * LD + st] : 0.0;
  }
  return solve_compact<QM>(a, rhs, q, lane);
}

template <int KM, int LD>
__device__ inline double solve_selected(const double *M, int sel, double rhs, int q, int lane) {
  if (q == 0) return 0.0;
  if (q <= 4) return gather_solve<4, LD>(M, sel, rhs, q, lane);
  if constexpr (KM > 8)
    if (q <= 8) return gather_solve<8, LD>(M, sel, rhs, q, lane);
  if constexpr (KM > 16) {
    if (q <= 12) return gather_solve<12, LD>(M, sel, rhs, q, lane);
    if (q <= 16) return gather_solve<16, LD>(M, sel, rhs, q, lane);
  }
  if constexpr (KM > 32) {
    if (q <= 20) return gather_solve<20, LD>(M, sel, rhs, q, lane);
    if (q <= 24) return gather_solve<24, LD>(M, sel, rhs, q, lane);
    if (q <= 28) return gather_solve<28, LD>(M, sel, rhs, q, lane);
    return gather_solve<32, LD>(M, sel, rhs, q, lane);
  }
  return 0.0;
}

// Block principal pivoting from the pair (G, H = G^-1).  With the passive
// set P and its complement R, the solution of a pivot step follows either
// from the |P| x |P| system G_PP x_P = b_P (y_R = G_RP x_P - b_R), or, with
// c = H b, from the |R| x |R| system H_RR w = c_R (x_P = c_P - H_PR w, y_R =
// -w); the smaller one is solved, so no system is larger than k / 2.  One
// wavefront per column, lane = variable; the selected variables are
// compacted to the first lanes.  When no variable is left to exchange, the
// residual of the true normal equations is formed (y = G x - b); if it says
// that x may be off by more than 1e-10 of its largest entry, one step of
// refinement is solved on the same set, and the signs are tested again on the
// final values.
template <int KM>
__global__ __launch_bounds__(512) void bpp_pair_kernel(const double *G, const double *H, const BppInfo *info, int k,
                                                       const float *B, long b_cs, long b_rs, long nrhs, float *X,
                                                       long x_cs, long x_rs, int maxit, int *iters_out) {
  constexpr int LD = KM + 1;
  __shared__ double Gs[KM * LD], Hs[KM * LD];
  if (!info->ok) return;
  const double hnorm = info->hnorm;
  for (int e = threadIdx.x; e < KM * KM; e += blockDim.x) {
    const int r = e % KM, c = e / KM;
    const bool in = r < k && c < k;
    Gs[r * LD + c] = in ? G[r + (size_t)k * c] : 0.0;
    Hs[r * LD + c] = in ? H[r + (size_t)k * c] : 0.0;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const bool live = lane < k;
  const int row = (lane < KM ? lane : KM - 1) * LD;
  const unsigned long long every = k < 64 ? (1ull << k) - 1ull : ~0ull;
  // sum_t M(lane, t) v_t over all variables t
  auto times = [&](const double *M, double v) {
    double s0 = 0.0, s1 = 0.0;
#pragma unroll 4
    for (int t = 0; t < KM; t += 2) {
      s0 = fma(M[row + t], bcast(v, t), s0);
      s1 = fma(M[row + t + 1], bcast(v, t + 1), s1);
    }
    return s0 + s1;
  };
  const long stride = (long)gridDim.x * nw;
  for (long col = (long)blockIdx.x * nw + wave; col < nrhs; col += stride) {
    const double b = live ? (double)B[col * b_cs + lane * b_rs] : 0.0;
    const double c = times(Hs, b);
    double bb = b, cc = c;  // right-hand side of the current solve and H times it
    double x = 0.0, y = -b, xbase = 0.0;
    Exchange ex(k);
    unsigned long long nonopt = ballot64(live && y < 0.0);
    unsigned long long infea = 0ull;
    int iter = 0;
    bool failed = false, refine = false;
    while (refine || (nonopt | infea)) {
      if (!refine) {
        if (++iter > maxit) {
          failed = true;
          break;
        }
        ex.step(nonopt, infea);
      }
      const unsigned long long P = ex.P & every;
      const int np = __popcll(P);
      const bool primal = 2 * np <= k;
      const int q = primal ? np : k - np;
      const unsigned long long Q = primal ? P : (every & ~P);
      const bool pi = (P >> lane) & 1ull, qi = (Q >> lane) & 1ull;
      // Lane order: the selected variables first (a permutation of the wave).
      const int before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(Q >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)Q, 0u));
      const int rank = qi ? before : q + lane - before;
      const int sel = __builtin_amdgcn_ds_permute(4 * rank, lane);
      const double rhs = __shfl(primal ? bb : cc, sel, 64);
      const double *M = primal ? Gs : Hs;
      const double w = solve_selected<KM, LD>(M, sel < KM ? sel : 0, lane < q ? rhs : 0.0, q, lane);
      const double wv = __shfl(w, rank, 64);  // back in variable order (Q only)
      double s0 = 0.0, s1 = 0.0;  // sum over Q of M(lane, j) w_j
      int j = 0;
      for (; j + 1 < q; j += 2) {
        s0 = fma(M[row + __builtin_amdgcn_readlane(sel, j)], bcast(w, j), s0);
        s1 = fma(M[row + __builtin_amdgcn_readlane(sel, j + 1)], bcast(w, j + 1), s1);
      }
      if (j < q) s0 = fma(M[row + __builtin_amdgcn_readlane(sel, j)], bcast(w, j), s0);
      const double s = s0 + s1;
      double xs, ys;
      if (primal) {
        xs = pi ? wv : 0.0;
        ys = s - bb;
      } else {
        xs = pi ? cc - s : 0.0;
        ys = -wv;
      }
      if (!refine) {
        x = xs;
        y = pi || !live ? 0.0 : ys;
        if (fabs(x) < 1e-12) x = 0.0;
        if (fabs(y) < 1e-12) y = 0.0;
        nonopt = ballot64(live && y < 0.0 && !pi);
        infea = ballot64(live && x < 0.0 && pi);
        if (nonopt | infea) continue;
      } else {
        x = pi ? xbase + xs : 0.0;
        if (fabs(x) < 1e-12) x = 0.0;
      }
      // Nothing left to exchange (or just refined): the true residual.
      y = live ? times(Gs, x) - b : 0.0;
      if (!refine) {
        float xm = fabsf((float)x);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) xm = fmaxf(xm, __shfl_xor(xm, off, 64));
        if (ballot64(pi && !(fabs(y) * hnorm <= 1e-10 * (double)xm))) {
          refine = true;
          xbase = x;
          bb = pi ? -y : 0.0;
          cc = times(Hs, bb);
          continue;
        }
      }
      refine = false;
      bb = b;
      cc = c;
      if (fabs(y) < 1e-12) y = 0.0;
      nonopt = ballot64(live && y < 0.0 && !pi);
      infea = ballot64(live && x < 0.0 && pi);
    }
    if (live && !failed) X[col * x_cs + lane * x_rs] = (float)x;
    if (lane == 0) iters_out[col] = failed ? -1 : iter;
  }
}

}  // namespace

// Solves every column; *d_failed (device int) is set to 1 when a column
// needed more than 5k pivot iterations.  The shared inverse and the pair
// kernel take well-conditioned Grams; the general kernel behind them takes
// the others and any column that the pair kernel gave up, and ends at once
// where there is none.
template <int KM>
static void bpp_launch(planc_ctx *ctx, const double *G, const double *H, const BppInfo *info, int k, const float *B,
                       long b_cs, long b_rs, long nrhs, float *X, long x_cs, long x_rs, int *iters, int *d_failed) {
  // Persistent waves (the pair of matrices fills a third of a CU's LDS at k =
  // 64); a few right-hand sides are spread over four-wave blocks instead.
  const int nw = nrhs <= 4L * ctx->num_cu ? 4 : 8;
  const long nb = std::min<long>((nrhs + nw - 1) / nw, 2L * ctx->num_cu);
  bpp_pair_kernel<KM><<<(unsigned)nb, 64 * nw, 0, ctx->stream>>>(G, H, info, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs,
                                                                5 * k, iters);
  const long gb = std::min<long>((nrhs + 3) / 4, 4L * ctx->num_cu);
  bpp_kernel<KM><<<(unsigned)gb, 256, 0, ctx->stream>>>(G, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs, 5 * k, info, iters,
                                                       d_failed);
}

int bpp_solve(planc_ctx *ctx, const double *G, int k, const float *B, long b_cs, long b_rs, long nrhs,
              float *X, long x_cs, long x_rs, int *d_failed) {
  if (k <= 0 || k > 64) return set_error(ctx, PLANC_EUNSUPPORTED, "bpp: k must be 1..64");
  if (nrhs <= 0) return PLANC_OK;
  // Workspace: H, its description, then the columns' pivot counts.
  double *H = (double *)ws_get(ctx, 10, sizeof(double) * 4096 + sizeof(BppInfo) + sizeof(int) * (size_t)nrhs);
  if (!H) return set_error(ctx, PLANC_ENOMEM, "bpp: workspace");
  BppInfo *info = (BppInfo *)(H + 4096);
  int *iters = (int *)(info + 1);
  bpp_invert_kernel<<<1, BPP_INV_THR, 0, ctx->stream>>>(G, k, H, info);
  PLANC_LAUNCH_CHECK(ctx);
  if (k <= 16)
    bpp_launch<16>(ctx, G, H, info, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs, iters, d_failed);
  else if (k <= 32)
    bpp_launch<32>(ctx, G, H, info, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs, iters, d_failed);
  else
    bpp_launch<64>(ctx, G, H, info, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs, iters, d_failed);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

}  // namespace planc
