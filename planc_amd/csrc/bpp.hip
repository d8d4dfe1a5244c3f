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
// is a 64-bit wave-uniform mask (ballots), the variables of a step's system are
// compacted to the first lanes.  Two forms of bpp_kernel:
//  * the pair: with H = G^-1 formed once for all columns, a step solves the
//    smaller of the passive and the complementary system (at most k / 2
//    variables).  Taken where G's 1-norm condition is at most BPP_COND.
//  * the passive system itself, for any other G, for a few columns of a small G
//    and for columns the pair gives up (more than 5 k steps, or H b not finite).
// Bound by FP64 arithmetic and the lane broadcasts of the elimination (two
// v_readlane per FMA).  One ANLS-BPP iteration at 65536 x 16384, k = 64 (81920
// columns, BF16 products): 70.8 ms with a masked elimination of all k columns
// per step, 1.86 ms so (0.87 ms are the products; 65536 columns by the pair 0.13
// ms, 16384 at a condition of 6e6 by the passive system 0.64 ms).
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

// ---------------------------------------------------------------------------
// H = G^-1 once for all columns (in-place Gauss-Jordan of the SPD Gram, one
// block), its 1-norm, and whether the pair form may use it: G positive
// definite with a 1-norm condition of at most BPP_COND, so that a solution
// formed from H is good to about eps cond^2 <= 2e-4, which each refinement
// multiplies by as much again.  Thread (ty, tx) of 16 x 16 keeps the entries (T
// ty + a, T tx + b), T = K / 16, in registers; a step passes the pivot's row and
// column through LDS (two buffers, one barrier a step: a chain of k LDS round
// trips and reciprocals; held in LDS with two barriers of 1024 threads a step it
// took 72 us at k = 64).  Rows past k are those of the identity.
constexpr double BPP_COND = 1e6;

template <int T>
__global__ __launch_bounds__(256) void bpp_invert_kernel(const double *G, int k, double *H, BppInfo *info) {
  constexpr int K = 16 * T;
  __shared__ __attribute__((aligned(16))) double row[2][K], col[2][K];
  __shared__ double out[K][K + 1];
  __shared__ double nrm[2][K];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  double s[T][T];
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b) {
      const int i = T * ty + a, t = T * tx + b;
      s[a][b] = i < k && t < k ? G[i + (size_t)k * t] : (i == t ? 1.0 : 0.0);
    }
  auto col_norms = [&](int which) {
#pragma unroll
    for (int a = 0; a < T; ++a)
#pragma unroll
      for (int b = 0; b < T; ++b) out[T * ty + a][T * tx + b] = s[a][b];
    __syncthreads();
    if (tid < K) {
      double v = 0.0;
      for (int i = 0; i < k; ++i) v += fabs(out[i][tid]);
      nrm[which][tid] = tid < k ? v : 0.0;
    }
    __syncthreads();
  };
  col_norms(0);
  bool pos = true;
  for (int jb = 0; jb * T < k; ++jb) {
#pragma unroll
    for (int jj = 0; jj < T; ++jj) {
      const int j = jb * T + jj, buf = (T % 2 == 0 ? jj : j) & 1;
      if (ty == jb)
#pragma unroll
        for (int b = 0; b < T; ++b) row[buf][T * tx + b] = s[jj][b];
      if (tx == jb)
#pragma unroll
        for (int a = 0; a < T; ++a) col[buf][T * ty + a] = s[a][jj];
      __syncthreads();
      const double d = row[buf][j];
      pos = pos && d > 0.0;
      const double p = 1.0 / d;
      double rv[T], cv[T];
#pragma unroll
      for (int b = 0; b < T; ++b) {
        rv[b] = row[buf][T * tx + b] * p;
        cv[b] = col[buf][T * ty + b];
      }
#pragma unroll
      for (int a = 0; a < T; ++a)
#pragma unroll
        for (int b = 0; b < T; ++b) {
          const bool ri = ty == jb && a == jj, ci = tx == jb && b == jj;
          const double e = fma(-cv[a], rv[b], s[a][b]);
          s[a][b] = ri ? (ci ? p : rv[b]) : (ci ? -cv[a] * p : e);
        }
    }
  }
  __syncthreads();
  col_norms(1);
  for (int e = tid; e < k * k; e += 256) H[e] = 0.5 * (out[e % k][e / k] + out[e / k][e % k]);
  if (tid < 64) {
    double g = tid < K ? nrm[0][tid] : 0.0, h = tid < K ? nrm[1][tid] : 0.0;
    const bool fin = __all(g < 1e300 && h < 1e300);  // NaN fails too
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      g = fmax(g, __shfl_xor(g, off, 64));
      h = fmax(h, __shfl_xor(h, off, 64));
    }
    if (tid == 0) {
      info->hnorm = h;
      info->ok = pos && fin && g * h <= BPP_COND;
    }
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

// QX: the largest q.  Steps of 4 up to 32, of 8 beyond (code size: a system of
// 64 is 50 KB of unrolled elimination).
template <int QX, int LD>
__device__ inline double solve_selected(const double *M, int sel, double rhs, int q, int lane) {
  if (q == 0) return 0.0;
  if (q <= 4) return gather_solve<4, LD>(M, sel, rhs, q, lane);
  if constexpr (QX > 4)
    if (q <= 8) return gather_solve<8, LD>(M, sel, rhs, q, lane);
  if constexpr (QX > 8) {
    if (q <= 12) return gather_solve<12, LD>(M, sel, rhs, q, lane);
    if (q <= 16) return gather_solve<16, LD>(M, sel, rhs, q, lane);
  }
  if constexpr (QX > 16) {
    if (q <= 20) return gather_solve<20, LD>(M, sel, rhs, q, lane);
    if (q <= 24) return gather_solve<24, LD>(M, sel, rhs, q, lane);
    if (q <= 28) return gather_solve<28, LD>(M, sel, rhs, q, lane);
    if (q <= 32) return gather_solve<32, LD>(M, sel, rhs, q, lane);
  }
  if constexpr (QX > 32) {
    if (q <= 40) return gather_solve<40, LD>(M, sel, rhs, q, lane);
    if (q <= 48) return gather_solve<48, LD>(M, sel, rhs, q, lane);
    if (q <= 56) return gather_solve<56, LD>(M, sel, rhs, q, lane);
    return gather_solve<64, LD>(M, sel, rhs, q, lane);
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
// residual of the true normal equations is formed (y = G x - b); while it says
// that x may be off by more than 1e-10 of its largest entry, a step of
// refinement is solved on the same set (at most BPP_REFINE), and the signs are
// tested again on the final values.
// PAIR = false is the form for any other G: every step solves the passive system
// itself, from G, and nothing is refined.  It takes all columns where there is no
// inverse (info null) or it is not usable, else only those that the pair gave up
// (iters < 0), and sets *failed_out for a column that needs more than maxit steps.
constexpr int BPP_REFINE = 3;
template <int KM, bool PAIR>
__global__ __launch_bounds__(512) void bpp_kernel(const double *G, const double *H, const BppInfo *info, int k,
                                                  const float *B, long b_cs, long b_rs, long nrhs, float *X,
                                                  long x_cs, long x_rs, int maxit, int *iters, int *failed_out) {
  constexpr int LD = KM + 1;
  __shared__ double Gs[KM * LD], Hs[PAIR ? KM * LD : 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const long stride = (long)gridDim.x * nw;
  const bool usable = info && info->ok != 0;
  if (PAIR && !usable) return;
  if (!PAIR && usable) {
    int any = 0;
    for (long c = (long)blockIdx.x * nw + threadIdx.x % nw + (threadIdx.x / nw) * stride; c < nrhs;
         c += (blockDim.x / nw) * stride)
      any |= iters[c] < 0;  // the block's columns, spread over its threads
    if (!__syncthreads_or(any)) return;
  }
  const double hnorm = PAIR ? info->hnorm : 0.0;
  for (int e = threadIdx.x; e < KM * KM; e += blockDim.x) {
    const int r = e % KM, c = e / KM;
    const bool in = r < k && c < k;
    Gs[r * LD + c] = in ? G[r + (size_t)k * c] : 0.0;
    if (PAIR) Hs[r * LD + c] = in ? H[r + (size_t)k * c] : 0.0;
  }
  __syncthreads();
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
  for (long col = (long)blockIdx.x * nw + wave; col < nrhs; col += stride) {
    if (!PAIR && usable && iters[col] >= 0) continue;
    const double b = live ? (double)B[col * b_cs + lane * b_rs] : 0.0;
    const double c = PAIR ? times(Hs, b) : 0.0;
    // H spreads an entry that is no finite number over the whole column; the
    // passive systems meet it only where its variable is passive.
    if (PAIR && ballot64(live && !isfinite(c))) {
      if (lane == 0) iters[col] = -1;
      continue;
    }
    double bb = b, cc = c;  // right-hand side of the current solve and H times it
    double x = 0.0, y = -b, xbase = 0.0;
    Exchange ex(k);
    unsigned long long nonopt = ballot64(live && y < 0.0);
    unsigned long long infea = 0ull;
    int iter = 0;
    bool failed = false, refine = false;
    int refined = 0;
    while (refine || (nonopt | infea)) {
      if (!refine) {
        if (++iter > maxit) {
          failed = true;
          break;
        }
        ex.step(nonopt, infea);
        refined = 0;
      }
      const unsigned long long P = ex.P & every;
      const int np = __popcll(P);
      const bool primal = !PAIR || 2 * np <= k;
      const int q = primal ? np : k - np;
      const unsigned long long Q = primal ? P : (every & ~P);
      const bool pi = (P >> lane) & 1ull, qi = (Q >> lane) & 1ull;
      // Lane order: the selected variables first (a permutation of the wave).
      const int before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(Q >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)Q, 0u));
      const int rank = qi ? before : q + lane - before;
      const int sel = __builtin_amdgcn_ds_permute(4 * rank, lane);
      const double rhs = __shfl(primal ? bb : cc, sel, 64);
      const double *M = primal ? Gs : Hs;
      const double w = solve_selected<PAIR ? KM / 2 : KM, LD>(M, sel < KM ? sel : 0, lane < q ? rhs : 0.0, q, lane);
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
        if (!PAIR || (nonopt | infea)) continue;
      } else {
        x = pi ? xbase + xs : 0.0;
        if (fabs(x) < 1e-12) x = 0.0;
      }
      // Nothing left to exchange (or just refined): the true residual.
      y = live ? times(Gs, x) - b : 0.0;
      if (refined < BPP_REFINE) {
        float xm = fabsf((float)x);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) xm = fmaxf(xm, __shfl_xor(xm, off, 64));
        if (ballot64(pi && !(fabs(y) * hnorm <= 1e-10 * (double)xm))) {
          refine = true;
          ++refined;
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
    if (PAIR) {
      if (live && !failed) X[col * x_cs + lane * x_rs] = (float)x;
      if (lane == 0) iters[col] = failed ? -1 : iter;
    } else {
      if (live) X[col * x_cs + lane * x_rs] = (float)x;
      if (failed && lane == 0 && failed_out) *failed_out = 1;
    }
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
  bpp_kernel<KM, true><<<(unsigned)nb, 64 * nw, 0, ctx->stream>>>(G, H, info, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs,
                                                                 5 * k, iters, nullptr);
  const long gb = std::min<long>((nrhs + 3) / 4, 3L * ctx->num_cu);
  bpp_kernel<KM, false><<<(unsigned)gb, 256, 0, ctx->stream>>>(G, nullptr, info, k, B, b_cs, b_rs, nrhs, X, x_cs,
                                                                  x_rs, 5 * k, iters, d_failed);
}

// A few right-hand sides of a Gram of up to 16 variables are solved by the general
// kernel alone: its systems are as small as the pair's would be within a step of
// four, and the call is bound by its launches.  16 variables, 60 columns: 37 us a
// call, 42 in three launches; 2 variables, 5 columns: 29 and 34 (32 with a masked
// elimination and a launch that gathered the failures).
constexpr int BPP_DIRECT_K = 16;

int bpp_solve(planc_ctx *ctx, const double *G, int k, const float *B, long b_cs, long b_rs, long nrhs,
              float *X, long x_cs, long x_rs, int *d_failed) {
  if (k <= 0 || k > 64) return set_error(ctx, PLANC_EUNSUPPORTED, "bpp: k must be 1..64");
  if (nrhs <= 0) return PLANC_OK;
  if (k <= BPP_DIRECT_K && nrhs <= 4L * ctx->num_cu) {
    const unsigned nb = (unsigned)((nrhs + 3) / 4);
    bpp_kernel<16, false><<<nb, 256, 0, ctx->stream>>>(G, nullptr, nullptr, k, B, b_cs, b_rs, nrhs, X, x_cs, x_rs, 5 * k,
                                                       nullptr, d_failed);
    PLANC_LAUNCH_CHECK(ctx);
    return PLANC_OK;
  }
  // Workspace: H, its description, then the columns' pivot counts.
  double *H = (double *)ws_get(ctx, 10, sizeof(double) * 4096 + sizeof(BppInfo) + sizeof(int) * (size_t)nrhs);
  if (!H) return set_error(ctx, PLANC_ENOMEM, "bpp: workspace");
  BppInfo *info = (BppInfo *)(H + 4096);
  int *iters = (int *)(info + 1);
  if (k <= 16) bpp_invert_kernel<1><<<1, 256, 0, ctx->stream>>>(G, k, H, info);
  else if (k <= 32) bpp_invert_kernel<2><<<1, 256, 0, ctx->stream>>>(G, k, H, info);
  else if (k <= 48) bpp_invert_kernel<3><<<1, 256, 0, ctx->stream>>>(G, k, H, info);
  else bpp_invert_kernel<4><<<1, 256, 0, ctx->stream>>>(G, k, H, info);
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
