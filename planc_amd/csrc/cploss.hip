// CP reconstruction loss 0.5 ||X - [[A_0 .. A_{N-1}]]||^2 and its gradient.
//
// Forward: with the modes split at s (left block L = prod_{i<=s} I_i, right
// R), the reconstruction is Xhat_(L x R) = KRP_L * KRP_R^T.  The fused kernel
// forms Xhat in tiles of 64 (l) x 128 (r) with v_mfma_f32_16x16x4f32 from
// Khatri-Rao rows that it builds from the factors (never stored in HBM), reads
// the matching X tile once and accumulates (x - xhat)^2 in FP64.  A block keeps
// its KRP_R rows in registers and walks several l tiles, whose KRP_L rows are
// staged in LDS.  Bound by FP32 MFMA and HBM about alike at k = 48 (96^4: 54 us
// of MFMA, 53 us of reading).  Partials per block are summed in block order.
//
// Backward: dL/dA_n = A_n * (Hadamard of the other Grams) - MTTKRP_n^T, the
// transposed NTFNES gradient S Y - M (ntf/ntfnes.hpp:138-147) without the
// lambda shift.  All N MTTKRPs come from the two partial contractions of
// the dimension tree, each one pass over X with the KRP fused.
#include <mutex>
#include <string>

#include "common.h"
#include "wave.h"

namespace planc {

namespace {

constexpr int RT = 128;  // right indexes r of an Xhat tile
constexpr int LT = 64;   // left indexes l

struct CPParams {
  const float *X;
  long L, R;
  int k;
  int nl, nr;  // modes in the left / right block
  const float *fl[6];
  long dl[6];
  const float *fr[6];
  long dr[6];
  int ltiles_per_block;
  double *part;
};

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// Next mixed-radix digit of rem.
__device__ inline long next_digit(long &rem, long dq) {
  long nx, d;
  if (rem < (1L << 31) && dq < (1L << 31)) {  // 64-bit division is a call of a hundred instructions
    nx = (unsigned)rem / (unsigned)dq;
    d = (unsigned)rem - (unsigned)nx * (unsigned)dq;
  } else {
    nx = rem / dq;
    d = rem - nx * dq;
  }
  rem = nx;
  return d;
}

// Columns c0 .. c0 + NC - 1 of Khatri-Rao row g (its digits lowest mode
// fastest), zero past the limit and past k, in two halves: load() issues the
// loads of the first two factors' entries, value() multiplies them and the
// further factors' in mode order.
template <int NC>
struct KrpRow {
  float x0[NC], x1[NC];
  long rem;
  bool in;
  __device__ void load(long g, long limit, int nf, const float *const *f, const long *dims, int c0, int k) {
    in = g < limit;
    rem = in ? g : 0;
    // (With a wave-uniform c0 the columns' bases are scalars and the digits the
    // only per-lane offsets.)
    const unsigned d0 = (unsigned)next_digit(rem, dims[0]);
    const unsigned d1 = nf > 1 ? (unsigned)next_digit(rem, dims[1]) : d0;
    const int g1 = nf > 1 ? 1 : 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int cc = c0 + c < k ? c0 + c : k - 1;  // past k: column k - 1, zeroed by value()
      x0[c] = (f[0] + dims[0] * cc)[d0];
      x1[c] = (f[g1] + dims[g1] * cc)[d1];
    }
  }
  __device__ void value(float (&v)[NC], int nf, const float *const *f, const long *dims, int c0, int k) {
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = nf > 1 ? x0[c] * x1[c] : x0[c];
    for (int q = 2; q < nf; ++q) {
      const long d = next_digit(rem, dims[q]);
#pragma unroll
      for (int c = 0; c < NC; ++c) v[c] *= c0 + c < k ? f[q][d + dims[q] * (c0 + c)] : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = in && c0 + c < k ? v[c] : 0.0f;
  }
};

// Wave w of the block's eight owns the 16 columns r0 + 16 w .. + 15 and all 64
// rows of an l tile (four 16-row MFMA tiles).  MFMA k-slot g of step s stands
// for column KS g + s, so a lane's operands of all steps are consecutive: KR in
// registers, KL one LDS row piece of KS floats (pitch KP + 4: rows 4 banks
// apart).  acc[b][i] = Xhat(l0 + 16 b + 4 (lane / 16) + i, r0 + 16 w + lane % 16):
// four consecutive l, one 16-byte load of X.  An l tile's X words and the next
// one's factor entries are issued before its MFMAs and stay in flight through
// them.  96^4, k = 48: 117 us (130 with two column tiles per wave in four-wave
// blocks, two wavefronts a SIMD; about 540 with element loads of X and 64-bit
// divisions for every Khatri-Rao entry).
constexpr int FWD_THR = 512;
template <int KP>
__global__ __launch_bounds__(FWD_THR) void cp_loss_fwd_kernel(CPParams p) {
  constexpr int KS = KP / 4;  // MFMA steps
  constexpr int LP = KP + 4;
  constexpr int CT = LT * KP / FWD_THR;  // KL entries per thread
  __shared__ __attribute__((aligned(16))) float KL[2][LT * LP];
  __shared__ double red[FWD_THR / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lc = lane & 15, lg = lane >> 4;
  const long r = (long)blockIdx.x * RT + 16 * wave + lc;
  const long ltiles = (p.L + LT - 1) / LT;
  const long lt_begin = (long)blockIdx.y * p.ltiles_per_block;
  const long lt_end = min(ltiles, lt_begin + p.ltiles_per_block);
  float kr[KS];
  {
    KrpRow<KS> kx;
    kx.load(r, p.R, p.nr, p.fr, p.dr, KS * lg, p.k);
    kx.value(kr, p.nr, p.fr, p.dr, KS * lg, p.k);
  }
  // Row `lane`, columns c0 .. of a KL tile.
  KrpRow<CT> kn;
  const int c0 = CT * __builtin_amdgcn_readfirstlane(wave);
  auto fetch = [&](long lt) { kn.load(lt * LT + lane, p.L, p.nl, p.fl, p.dl, c0, p.k); };
  auto form = [&](int buf) {
    float v[CT];
    kn.value(v, p.nl, p.fl, p.dl, c0, p.k);
    static_assert(CT % 2 == 0, "pairs");
#pragma unroll
    for (int c = 0; c < CT; c += 2) *(float2 *)&KL[buf][lane * LP + c0 + c] = float2{v[c], v[c + 1]};
  };
  if (lt_begin < lt_end) {
    fetch(lt_begin);
    form(0);
  }
  double acc2 = 0.0;
  const float *xcol = p.X + p.L * (r < p.R ? r : p.R - 1) + 4 * lg;  // columns past R are left out of the sum
  for (long lt = lt_begin; lt < lt_end; ++lt) {
    const int buf = (int)(lt - lt_begin) & 1;
    const long l0 = lt * LT;
    const bool full = l0 + LT <= p.L;  // uniform
    floatx4 x[4];
    __syncthreads();
    if (full) {
#pragma unroll
      for (int b = 0; b < 4; ++b) x[b] = *(const floatx4u *)(xcol + l0 + 16 * b);
    }
    if (lt + 1 < lt_end) fetch(lt + 1);
    __builtin_amdgcn_sched_barrier(0);
    floatx4 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s4 = 0; s4 < KS / 4; ++s4) {
      floatx4 kl[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) kl[b] = *(const floatx4 *)&KL[buf][(16 * b + lc) * LP + KS * lg + 4 * s4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kl[b][j], kr[4 * s4 + j], acc[b], 0, 0, 0);
    }
    if (lt + 1 < lt_end) form(buf ^ 1);
    if (r >= p.R) continue;
    if (full) {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float d = x[b][i] - acc[b][i];
          acc2 += (double)d * (double)d;
        }
    } else {
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (l0 + 16 * b + 4 * lg + i < p.L) {
            const float d = xcol[l0 + 16 * b + i] - acc[b][i];
            acc2 += (double)d * (double)d;
          }
    }
  }
  // Block reduction (fixed order).
  acc2 = wave_sum(acc2);
  if (lane == 0) red[wave] = acc2;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < FWD_THR / 64; ++w) t += red[w];
    p.part[blockIdx.y * gridDim.x + blockIdx.x] = t;
  }
}

// Half the sum of n block partials, eight loads in flight per thread.
__global__ __launch_bounds__(256) void sum_half_kernel(const double *part, long n, double *out) {
  __shared__ double red[4];
  double t = 0.0;
  long b = threadIdx.x;
  for (; b + 7 * 256 < n; b += 8 * 256) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = part[b + 256 * u];
#pragma unroll
    for (int u = 0; u < 8; ++u) t += v[u];
  }
  for (; b < n; b += 256) t += part[b];
  t = wave_sum(t);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) *out = 0.5 * (red[0] + red[1] + red[2] + red[3]);
}

// grad_n(i, c) = sum_t A_n(i, t) S_n(t, c) - M_n(c, i) for every mode n in one
// launch; A_n I x k, M_n k x I, S_n the Hadamard product of the other modes'
// k x k Grams, formed in LDS.  A block takes 256 / KP rows at a time.
struct GradSet {
  const float *a[8], *m[8];
  float *grad[8];
  const double *g[8];
  long dim[8];
  int n;
};

template <int KP>
__global__ __launch_bounds__(256) void cp_grad_kernel(GradSet gs, int k) {
  __shared__ double S[KP * KP];  // S(t, c) at t + KP c
  const int mode = blockIdx.y;
  const long I = gs.dim[mode];
  constexpr int ROWS = 256 / KP;
  const long i0 = (long)blockIdx.x * ROWS;
  if (i0 >= I) return;
  constexpr int PER = KP * KP / 256;
  double sv[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) sv[j] = 1.0;
  for (int q = 0; q < gs.n; ++q) {
    if (q == mode) continue;
    double g[PER];  // a Gram's entries in flight together
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int e = threadIdx.x + 256 * j, t = e % KP, c = e / KP;
      g[j] = t < k && c < k ? gs.g[q][t + (long)k * c] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) sv[j] *= g[j];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) S[threadIdx.x + 256 * j] = sv[j];
  __syncthreads();
  const int c = threadIdx.x % KP, ri = threadIdx.x / KP;
  const float *A = gs.a[mode];
  for (long i = i0 + ri; i < I; i += (long)gridDim.x * ROWS) {
    if (ri >= ROWS || c >= k) continue;
    double s = 0.0;
    for (int t = 0; t < k; ++t) s += (double)A[i + I * t] * S[c + KP * t];  // S is symmetric
    gs.grad[mode][i + I * c] = (float)(s - (double)gs.m[mode][c + (long)k * i]);
  }
}

int balanced(int N, const long *dims) {
  int best = N / 2 < N - 1 ? N / 2 : N - 2;
  long bestv = -1;
  for (int s = 0; s <= N - 2; ++s) {
    long L = 1, R = 1;
    for (int i = 0; i <= s; ++i) L *= dims[i];
    for (int i = s + 1; i < N; ++i) R *= dims[i];
    long v = L > R ? L : R;
    if (bestv < 0 || v < bestv || (v == bestv && s == N / 2)) {
      bestv = v;
      best = s;
    }
  }
  return best;
}

}  // namespace

namespace {

// Block partition of one forward evaluation: the grid and how many FP64
// block partials it writes.  Both entry points use the same partition, so
// their sums are formed in the same order.
struct CPLaunch {
  CPParams p;
  dim3 grid;
  long nparts;
};

int cp_loss_plan(planc_ctx *ctx, const float *X, int N, const long *dims, const float *const *F,
                 int k, CPLaunch *out) {
  if (N < 2 || N > 7 || k <= 0 || k > 64) return set_error(ctx, PLANC_EINVAL, "cp_loss: 2..7 modes, k 1..64");
  int s = balanced(N, dims);
  CPParams p{};
  p.X = X;
  p.k = k;
  p.L = 1;
  p.R = 1;
  p.nl = s + 1;
  p.nr = N - 1 - s;
  if (p.nl > 6 || p.nr > 6) return set_error(ctx, PLANC_EINVAL, "cp_loss: too many modes per side");
  for (int i = 0; i <= s; ++i) {
    p.fl[i] = F[i];
    p.dl[i] = dims[i];
    p.L *= dims[i];
  }
  for (int i = s + 1; i < N; ++i) {
    p.fr[i - s - 1] = F[i];
    p.dr[i - s - 1] = dims[i];
    p.R *= dims[i];
  }
  long rblocks = (p.R + RT - 1) / RT;
  long ltiles = (p.L + LT - 1) / LT;
  long want = (2L * ctx->num_cu * 3 + rblocks - 1) / rblocks;  // six blocks per CU in all
  if (want < 1) want = 1;
  if (want > ltiles) want = ltiles;
  p.ltiles_per_block = (int)((ltiles + want - 1) / want);
  long lgroups = (ltiles + p.ltiles_per_block - 1) / p.ltiles_per_block;
  out->p = p;
  out->grid = dim3((unsigned)rblocks, (unsigned)lgroups);
  out->nparts = rblocks * lgroups;
  return PLANC_OK;
}

// Every block writes its own partial (nothing is accumulated into part), and
// the final kernel reads exactly nparts of them: part needs no clearing.
int cp_loss_launch(planc_ctx *ctx, CPLaunch &c, double *part, double *d_loss) {
  c.p.part = part;
  const int k = c.p.k;
  if (k <= 16)
    cp_loss_fwd_kernel<16><<<c.grid, FWD_THR, 0, ctx->stream>>>(c.p);
  else if (k <= 32)
    cp_loss_fwd_kernel<32><<<c.grid, FWD_THR, 0, ctx->stream>>>(c.p);
  else if (k <= 48)
    cp_loss_fwd_kernel<48><<<c.grid, FWD_THR, 0, ctx->stream>>>(c.p);
  else
    cp_loss_fwd_kernel<64><<<c.grid, FWD_THR, 0, ctx->stream>>>(c.p);
  PLANC_LAUNCH_CHECK(ctx);
  sum_half_kernel<<<1, 256, 0, ctx->stream>>>(part, c.nparts, d_loss);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

// Partials of the allocation-free forward: a file-scope device array, one
// copy per GPU, held until the process ends.  Its name is a host-side
// stand-in; kernels get the per-device address that hipGetSymbolAddress
// returns at context creation (cp_noalloc_setup), never the name itself.
constexpr long kNoallocParts = 16384;  // 128 KiB
static __device__ __align__(256) double scratch[kNoallocParts];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices];
int g_scratch_state[kMaxDevices];  // 0 not set up, 1 ready, -1 lookup failed

}  // namespace

int cp_loss_forward(planc_ctx *ctx, const float *X, int N, const long *dims, const float *const *F,
                    int k, double *d_loss) {
  CPLaunch c;
  int rc = cp_loss_plan(ctx, X, N, dims, F, k, &c);
  if (rc) return rc;
  double *part = (double *)ws_get(ctx, 3, sizeof(double) * (size_t)c.nparts);
  if (!part) return set_error(ctx, PLANC_ENOMEM, "cp_loss: workspace");
  return cp_loss_launch(ctx, c, part, d_loss);
}

// Called by planc_create with `device` current: looks up this device's copy
// of the partials array once per process.
int cp_noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices) return PLANC_EUNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_state[device] != 0) return g_scratch_state[device] > 0 ? PLANC_OK : PLANC_EHIP;
  void *ptr = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    g_scratch_state[device] = -1;
    return PLANC_EHIP;
  }
  g_scratch_ptr[device] = (double *)ptr;
  g_scratch_state[device] = 1;
  return PLANC_OK;
}

int cp_loss_forward_noalloc(planc_ctx *ctx, const float *X, int N, const long *dims,
                            const float *const *F, int k, double *d_loss) {
  const int dev = ctx->device;
  double *part = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (dev >= 0 && dev < kMaxDevices && g_scratch_state[dev] > 0) part = g_scratch_ptr[dev];
  }
  if (!part)
    return set_error(ctx, PLANC_EHIP,
                     "cp_loss_fwd_noalloc: the device's partials array could not be located "
                     "(hipGetSymbolAddress failed at context creation)");
  CPLaunch c;
  int rc = cp_loss_plan(ctx, X, N, dims, F, k, &c);
  if (rc) return rc;
  if (c.nparts > kNoallocParts)
    return set_error(ctx, PLANC_EINVAL,
                     "cp_loss_fwd_noalloc: " + std::to_string(c.nparts) +
                         " block partials exceed the fixed array of " + std::to_string(kNoallocParts) +
                         " (the right block of modes has too many rows); use planc_cp_loss_fwd");
  return cp_loss_launch(ctx, c, part, d_loss);
}

int cp_grads(planc_ctx *ctx, int N, const long *dims, const float *const *F, int k, const double *const *G,
             const float *const *M, float *const *grads) {
  GradSet gs{};
  gs.n = N;
  long Imax = 0;
  for (int i = 0; i < N; ++i) {
    gs.a[i] = F[i];
    gs.m[i] = M[i];
    gs.grad[i] = grads[i];
    gs.g[i] = G[i];
    gs.dim[i] = dims[i];
    if (dims[i] > Imax) Imax = dims[i];
  }
  auto grid = [&](int rows) {
    const long nb = (Imax + rows - 1) / rows;
    return dim3((unsigned)(nb < 1024 ? nb : 1024), (unsigned)N);
  };
  if (k <= 16) cp_grad_kernel<16><<<grid(16), 256, 0, ctx->stream>>>(gs, k);
  else if (k <= 32) cp_grad_kernel<32><<<grid(8), 256, 0, ctx->stream>>>(gs, k);
  else cp_grad_kernel<64><<<grid(4), 256, 0, ctx->stream>>>(gs, k);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

int cp_split(int N, const long *dims) { return balanced(N, dims); }

}  // namespace planc
