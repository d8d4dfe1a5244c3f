// Sparse-input NMF (the reference's BUILD_SPARSE build of nmf/nmf.cpp with
// SP_MAT A): the update rules are those of the dense path, only the two
// products with A change.  A is held as CSR (row pointers int64, column
// indices int32, FP32 values) and, for W^T A, as the CSR of A^T (built once
// per run on the device by a stable sort of the entries by column, the
// analogue of the reference's At = A.t() in the constructors).
//
// Products: out(r, :) = sum_e val(e) F(col(e), :) over the entries of row r
// (SpMM), FP32 sums; the dense factor is read from a row-major (k-major) copy
// so every entry gathers one contiguous row of F, 16 bytes a lane.  Bound by
// the gathers' latency and L2 rate, so what counts is entries in flight, on
// rows whose lengths follow a power law: rows of up to SP_SHORT entries are
// walked by a lane group each (several rows per wavefront), longer ones are
// cut into segments of SP_SEG entries that a whole wavefront walks, its groups
// taking entries in turn, and a row's segments are added in order.  Term-
// document matrix 100000 x 40000, 2.6 M entries, k = 32 (its longest row has
// 40000): a wavefront per row walking its entries one by one took 4983 us a
// product, this takes 28 and 5.6 to add the pieces; a run of five MU
// iterations 51.1 -> 0.97 ms.
//
// Also the sparse error helper of common/utils.hpp:190-241 (sum over the
// non-zeros of (a_ij - w_i h_j)^2 and of (w_i h_j)^2, plus ||W H^T||_F^2).
#include <algorithm>

#include "common.h"
#include "wave.h"

// After common.h: hipCUB picks its backend from the platform macro that
// hip_runtime.h defines.
#include <hipcub/device/device_radix_sort.hpp>

namespace planc {

namespace {

constexpr int kSparseSlot0 = 24;  // context workspace slots 24..31 belong to this file

__global__ __launch_bounds__(256) void csr_entry_rows_kernel(long m, const long *indptr, int *rowid) {
  const long r = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= m) return;
  const int lane = threadIdx.x & 63;
  for (long e = indptr[r] + lane; e < indptr[r + 1]; e += 64) rowid[e] = (int)r;
}

__global__ void iota_kernel(long n, int *v) {
  long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) v[e] = (int)e;
}

// Row pointers of A^T by the first nptr blocks, its entries in their sorted order
// by the others.  Pointer j is the number of keys below j, found by bisection, so
// that a run of empty columns costs no more than others (1000 entries in the
// first 100 of 2 M columns: 89 us, 64 ms with the pointers between two entries'
// columns written by one lane).
__global__ void csr_t_gather_kernel(long nnz, long n, const int *ent, const unsigned *key, const int *rowid,
                                    const float *values, int *out_indices, float *out_values, long *out_indptr,
                                    int *out_entries, int nptr) {
  if ((int)blockIdx.x < nptr) {
    for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j <= n; j += (long)nptr * blockDim.x) {
      long lo = 0, hi = nnz;
      while (lo < hi) {
        const long mid = (lo + hi) / 2;
        if ((long)key[mid] < j) lo = mid + 1;
        else hi = mid;
      }
      out_indptr[j] = lo;
    }
    return;
  }
  const long p = (long)(blockIdx.x - nptr) * blockDim.x + threadIdx.x;
  if (p >= nnz) return;
  const int e = ent[p];
  out_indices[p] = rowid[e];
  out_values[p] = values[e];
  if (out_entries) out_entries[p] = e;
}

constexpr int SP_SHORT = 64;
constexpr int SP_SEG = 512;
constexpr int SP_WIDE = SP_SEG;

// A piece of a row longer than SP_SHORT: entries part * SP_SEG .. of row
// `row`; with nseg > 1 its sums go to partial row pslot, the row's pieces in
// consecutive ones.
struct SpSeg {
  int row, part, nseg, pslot;
};

__global__ void spmm_plan_zero_kernel(int *cnt) {
  if (threadIdx.x < 2) cnt[threadIdx.x] = 0;
}

// cnt[0] pieces and cnt[1] partial rows.  Their order depends on the atomics,
// the values computed from them do not.
__global__ void spmm_plan_kernel(long rows, const long *indptr, int *cnt, SpSeg *seg) {
  const long r = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const long len = indptr[r + 1] - indptr[r];
  if (len <= SP_SHORT) return;
  const int ns = (int)((len + SP_SEG - 1) / SP_SEG);
  const int slot = atomicAdd(&cnt[0], ns);
  const int ps = ns > 1 ? atomicAdd(&cnt[1], ns) : 0;
  for (int p = 0; p < ns; ++p) seg[slot + p] = SpSeg{(int)r, p, ns, ps + p};
}

__device__ inline void spmm_store4(float *out, long r, int c, int k, long ors, long ocs, floatx4 v) {
  if (ocs == 1 && c + 3 < k) {
    typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
    *(floatx4u *)(out + r * ors + c) = v;
    return;
  }
#pragma unroll
  for (int u = 0; u < 4; ++u)
    if (c + u < k) out[r * ors + (c + u) * ocs] = v[u];
}

// out(r, c) at out[r * ors + c * ocs], F k-major (element (j, c) at F[j * ldf
// + c], ldf a multiple of 4).  G lanes (4 G >= k) hold an output row, four
// columns each.  PLAN: blocks below nsegb walk the pieces, the others the short
// rows.  Without a plan (a single product whose entry count the host does not
// know) the first nsegb blocks take four rows at a time: a row of more than SP_SHORT
// entries is walked by a wavefront, one of more than SP_WIDE by the block's four
// together.  k = 16, 10000 rows of 100 entries: 14 us, of 1000: 58 (67 and 189
// where the long ones among a block's rows were walked one after the other by all
// four, 46 and 417 with a wavefront per row and an entry at a time).
template <int G, bool PLAN>
__global__ __launch_bounds__(256) void spmm_kernel(long rows, const long *indptr, const int *indices,
                                                   const float *values, const float *F, long ldf, int k, float *out,
                                                   long ors, long ocs, int nsegb, const int *cnt, const SpSeg *seg,
                                                   float *partial) {
  constexpr int NG = 64 / G;  // groups per wavefront
  constexpr int U = 4;        // entries in flight per group
  const int lane = threadIdx.x & 63, gl = lane % G, grp = lane / G;
  const int c = 4 * gl < ldf ? 4 * gl : 0;  // lanes past the row re-read its first columns (not stored)
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  // Entries e0, e0 + st, ... below e1.
  auto walk = [&](long e0, long e1, int st) {
    long e = e0;
    for (; e + (U - 1) * st < e1; e += U * st) {
      int j[U];
      float v[U];
      floatx4 f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        j[u] = indices[e + u * st];
        v[u] = values[e + u * st];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] = *(const floatx4 *)(F + (long)j[u] * ldf + c);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = fmaf(v[u], f[u][q], acc[q]);
    }
    if (e < e1) {  // the rest, in flight together: entries past the end weigh nothing
      int j[U - 1];
      float v[U - 1];
      floatx4 f[U - 1];
#pragma unroll
      for (int u = 0; u < U - 1; ++u) {
        const long x = e + u * st < e1 ? e + u * st : e;
        j[u] = indices[x];
        v[u] = values[x];
      }
#pragma unroll
      for (int u = 0; u < U - 1; ++u) f[u] = *(const floatx4 *)(F + (long)j[u] * ldf + c);
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (e + u * st < e1)
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] = fmaf(v[u], f[u][q], acc[q]);
    }
  };
  if ((int)blockIdx.x >= nsegb) {
    const long r = ((long)blockIdx.x - nsegb) * (256 / G) + threadIdx.x / G;
    const long b = r < rows ? indptr[r] : 0, e = r < rows ? indptr[r + 1] : 0;
    const bool is_long = e - b > SP_SHORT;
    if (r < rows && !is_long) {
      walk(b, e, 1);
      spmm_store4(out, r, 4 * gl, k, ors, ocs, acc);
    }
    return;
  }
  if constexpr (!PLAN) {
    __shared__ floatx4 red[4][G];
    const int wave = threadIdx.x >> 6;
    auto add_groups = [&]() {
#pragma unroll
      for (int off = G; off < 64; off <<= 1)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += __shfl_xor(acc[q], off, 64);
    };
    for (long r0 = 4L * blockIdx.x; r0 < rows; r0 += 4L * nsegb) {
      long b[5];
#pragma unroll
      for (int i = 0; i < 5; ++i) b[i] = indptr[min(r0 + i, rows)];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long len = b[i + 1] - b[i];
        if (len <= SP_WIDE) {
          if (wave == i && len > SP_SHORT) {
            acc = floatx4{0.f, 0.f, 0.f, 0.f};
            walk(b[i] + grp, b[i + 1], NG);
            add_groups();
            if (grp == 0) spmm_store4(out, r0 + i, 4 * gl, k, ors, ocs, acc);
          }
          continue;
        }
        acc = floatx4{0.f, 0.f, 0.f, 0.f};
        walk(b[i] + wave * NG + grp, b[i + 1], 4 * NG);
        add_groups();
        if (grp == 0) red[wave][gl] = acc;
        __syncthreads();
        if (threadIdx.x < G)
          spmm_store4(out, r0 + i, 4 * gl, k, ors, ocs, (red[0][gl] + red[1][gl]) + (red[2][gl] + red[3][gl]));
        __syncthreads();
      }
    }
    return;
  }
  const int n = cnt[0];
  for (int s = blockIdx.x * 4 + (threadIdx.x >> 6); s < n; s += nsegb * 4) {
    const SpSeg sg = seg[s];
    const long b = indptr[sg.row] + (long)sg.part * SP_SEG;
    const long e = min(b + SP_SEG, indptr[sg.row + 1]);
    acc = floatx4{0.f, 0.f, 0.f, 0.f};
    walk(b + grp, e, NG);
#pragma unroll
    for (int off = G; off < 64; off <<= 1)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] += __shfl_xor(acc[q], off, 64);
    if (grp == 0) {
      if (sg.nseg == 1) spmm_store4(out, sg.row, 4 * gl, k, ors, ocs, acc);
      else *(floatx4 *)(partial + ((long)sg.pslot * G + gl) * 4) = acc;
    }
  }
}

// Rows of more than one piece: their partial sums in piece order.
template <int G>
__global__ __launch_bounds__(256) void spmm_finish_kernel(const int *cnt, const SpSeg *seg, const float *partial, int k,
                                                          float *out, long ors, long ocs) {
  const int gl = threadIdx.x % G;
  const int n = cnt[0];
  for (int s = (blockIdx.x * 256 + threadIdx.x) / G; s < n; s += gridDim.x * (256 / G)) {
    const SpSeg sg = seg[s];
    if (sg.part != 0 || sg.nseg == 1) continue;
    const floatx4 *p = (const floatx4 *)partial + (long)sg.pslot * G + gl;
    floatx4 t = {0.f, 0.f, 0.f, 0.f};
    int i = 0;
    for (; i + 8 <= sg.nseg; i += 8) {
      floatx4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[(long)(i + u) * G];
#pragma unroll
      for (int u = 0; u < 8; ++u) t += v[u];
    }
    for (; i < sg.nseg; ++i) t += p[(long)i * G];
    spmm_store4(out, sg.row, 4 * gl, k, ors, ocs, t);
  }
}

// Per block: sum over the non-zeros of its rows of (a - t)^2 and t^2 with
// t = w_i . h_j (FP64), W and H k-major.  part[2 * block + {0, 1}].
__global__ __launch_bounds__(256) void sparse_fit_kernel(long m, const long *indptr, const int *indices,
                                                          const float *values, const float *Wk,
                                                          const float *Hk, int k, double *part) {
  __shared__ double red[2][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double sse = 0.0, wh2 = 0.0;
  for (long r = (long)blockIdx.x * 4 + wave; r < m; r += (long)gridDim.x * 4) {
    const double w = lane < k ? (double)Wk[r * k + lane] : 0.0;
    for (long e = indptr[r]; e < indptr[r + 1]; ++e) {
      const int j = indices[e];
      double t = lane < k ? w * (double)Hk[(long)j * k + lane] : 0.0;
      t = wave_sum(t);
      const double d = (double)values[e] - t;
      sse += d * d;  // identical in every lane
      wh2 += t * t;
    }
  }
  if (lane == 0) {
    red[0][wave] = sse;
    red[1][wave] = wh2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    part[2 * blockIdx.x + 1] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
  }
}

// err = sqrt(nnzsse + (||W H^T||^2 - nnzwh)) with ||W H^T||^2 = tr(WtW HtH)
// (the reference takes it as ||R_W R_H^T||_F^2 from economy QRs, the same
// quantity).
__global__ void sparse_fit_finalize_kernel(const double *part, int nb, const double *WtW,
                                           const double *HtH, int k, double *err) {
  if (threadIdx.x != 0) return;
  double sse = 0.0, wh2 = 0.0;
  for (int b = 0; b < nb; ++b) {
    sse += part[2 * b];
    wh2 += part[2 * b + 1];
  }
  double tr = 0.0;
  for (int a = 0; a < k; ++a)
    for (int c = 0; c < k; ++c) tr += WtW[a + (long)k * c] * HtH[c + (long)k * a];
  *err = sqrt(sse + (tr - wh2));
}

}  // namespace

// Stable transpose of a CSR matrix (m x n) into the CSR of its transpose
// (n x m): entries grouped by column, rows increasing within a column.
int csr_transpose(planc_ctx *ctx, long m, long n, long nnz, const long *indptr, const int *indices,
                  const float *values, long *out_indptr, int *out_indices, float *out_values, int *out_entries) {
  if (nnz >= (1L << 31) || n >= (1L << 31) || m >= (1L << 31))
    return set_error(ctx, PLANC_EUNSUPPORTED, "csr_transpose: at most 2^31-1 rows, columns and entries");
  if (nnz == 0) {
    PLANC_HIP_CHECK(ctx, hipMemsetAsync(out_indptr, 0, sizeof(long) * (n + 1), ctx->stream));
    return PLANC_OK;
  }
  int bits = 1;
  while (bits < 31 && (1L << bits) < n) ++bits;
  int *rowid = (int *)ws_get(ctx, kSparseSlot0 + 4, sizeof(int) * (size_t)nnz);
  unsigned *keys = (unsigned *)ws_get(ctx, kSparseSlot0 + 5, sizeof(unsigned) * 2 * (size_t)nnz);
  int *ent = (int *)ws_get(ctx, kSparseSlot0 + 6, sizeof(int) * 2 * (size_t)nnz);
  if (!rowid || !keys || !ent) return set_error(ctx, PLANC_ENOMEM, "csr_transpose: workspace");
  unsigned *keys_s = keys + nnz;
  int *ent_s = ent + nnz;
  csr_entry_rows_kernel<<<(unsigned)((m + 3) / 4), 256, 0, ctx->stream>>>(m, indptr, rowid);
  PLANC_LAUNCH_CHECK(ctx);
  iota_kernel<<<(unsigned)((nnz + 255) / 256), 256, 0, ctx->stream>>>(nnz, ent);
  PLANC_LAUNCH_CHECK(ctx);
  PLANC_HIP_CHECK(ctx, hipMemcpyAsync(keys, indices, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToDevice,
                                      ctx->stream));
  size_t bytes = 0;
  PLANC_HIP_CHECK(ctx, hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys, keys_s, ent, ent_s, (int)nnz, 0,
                                                          bits, ctx->stream));
  void *temp = ws_get(ctx, kSparseSlot0 + 7, bytes);
  if (!temp) return set_error(ctx, PLANC_ENOMEM, "csr_transpose: sort workspace");
  PLANC_HIP_CHECK(ctx, hipcub::DeviceRadixSort::SortPairs(temp, bytes, keys, keys_s, ent, ent_s, (int)nnz, 0,
                                                          bits, ctx->stream));
  const int nptr = (int)std::min<long>((n + 256) / 256, 1L << 20);  // n + 1 pointers
  csr_t_gather_kernel<<<(unsigned)(nptr + (nnz + 255) / 256), 256, 0, ctx->stream>>>(
      nnz, n, ent_s, keys_s, rowid, values, out_indices, out_values, out_indptr, out_entries, nptr);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

// The pieces of a CSR's long rows, in workspace slot `slot` (two counts, then
// room for all that nnz entries can make).
int spmm_plan(planc_ctx *ctx, int slot, long rows, const long *indptr, long nnz, SpmmPlan *plan) {
  const long cap = nnz / SP_SHORT + nnz / SP_SEG + 1;
  char *w = (char *)ws_get(ctx, slot, 256 + sizeof(SpSeg) * (size_t)cap);
  if (!w) return set_error(ctx, PLANC_ENOMEM, "spmm: workspace");
  plan->cnt = (int *)w;
  plan->seg = w + 256;
  plan->segs = cap - 1;
  plan->parts = 2 * (nnz / SP_SEG);
  if (rows <= 0) return PLANC_OK;
  spmm_plan_zero_kernel<<<1, 64, 0, ctx->stream>>>(plan->cnt);
  PLANC_LAUNCH_CHECK(ctx);
  spmm_plan_kernel<<<(unsigned)((rows + 255) / 256), 256, 0, ctx->stream>>>(rows, indptr, plan->cnt,
                                                                           (SpSeg *)plan->seg);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

template <int G>
static int spmm_launch(planc_ctx *ctx, const SpmmPlan &pl, long rows, const long *indptr, const int *indices,
                       const float *values, const float *F, long ldf, int k, float *out, long ors, long ocs) {
  if (!pl.cnt) {
    const int nsegb = (int)std::min<long>((rows + 3) / 4, 1L << 20);
    const long nb = nsegb + (rows + 256 / G - 1) / (256 / G);
    spmm_kernel<G, false><<<(unsigned)nb, 256, 0, ctx->stream>>>(rows, indptr, indices, values, F, ldf, k, out, ors, ocs,
                                                                nsegb, nullptr, nullptr, nullptr);
    PLANC_LAUNCH_CHECK(ctx);
    return PLANC_OK;
  }
  float *partial = (float *)ws_get(ctx, 21, sizeof(float) * 4 * G * (size_t)std::max(pl.parts, 1L));
  if (!partial) return set_error(ctx, PLANC_ENOMEM, "spmm: workspace");
  const int nsegb = (int)std::min<long>((pl.segs + 3) / 4, 8L * ctx->num_cu);
  const long nb = nsegb + (rows + 256 / G - 1) / (256 / G);
  const SpSeg *seg = (const SpSeg *)pl.seg;
  spmm_kernel<G, true><<<(unsigned)nb, 256, 0, ctx->stream>>>(rows, indptr, indices, values, F, ldf, k, out, ors, ocs,
                                                              nsegb, pl.cnt, seg, partial);
  PLANC_LAUNCH_CHECK(ctx);
  if (pl.parts > 0) {
    const long fb = std::min<long>((pl.segs + 256 / G - 1) / (256 / G), 4L * ctx->num_cu);
    spmm_finish_kernel<G><<<(unsigned)fb, 256, 0, ctx->stream>>>(pl.cnt, seg, partial, k, out, ors, ocs);
    PLANC_LAUNCH_CHECK(ctx);
  }
  return PLANC_OK;
}

int spmm_csr(planc_ctx *ctx, const SpmmPlan &plan, long rows, const long *indptr, const int *indices,
             const float *values, const float *F, long ldf, int k, float *out, long ors, long ocs) {
  if (k <= 0 || k > 64) return set_error(ctx, PLANC_EUNSUPPORTED, "spmm: k must be 1..64");
  if (rows <= 0) return PLANC_OK;
  if (k <= 16) return spmm_launch<4>(ctx, plan, rows, indptr, indices, values, F, ldf, k, out, ors, ocs);
  if (k <= 32) return spmm_launch<8>(ctx, plan, rows, indptr, indices, values, F, ldf, k, out, ors, ocs);
  return spmm_launch<16>(ctx, plan, rows, indptr, indices, values, F, ldf, k, out, ors, ocs);
}

// k-major copies of W (m x k) and H (n x k) in workspace slots; returns them.
static int kmajor(planc_ctx *ctx, int slot, const float *X, long rows, long ldx, int k, float **out) {
  float *p = (float *)ws_get(ctx, slot, sizeof(float) * (size_t)rows * k);
  if (!p) return set_error(ctx, PLANC_ENOMEM, "sparse: factor copy");
  *out = p;
  return transpose_to_k_major(ctx, X, rows, ldx, k, p, k);
}

// Row pitch of the products' k-major copies: rows of whole 16-byte words (what
// lies past k is read into lanes that are not stored).
static long pitch4(int k) { return (k + 3) / 4 * 4; }

static int kmajor4(planc_ctx *ctx, int slot, const float *X, long rows, long ldx, int k, float **out) {
  float *p = (float *)ws_get(ctx, slot, sizeof(float) * (size_t)rows * pitch4(k));
  if (!p) return set_error(ctx, PLANC_ENOMEM, "sparse: factor copy");
  *out = p;
  return transpose_to_k_major(ctx, X, rows, ldx, k, p, pitch4(k));
}

int spmm_colmajor(planc_ctx *ctx, long rows, long cols, const long *indptr, const int *indices,
                  const float *values, const float *F, long ldf, int k, float *out, long ldo) {
  float *Fk = nullptr;
  int rc = kmajor4(ctx, kSparseSlot0 + 1, F, cols, ldf, k, &Fk);
  if (rc) return rc;
  return spmm_csr(ctx, SpmmPlan{}, rows, indptr, indices, values, Fk, pitch4(k), k, out, 1, ldo);
}

int sparse_fit_error(planc_ctx *ctx, long m, long n, const long *indptr, const int *indices,
                     const float *values, const float *W, long ldw, const float *H, long ldh, int k,
                     double *d_err) {
  if (k <= 0 || k > 64) return set_error(ctx, PLANC_EUNSUPPORTED, "sparse error: k must be 1..64");
  float *Wk = nullptr, *Hk = nullptr;
  int rc = kmajor(ctx, kSparseSlot0 + 0, W, m, ldw, k, &Wk);
  if (rc) return rc;
  if ((rc = kmajor(ctx, kSparseSlot0 + 1, H, n, ldh, k, &Hk))) return rc;
  const int nb = (int)std::min<long>(1024, std::max<long>(1, (m + 3) / 4));
  double *part = (double *)ws_get(ctx, kSparseSlot0 + 2, sizeof(double) * (2 * (size_t)nb + 2 * (size_t)k * k));
  if (!part) return set_error(ctx, PLANC_ENOMEM, "sparse error: workspace");
  double *WtW = part + 2 * nb, *HtH = WtW + (size_t)k * k;
  sparse_fit_kernel<<<nb, 256, 0, ctx->stream>>>(m, indptr, indices, values, Wk, Hk, k, part);
  PLANC_LAUNCH_CHECK(ctx);
  if ((rc = gram(ctx, W, m, k, ldw, WtW))) return rc;
  if ((rc = gram(ctx, H, n, k, ldh, HtH))) return rc;
  sparse_fit_finalize_kernel<<<1, 64, 0, ctx->stream>>>(part, nb, WtW, HtH, k, d_err);
  PLANC_LAUNCH_CHECK(ctx);
  return PLANC_OK;
}

int sparse_products(planc_ctx *ctx, long m, long n, long nnz, const long *indptr, const int *indices,
                    const float *values, SparseOps *ops) {
  long *tptr = (long *)ws_get(ctx, kSparseSlot0 + 3, sizeof(long) * (size_t)(n + 1) +
                                                         (sizeof(int) + sizeof(float)) * (size_t)std::max(nnz, 1L));
  if (!tptr) return set_error(ctx, PLANC_ENOMEM, "sparse: transposed copy");
  int *tidx = (int *)(tptr + n + 1);
  float *tval = (float *)(tidx + std::max(nnz, 1L));
  int rc = csr_transpose(ctx, m, n, nnz, indptr, indices, values, tptr, tidx, tval);
  if (rc) return rc;
  ops->t_indptr = tptr;
  ops->t_indices = tidx;
  ops->t_values = tval;
  if ((rc = spmm_plan(ctx, 19, m, indptr, nnz, &ops->plan))) return rc;
  return spmm_plan(ctx, 20, n, tptr, nnz, &ops->t_plan);
}

int sparse_wta(planc_ctx *ctx, const SparseOps &o, long m, long n, const float *W, int k, float *out) {
  float *Wk = nullptr;
  int rc = kmajor4(ctx, kSparseSlot0 + 0, W, m, m, k, &Wk);
  if (rc) return rc;
  return spmm_csr(ctx, o.t_plan, n, o.t_indptr, o.t_indices, o.t_values, Wk, pitch4(k), k, out, k, 1);
}

int sparse_ah(planc_ctx *ctx, const SparseOps &o, long m, long n, const long *indptr, const int *indices,
              const float *values, const float *H, int k, float *out) {
  float *Hk = nullptr;
  int rc = kmajor4(ctx, kSparseSlot0 + 1, H, n, n, k, &Hk);
  if (rc) return rc;
  return spmm_csr(ctx, o.plan, m, indptr, indices, values, Hk, pitch4(k), k, out, 1, m);
}

}  // namespace planc
