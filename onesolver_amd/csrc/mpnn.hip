// mpnn.hip -- training and inference kernels of the warm-start network.
//
// A 3-layer message-passing network over the coupling graph of a dense
// instance predicts per-spin marginals of good annealed states.  Per layer
//   M = A r(H)                (neighbour aggregation, bf16 MFMA, fp32 acc)
//   Z = H r(Ws) + M r(Wm) + b,  H' = relu(Z)          (node update, fp32)
// with A = offdiag(Q) / scale (bf16), r = bf16 rounding of the weights and
// of the aggregation input; head: logit = H r(wo) + bo, p = sigmoid(logit).
// Features of spin i: (Q_ii, sum_j Q_ij) / scale, [i == 0], 1; padded to 64
// columns so every layer has 64 inputs (the zero columns of layer 1 stay
// zero in value and gradient).  Rows are padded to a multiple of 64 with
// zero features and zero couplings; they take no part in the loss, and
// their gradients are zero.
//
// Activations of a minibatch of B instances live in [B][Np][64] fp32 arrays
// (row = spin) and, as MFMA B operands, in [B][64][Np] bf16 (feature-major).
// A layer is one launch in each direction, a work-group 64 rows of one
// instance: the aggregation's 64 x 64 tile goes through LDS straight into the
// node update (forward) or the activation's gradient (backward), and the
// backward launch also makes the rows' share of the weight gradients.  Those
// are reduced deterministically: rows of a work-group in order, then the
// work-groups in a fixed tree.
#include "os_mpnn.h"

namespace os {

typedef __bf16 mp_bf16x8 __attribute__((ext_vector_type(8)));
typedef float mp_f32x16 __attribute__((ext_vector_type(16)));

namespace {

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__device__ __forceinline__ float bf16_round(float f) {
  return __uint_as_float((uint32_t)to_bf16(f) << 16);
}

}  // namespace

// ---- features --------------------------------------------------------------

// rowstat[b][i] = (sum_{j != i} Q_ij^2, sum_{j != i} Q_ij) of instance q[b]:
// one wave per row, so the FP64 matrices are read once in 512-byte requests
// (one thread per row, 8 KB apart, took 146 us for 16 x n=1024; 21 us now).
__global__ __launch_bounds__(256) void mp_rowstat_kernel(int B, int n, const double *__restrict__ q,
                                                         double *__restrict__ rowstat) {
  const size_t t = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= (size_t)B * n) return;
  const int i = (int)(t % n), lane = threadIdx.x & 63;
  const double *row = q + t * n;
  double s2 = 0.0, s1 = 0.0;
#pragma unroll 4
  for (int j = lane; j < n; j += 64) {
    const double v = j == i ? 0.0 : row[j];
    s2 = fma(v, v, s2);
    s1 += v;
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    s2 += __shfl_xor(s2, o);
    s1 += __shfl_xor(s1, o);
  }
  if (lane == 0) {
    rowstat[2 * t] = s2;
    rowstat[2 * t + 1] = s1;
  }
}

__global__ __launch_bounds__(256) void mp_scale_kernel(int n, const double *__restrict__ rowstat,
                                                       double *__restrict__ scale) {
  __shared__ double part[256];
  const int b = blockIdx.x;
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += rowstat[2 * ((size_t)b * n + i)];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    s = sqrt(part[0] / n);
    scale[b] = s > 0.0 ? s : 1.0;
  }
}

// A[b][i][j] (bf16) and the features X0[b][i][:], XT0[b][:][i] (bf16).  A
// work-group is one row.  The quotient by the scale is formed from its
// reciprocal with one correction by the remainder: three products instead of
// a division's sequence per coupling.
__global__ __launch_bounds__(256) void mp_fill_kernel(int n, int Np, const double *__restrict__ q,
                                                      const double *__restrict__ rowstat,
                                                      const double *__restrict__ scale,
                                                      uint16_t *__restrict__ A,
                                                      float *__restrict__ X0,
                                                      uint16_t *__restrict__ XT0) {
  const int b = blockIdx.y, i = blockIdx.x;
  const double sc = scale[b], rc = 1.0 / sc;
  const double *row = q + ((size_t)b * n + i) * n;
  uint16_t *a = A + ((size_t)b * Np + i) * Np;
  for (int j = threadIdx.x; j < Np; j += 256) {
    float v = 0.0f;
    if (i < n && j < n && i != j) {
      const double x = row[j], t = x * rc;
      v = (float)fma(fma(-t, sc, x), rc, t);
      if (!isfinite(v)) v = (float)(x / sc);  // the remainder of an infinity is NaN
    }
    a[j] = to_bf16(v);
  }
  const int j = threadIdx.x;
  if (j < 64) {
    float f = 0.0f;
    if (i < n) {
      if (j == 0) f = (float)(row[i] / sc);
      else if (j == 1) f = (float)(rowstat[2 * ((size_t)b * n + i) + 1] / sc);
      else if (j == 2) f = i == 0 ? 1.0f : 0.0f;
      else if (j == 3) f = 1.0f;
    }
    X0[((size_t)b * Np + i) * 64 + j] = f;
    XT0[((size_t)b * 64 + j) * Np + i] = to_bf16(f);
  }
}

// ---- sparse instances (CSR batch) -------------------------------------------
// The network on a batch of CSR instances, as on each instance's dense
// matrix: one row per spin, instance i at rows spin_off.. (instance-major,
// padded to a multiple of 64 with zero rows).  The scale of instance i is
// the dense one over scale_rows[i] rows (its size in the dense layout the
// network was trained on; n when null): rows without couplings add nothing
// but the row count.  A_jl = bf16((float)(Q_jl / scale)) as in mp_fill_kernel.

// scale[i] = sqrt(sum_j (sum_{l != j} Q_jl^2) / rows_i), the row sums first
__global__ void mp_csr_scale_kernel(int I, const CsrInst *__restrict__ inst,
                                    const int32_t *__restrict__ row_ptr,
                                    const double *__restrict__ val,
                                    const int32_t *__restrict__ scale_rows,
                                    double *__restrict__ scale) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= I) return;
  const CsrInst d = inst[i];
  const int32_t *rp = row_ptr + d.row_off;
  const double *vl = val + d.csr_off;
  double s = 0.0;
  for (int j = 0; j < d.n; ++j) {
    double s2 = 0.0;
    for (int k = rp[j]; k < rp[j + 1]; ++k) s2 += vl[k] * vl[k];
    s += s2;
  }
  const int rows = scale_rows ? scale_rows[i] : d.n;
  s = sqrt(s / rows);
  scale[i] = s > 0.0 ? s : 1.0;
}

// features of spin j: (Q_jj, sum_l Q_jl) / scale, 0, 1 (grid: rows / 256, I)
__global__ __launch_bounds__(256) void mp_csr_features_kernel(
    const CsrInst *__restrict__ inst, const int32_t *__restrict__ row_ptr,
    const double *__restrict__ val, const double *__restrict__ diag,
    const double *__restrict__ scale, float *__restrict__ X0) {
  const CsrInst d = inst[blockIdx.y];
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= d.n) return;
  const int32_t *rp = row_ptr + d.row_off;
  const double *vl = val + d.csr_off;
  const double sc = scale[blockIdx.y];
  double s1 = 0.0;
  for (int k = rp[j]; k < rp[j + 1]; ++k) s1 += vl[k];
  float *x = X0 + (size_t)(d.spin_off + j) * 64;
  x[0] = (float)(diag[d.spin_off + j] / sc);
  x[1] = (float)(s1 / sc);
  x[2] = 0.0f;
  x[3] = 1.0f;
  for (int f = 4; f < 64; ++f) x[f] = 0.0f;
}

// M[row j] = sum_k A_{j col_k} bf16(Hin[col_k]) in fp32 (one wave per spin,
// lane = feature; grid: rows / 4, I)
__global__ __launch_bounds__(256) void mp_csr_agg_kernel(
    const CsrInst *__restrict__ inst, const int32_t *__restrict__ row_ptr,
    const int32_t *__restrict__ col, const double *__restrict__ val,
    const double *__restrict__ scale, const float *__restrict__ Hin, float *__restrict__ M) {
  const CsrInst d = inst[blockIdx.y];
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int f = threadIdx.x & 63;
  if (j >= d.n) return;
  const int32_t *rp = row_ptr + d.row_off;
  const int32_t *cl = col + d.csr_off;
  const double *vl = val + d.csr_off;
  const double sc = scale[blockIdx.y];
  const float *h = Hin + (size_t)d.spin_off * 64 + f;
  float acc = 0.0f;
  for (int k = rp[j]; k < rp[j + 1]; ++k) {
    const float a = bf16_round((float)(vl[k] / sc));
    acc = fmaf(a, bf16_round(h[(size_t)cl[k] * 64]), acc);
  }
  M[(size_t)(d.spin_off + j) * 64 + f] = acc;
}

void mp_launch_csr_features(hipStream_t st, int I, int max_n, const CsrInst *inst,
                            const int32_t *row_ptr, const double *val, const double *diag,
                            const int32_t *scale_rows, double *scale, float *X0) {
  if (I == 0 || max_n == 0) return;
  mp_csr_scale_kernel<<<(I + 63) / 64, 64, 0, st>>>(I, inst, row_ptr, val, scale_rows, scale);
  OS_HIP_CHECK(hipGetLastError());
  mp_csr_features_kernel<<<dim3((max_n + 255) / 256, I), 256, 0, st>>>(inst, row_ptr, val, diag,
                                                                       scale, X0);
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_csr_agg(hipStream_t st, int I, int max_n, const CsrInst *inst,
                       const int32_t *row_ptr, const int32_t *col, const double *val,
                       const double *scale, const float *Hin, float *M) {
  if (I == 0 || max_n == 0) return;
  mp_csr_agg_kernel<<<dim3((max_n + 3) / 4, I), 256, 0, st>>>(inst, row_ptr, col, val, scale,
                                                              Hin, M);
  OS_HIP_CHECK(hipGetLastError());
}

// ---- layers ------------------------------------------------------------------
namespace {

constexpr int kRows = 64;  // rows of a work-group
constexpr int kLd = 68;    // row stride of the LDS tiles: 16-byte rows, no bank conflicts
constexpr int kUnroll = 4;  // aggregation: k steps (of 16) requested at once, twice

typedef float Tile[kRows][kLd];

__device__ __forceinline__ void load_tile(Tile &dst, const float *__restrict__ src) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int idx = threadIdx.x + 256 * k;
    *reinterpret_cast<float4 *>(&dst[idx >> 4][4 * (idx & 15)]) =
        reinterpret_cast<const float4 *>(src)[idx];
  }
}

// Rows r0.. of A . X (A row-major, X feature-major, both bf16, fp32 sums) into
// y: wave w makes rows 32 (w/2).. x features 32 (w%2)...  Four k steps are in
// flight while four are multiplied; requested one by one, each step waited
// for L2 (a layer's aggregation and node update took 19 + 21 us at 16 x n=1024,
// the one launch takes 27).
__device__ __forceinline__ void agg_tile(int Np, const uint16_t *__restrict__ A,
                                         const uint16_t *__restrict__ XT, int r0, Tile &y) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int lc = lane & 31, kh = lane >> 5;
  const int rw = 32 * (w >> 1), f0 = 32 * (w & 1);
  const uint4 *arow = reinterpret_cast<const uint4 *>(A + (size_t)(r0 + rw + lc) * Np) + kh;
  const uint4 *xrow = reinterpret_cast<const uint4 *>(XT + (size_t)(f0 + lc) * Np) + kh;
  mp_f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  const int steps = Np / 16;  // a multiple of kUnroll: Np is one of 64
  uint4 a[kUnroll], x[kUnroll];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    a[u] = arow[2 * u];
    x[u] = xrow[2 * u];
  }
  for (int s = kUnroll; s <= steps; s += kUnroll) {
    uint4 a1[kUnroll], x1[kUnroll];
    const int sn = min(s, steps - kUnroll);  // past the end: the last steps again, unused
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      a1[u] = arow[2 * (sn + u)];
      x1[u] = xrow[2 * (sn + u)];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mp_bf16x8, a[u]),
                                                    __builtin_bit_cast(mp_bf16x8, x[u]), acc, 0,
                                                    0, 0);
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      a[u] = a1[u];
      x[u] = x1[u];
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) y[rw + 8 * (i >> 2) + 4 * kh + (i & 3)][f0 + lc] = acc[i];
}

// c[i][j] += sum_k x[tr + 16 i][k] w[k][4 to + j] in order of k, for this
// thread's 4 x 4 part (tr = tid % 16, to = tid / 16): eight 16-byte reads for
// 64 products.
__device__ __forceinline__ void rows_times(const Tile &x, const Tile &w, int tr, int to,
                                           float (&c)[4][4]) {
  for (int k = 0; k < 64; k += 4) {
    float xv[4][4], wv[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<float4 *>(xv[i]) = *reinterpret_cast<const float4 *>(&x[tr + 16 * i][k]);
      *reinterpret_cast<float4 *>(wv[i]) = *reinterpret_cast<const float4 *>(&w[k + i][4 * to]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) c[i][j] = fmaf(xv[i][u], wv[u][j], c[i][j]);
  }
}

// c[i][j] += sum_k x[tr + 16 i][k] w[4 to + j][k] in order of k.
__device__ __forceinline__ void rows_times_t(const Tile &x, const Tile &w, int tr, int to,
                                             float (&c)[4][4]) {
  for (int k = 0; k < 64; k += 4) {
    float xv[4][4], wv[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<float4 *>(xv[i]) = *reinterpret_cast<const float4 *>(&x[tr + 16 * i][k]);
      *reinterpret_cast<float4 *>(wv[i]) = *reinterpret_cast<const float4 *>(&w[4 * to + i][k]);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) c[i][j] = fmaf(xv[i][u], wv[j][u], c[i][j]);
  }
}

// out[a][o] = sum_r x[r][a] g[r][o] in order of r (a = 4 (tid / 16).., o = 4 (tid % 16)..).
__device__ __forceinline__ void cols_times(const Tile &x, const Tile &g, float *__restrict__ out) {
  const int ta = threadIdx.x >> 4, to = threadIdx.x & 15;
  float c[4][4] = {};
#pragma unroll 4
  for (int r = 0; r < kRows; ++r) {
    float xv[4], gv[4];
    *reinterpret_cast<float4 *>(xv) = *reinterpret_cast<const float4 *>(&x[r][4 * ta]);
    *reinterpret_cast<float4 *>(gv) = *reinterpret_cast<const float4 *>(&g[r][4 * to]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) c[i][j] = fmaf(xv[i], gv[j], c[i][j]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4 *>(out + (4 * ta + i) * 64 + 4 * to) =
        make_float4(c[i][0], c[i][1], c[i][2], c[i][3]);
}

// bf16 of a thread's 4 x 4 part (rows tr + 16 i, features 4 to + j) into the
// feature-major array xt at row r0 of its instance, through LDS so that the
// stores are 16 bytes.  t: 64 x 72 bf16 of LDS nobody reads any more.
__device__ __forceinline__ void store_feature_major(const float (&c)[4][4], int tr, int to,
                                                    uint16_t (*t)[72], int Np, int r0,
                                                    uint16_t *__restrict__ xt) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) t[4 * to + j][tr + 16 * i] = to_bf16(c[i][j]);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int idx = threadIdx.x + 256 * k;
    *reinterpret_cast<uint4 *>(xt + (size_t)(idx >> 3) * Np + r0 + 8 * (idx & 7)) =
        *reinterpret_cast<const uint4 *>(&t[idx >> 3][8 * (idx & 7)]);
  }
}

}  // namespace

// Forward: M = A r(Hin) (kAgg: from XT, also stored; otherwise M is given),
// Z = Hin Ws + M Wm + b, H = relu(Z), HT = bf16(H) feature-major.  kHead: the
// last layer -- instead of H and HT the head: logit = bo + H wo, p =
// sigmoid(logit) and, with labels, dlogit and the work-group's sum of BCE
// terms.  Canonical labels: y_i = x_i xor (1 - x_0) (spin 0 is pinned to 1).
template <bool kAgg, bool kHead>
__global__ __launch_bounds__(256) void mp_layer_fwd_kernel(
    int n, int Np, const uint16_t *__restrict__ A, const uint16_t *__restrict__ XT,
    const float *__restrict__ Hin, float *__restrict__ M, const float *__restrict__ wl,
    float *__restrict__ Z, float *__restrict__ H, uint16_t *__restrict__ HT,
    const float *__restrict__ wo, const uint8_t *__restrict__ labels, float inv_count,
    float *__restrict__ p, float *__restrict__ dlogit, double *__restrict__ lossblock) {
  __shared__ __align__(16) Tile ws, wm, xs, ms;
  const int b = blockIdx.y, r0 = blockIdx.x * kRows;
  const size_t row0 = (size_t)b * Np + r0;
  load_tile(ws, wl);
  load_tile(wm, wl + 4096);
  load_tile(xs, Hin + row0 * 64);
  if (kAgg)
    agg_tile(Np, A + (size_t)b * Np * Np, XT + (size_t)b * 64 * Np, r0, ms);
  else
    load_tile(ms, M + row0 * 64);
  __syncthreads();
  if (kAgg) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int idx = threadIdx.x + 256 * k;
      reinterpret_cast<float4 *>(M + row0 * 64)[idx] =
          *reinterpret_cast<const float4 *>(&ms[idx >> 4][4 * (idx & 15)]);
    }
  }
  const int tr = threadIdx.x & 15, to = threadIdx.x >> 4;
  float z[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float bias = wl[8192 + 4 * to + j];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i][j] = bias;
  }
  rows_times(xs, ws, tr, to, z);
  rows_times(ms, wm, tr, to, z);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const size_t at = (row0 + tr + 16 * i) * 64 + 4 * to;
    *reinterpret_cast<float4 *>(Z + at) = make_float4(z[i][0], z[i][1], z[i][2], z[i][3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) z[i][j] = fmaxf(z[i][j], 0.0f);
    if (!kHead)
      *reinterpret_cast<float4 *>(H + at) = make_float4(z[i][0], z[i][1], z[i][2], z[i][3]);
  }
  __syncthreads();  // the tiles are read
  if (!kHead) {
    if (HT)
      store_feature_major(z, tr, to, reinterpret_cast<uint16_t(*)[72]>(&ws[0][0]), Np, r0,
                          HT + (size_t)b * 64 * Np);
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4 *>(&xs[tr + 16 * i][4 * to]) =
        make_float4(z[i][0], z[i][1], z[i][2], z[i][3]);
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int r = threadIdx.x, i = r0 + r;
  float l = wo[64];
  for (int a = 0; a < 64; a += 4) {
    const float4 h = *reinterpret_cast<const float4 *>(&xs[r][a]);
    l = fmaf(h.x, wo[a], l);
    l = fmaf(h.y, wo[a + 1], l);
    l = fmaf(h.z, wo[a + 2], l);
    l = fmaf(h.w, wo[a + 3], l);
  }
  const float pr = 1.0f / (1.0f + expf(-l));
  p[row0 + r] = pr;
  if (!labels) return;
  float g = 0.0f;
  double term = 0.0;
  if (i < n) {
    const uint8_t *x = labels + (size_t)b * n;
    const float y = (float)(x[i] ^ (uint8_t)(1 - x[0]));
    const double ld = (double)l;
    term = (ld > 0.0 ? ld : 0.0) - ld * (double)y + log1p(exp(-fabs(ld)));
    g = (pr - y) * inv_count;
  }
  dlogit[row0 + r] = g;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) term += __shfl_xor(term, o);
  if (r == 0) lossblock[(size_t)b * gridDim.x + blockIdx.x] = term;
}

// Backward: dH is dlogit wo^T (kTop: the last layer) or dHin + A dMsg (the
// layer above's share through its own rows and through its messages);
// dZ = dH * (Z > 0); with kPrev dHprev = dZ Ws^T and dMsgT = bf16(dZ Wm^T)
// feature-major for the layer below.  The 64 rows' weight gradients
// (Hin^T dZ, M^T dZ, sum dZ, in the layout of the parameters) go to
// partial[work-group], with kTop those of the head (relu(Z)^T dlogit, sum
// dlogit) to head_partial[work-group].
template <bool kTop, bool kPrev>
__global__ __launch_bounds__(256) void mp_layer_bwd_kernel(
    int Np, const uint16_t *__restrict__ A, const uint16_t *__restrict__ dMsgTin,
    const float *__restrict__ dHin, const float *__restrict__ dlogit,
    const float *__restrict__ wo, const float *__restrict__ Z, const float *__restrict__ wl,
    const float *__restrict__ Hin, const float *__restrict__ M, float *__restrict__ dHprev,
    uint16_t *__restrict__ dMsgT, float *__restrict__ partial, float *__restrict__ head_partial) {
  __shared__ __align__(16) Tile dz, hs, ms;
  const int b = blockIdx.y, r0 = blockIdx.x * kRows;
  const size_t row0 = (size_t)b * Np + r0;
  const size_t wg = (size_t)b * gridDim.x + blockIdx.x;
  const int tid = threadIdx.x;
  if (kTop) {
    load_tile(hs, Z + row0 * 64);
    __syncthreads();
    if (tid < 65) {
      float s = 0.0f;
      for (int r = 0; r < kRows; ++r) {
        const float g = dlogit[row0 + r];
        s = tid < 64 ? fmaf(fmaxf(hs[r][tid], 0.0f), g, s) : s + g;
      }
      head_partial[wg * 65 + tid] = s;
    }
    for (int k = tid; k < kRows * 64; k += 256) {
      const int r = k >> 6, o = k & 63;
      dz[r][o] = hs[r][o] > 0.0f ? dlogit[row0 + r] * wo[o] : 0.0f;
    }
    __syncthreads();  // hs is read
  } else {
    agg_tile(Np, A + (size_t)b * Np * Np, dMsgTin + (size_t)b * 64 * Np, r0, dz);
    __syncthreads();
    for (int k = tid; k < kRows * 64; k += 256) {
      const int r = k >> 6, o = k & 63;
      dz[r][o] = Z[row0 * 64 + k] > 0.0f ? dHin[row0 * 64 + k] + dz[r][o] : 0.0f;
    }
  }
  load_tile(hs, Hin + row0 * 64);
  load_tile(ms, M + row0 * 64);
  __syncthreads();
  float *out = partial + wg * 8256;
  cols_times(hs, dz, out);
  cols_times(ms, dz, out + 4096);
  if (tid < 64) {
    float s = 0.0f;
    for (int r = 0; r < kRows; ++r) s += dz[r][tid];
    out[8192 + tid] = s;
  }
  if (!kPrev) return;
  __syncthreads();  // hs and ms are read: they take the weights
  load_tile(hs, wl);
  load_tile(ms, wl + 4096);
  __syncthreads();
  const int tr = tid & 15, to = tid >> 4;
  float c[4][4] = {};
  rows_times_t(dz, hs, tr, to, c);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4 *>(dHprev + (row0 + tr + 16 * i) * 64 + 4 * to) =
        make_float4(c[i][0], c[i][1], c[i][2], c[i][3]);
  float e[4][4] = {};
  rows_times_t(dz, ms, tr, to, e);
  __syncthreads();
  store_feature_major(e, tr, to, reinterpret_cast<uint16_t(*)[72]>(&hs[0][0]), Np, r0,
                      dMsgT + (size_t)b * 64 * Np);
}

// grad[k] = sum of the work-groups' shares: partial[layer][group][8256] for
// the layers' parameters, head_partial[group][65] behind them.  Eight waves
// share 64 parameters: wave w adds groups w, w + 8, ..., then the eight sums
// are added in wave order (one thread per parameter adding all 256 in turn
// took 58 us a matrix at 16 x n=1024; all parameters now take 5.5 us).
__global__ __launch_bounds__(512) void mp_grad_sum_kernel(int layers, int groups,
                                                          const float *__restrict__ partial,
                                                          const float *__restrict__ head_partial,
                                                          float *__restrict__ grad) {
  __shared__ float sums[8][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int k = blockIdx.x * 64 + lane;  // 8256 is a multiple of 64: one layer per block
  const int layer = blockIdx.x * 64 / 8256;
  float s = 0.0f;
  if (layer < layers) {
    const float *src = partial + (size_t)layer * groups * 8256 + (k - layer * 8256);
#pragma unroll 8
    for (int g = w; g < groups; g += 8) s += src[(size_t)g * 8256];
  } else if (k - layers * 8256 < 65) {
    const float *src = head_partial + (k - layers * 8256);
#pragma unroll 8
    for (int g = w; g < groups; g += 8) s += src[(size_t)g * 65];
  }
  sums[w][lane] = s;
  __syncthreads();
  if (w != 0 || k >= layers * 8256 + 65) return;
#pragma unroll
  for (int q = 1; q < 8; ++q) s += sums[q][lane];
  grad[k] = s;
}

// sum of the work-groups' loss terms in a fixed order (one work-group)
__global__ __launch_bounds__(256) void mp_loss_sum_kernel(size_t count,
                                                          const double *__restrict__ terms,
                                                          double *__restrict__ out) {
  __shared__ double part[256];
  double s = 0.0;
  for (size_t k = threadIdx.x; k < count; k += 256) s += terms[k];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = part[0];
}

// Adam on the fp32 master weights; the compute copy rounds weight matrices
// and the head weights to bf16 (biases stay fp32).  mask[k] = 0: padding.
__global__ __launch_bounds__(256) void mp_adam_kernel(int P, const float *__restrict__ grad,
                                                      const uint8_t *__restrict__ kind,
                                                      float *__restrict__ w,
                                                      float *__restrict__ m,
                                                      float *__restrict__ v,
                                                      float *__restrict__ wc, float lr,
                                                      float b1, float b2, float eps, float c1,
                                                      float c2) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= P) return;
  const uint8_t kd = kind[k];
  if (kd == 0) return;
  const float g = grad[k];
  const float mk = b1 * m[k] + (1.0f - b1) * g;
  const float vk = b2 * v[k] + (1.0f - b2) * g * g;
  m[k] = mk;
  v[k] = vk;
  const float wk = w[k] - lr * (mk / c1) / (sqrtf(vk / c2) + eps);
  w[k] = wk;
  wc[k] = kd == 1 ? bf16_round(wk) : wk;
}

__global__ __launch_bounds__(256) void mp_compute_copy_kernel(int P,
                                                              const uint8_t *__restrict__ kind,
                                                              const float *__restrict__ w,
                                                              float *__restrict__ wc) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k >= P) return;
  const uint8_t kd = kind[k];
  wc[k] = kd == 1 ? bf16_round(w[k]) : (kd == 2 ? w[k] : 0.0f);
}

// ---- launchers -----------------------------------------------------------------

void mp_launch_features(hipStream_t st, int B, int n, int Np, const double *q, double *rowstat,
                        double *scale, uint16_t *A, float *X0, uint16_t *XT0) {
  mp_rowstat_kernel<<<(unsigned)(((size_t)B * n + 3) / 4), 256, 0, st>>>(B, n, q, rowstat);
  OS_HIP_CHECK(hipGetLastError());
  mp_scale_kernel<<<B, 256, 0, st>>>(n, rowstat, scale);
  OS_HIP_CHECK(hipGetLastError());
  mp_fill_kernel<<<dim3(Np, B), 256, 0, st>>>(n, Np, q, rowstat, scale, A, X0, XT0);
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_layer_fwd(hipStream_t st, int B, int n, int Np, const uint16_t *A,
                         const uint16_t *XT, const float *Hin, float *M, const float *wl,
                         float *Z, float *H, uint16_t *HT, const MpHead *head) {
  const dim3 grid(Np / kRows, B);
  const MpHead h = head ? *head : MpHead{};
#define OS_FWD(AGG, HEAD)                                                                        \
  mp_layer_fwd_kernel<AGG, HEAD><<<grid, 256, 0, st>>>(n, Np, A, XT, Hin, M, wl, Z, H, HT, h.wo, \
                                                       h.labels, h.inv_count, h.p, h.dlogit,     \
                                                       h.lossblock)
  if (A) {
    if (head) OS_FWD(true, true);
    else OS_FWD(true, false);
  } else {
    if (head) OS_FWD(false, true);
    else OS_FWD(false, false);
  }
#undef OS_FWD
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_layer_bwd(hipStream_t st, int B, int Np, const uint16_t *A,
                         const uint16_t *dMsgTin, const float *dHin, const MpHead *head,
                         const float *Z, const float *wl, const float *Hin, const float *M,
                         float *dHprev, uint16_t *dMsgT, float *partial, float *head_partial) {
  const dim3 grid(Np / kRows, B);
  const MpHead h = head ? *head : MpHead{};
#define OS_BWD(TOP, PREV)                                                                       \
  mp_layer_bwd_kernel<TOP, PREV><<<grid, 256, 0, st>>>(Np, A, dMsgTin, dHin, h.dlogit, h.wo, Z, \
                                                       wl, Hin, M, dHprev, dMsgT, partial,      \
                                                       head_partial)
  if (head) OS_BWD(true, true);
  else if (dHprev) OS_BWD(false, true);
  else OS_BWD(false, false);
#undef OS_BWD
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_grad_sum(hipStream_t st, int layers, int groups, const float *partial,
                        const float *head_partial, float *grad) {
  mp_grad_sum_kernel<<<(layers * 8256 + 65 + 63) / 64, 512, 0, st>>>(layers, groups, partial,
                                                                     head_partial, grad);
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_loss_sum(hipStream_t st, size_t count, const double *terms, double *out) {
  mp_loss_sum_kernel<<<1, 256, 0, st>>>(count, terms, out);
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_adam(hipStream_t st, int P, const float *grad, const uint8_t *kind, float *w,
                    float *m, float *v, float *wc, float lr, float b1, float b2, float eps,
                    int step) {
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  mp_adam_kernel<<<(P + 255) / 256, 256, 0, st>>>(P, grad, kind, w, m, v, wc, lr, b1, b2, eps,
                                                  c1, c2);
  OS_HIP_CHECK(hipGetLastError());
}

void mp_launch_compute_copy(hipStream_t st, int P, const uint8_t *kind, const float *w,
                            float *wc) {
  mp_compute_copy_kernel<<<(P + 255) / 256, 256, 0, st>>>(P, kind, w, wc);
  OS_HIP_CHECK(hipGetLastError());
}

}  // namespace os
