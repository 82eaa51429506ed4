// energy.hip -- FP64 QUBO energies and field refresh on the GPU.
//
// For states X (R x N, bit-packed rows of W = ceil(N/32) words) and the
// symmetric FP64 matrix Q, Y = X Q is accumulated in FP64 on
// v_mfma_f64_16x16x4_f64, and
//   E_r   = 1/2 * sum_j x_rj (Y_rj + Q_jj)           (= sum_{i<=j} Q_ij x_ri x_rj,
//                                                      annealing.hpp:31-40)
//   h_rj  = Q_jj + Y_rj - Q_jj x_rj                  (local field of spin j)
// The matrix instruction adds its four products as a chain of fused
// multiply-adds in ascending k, so Y_rj is the same chain over k = 0 .. N-1
// whatever the tile.  Energies are reduced in a fixed order (columns 16 apart,
// 16-lane shuffle tree, then blocks of 128 columns in ascending order), also
// the same for every tile, so results are bit-reproducible run to run.
#include "os_kernels.h"

namespace os {

namespace {
constexpr int kTN = 128;  // columns per tile

typedef double f64x4 __attribute__((ext_vector_type(4)));
}  // namespace

__global__ __launch_bounds__(256) void pack_bytes_kernel(const uint8_t *__restrict__ bytes, int n,
                                                          int count, int W,
                                                          uint32_t *__restrict__ bits) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total = (size_t)count * W;
  if (idx >= total) return;
  const size_t r = idx / W;
  const int w = (int)(idx % W);
  uint32_t v = 0;
  for (int b = 0; b < 32; ++b) {
    const int j = w * 32 + b;
    if (j < n && bytes[r * n + j]) v |= 1u << b;
  }
  bits[idx] = v;
}

__global__ __launch_bounds__(256) void unpack_bits_kernel(const uint32_t *__restrict__ bits, int n,
                                                           int count, int W,
                                                           uint8_t *__restrict__ bytes) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total = (size_t)count * n;
  if (idx >= total) return;
  const size_t r = idx / n;
  const int j = (int)(idx % n);
  bytes[idx] = (uint8_t)((bits[r * W + (j >> 5)] >> (j & 31)) & 1u);
}

// Work-group: four waves of two column tiles each share 16 RT states, so its
// tile is 16 RT states x 128 columns.  Lane (lk = lane / 16, li = lane % 16)
// supplies x of state li and Q of column li at k = lk and holds, in element e
// of a tile, state lk + 4 e and column li.  Each wave reads its columns of Q
// straight into operand registers, 32 k ahead: no LDS stage and no barrier on
// the way (a form with both spent ~4000 cycles a stage waiting).
//
// FP64 matrix rate bounds it where the chip is full: 4096 states at N = 8192
// 14.0 -> 9.4 ms (59 of the 72 TFLOP/s that a large FP64 product reaches here),
// 16384 at N = 1024 0.90 -> 0.65 ms; below that the chain over k: 1024 at
// N = 1024 294 -> 56 us, 460 at N = 512 152 -> 19 us.  Before: 8 x 8 outputs a
// thread on the vector unit, both operands from LDS, 128 states a work-group.
//
// kFields: also write h_rj as fp32 into fields[r*ldf + j] and raise
// drift_max (fp32 bits, non-negative) to max |h_rj - old fields value|.
template <bool kFields, int RT>
__global__ __launch_bounds__(256) void xq_mfma_kernel(
    int n, int W, const double *__restrict__ q, int R, const uint32_t *__restrict__ bits,
    double *__restrict__ partial, int ncb, float *__restrict__ fields, int ldf,
    unsigned int *__restrict__ drift_max) {
  constexpr int WC = 4;       // waves, side by side over the columns
  constexpr int CT = 8 / WC;  // column tiles a wave
  constexpr int D = 8;        // steps of 4 k in the ring: one word of a state
  __shared__ double sl[RT * 4][64];
  const int lane = threadIdx.x & 63;
  const int wc = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  // columns fastest, then tiles of states, over two grid dimensions (xq_grid)
  const int cb = blockIdx.x % (unsigned)ncb;
  const int c0 = cb * kTN + 16 * CT * wc;
  unsigned tile = blockIdx.x / (unsigned)ncb;
  if (blockIdx.y) tile += blockIdx.y * (gridDim.x / (unsigned)ncb);
  if ((int64_t)tile * (16 * RT) >= R) return;
  const int r0 = (int)(tile * (16 * RT));
  // instance blockIdx.z: its matrix and its R rows of states / outputs
  q += (size_t)blockIdx.z * n * n;
  bits += (size_t)blockIdx.z * R * W;
  partial += (size_t)blockIdx.z * R * ncb;
  if (kFields) fields += (size_t)blockIdx.z * R * ldf;

  f64x4 acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[t][j][e] = 0.0;

  if (c0 < n) {
    // step s covers k = 4 s + lk; the last step's rows past n are read as row
    // n - 1 and taken as zero, columns past n as column n - 1 and not used
    const int steps = (n + 3) >> 2, last = steps - 1;
    const int lk_last = min(4 * last + lk, n - 1) - 4 * last;
    uint32_t off[CT], off_last[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const uint32_t c = min(c0 + 16 * j + li, n - 1);
      off[j] = (uint32_t)lk * n + c;
      off_last[j] = (uint32_t)lk_last * n + c;
    }
    double b[D][CT];
    auto fetch = [&](int d, int s) {
      const int sp = min(s, last);
      const double *row = q + (size_t)(4 * sp) * n;
#pragma unroll
      for (int j = 0; j < CT; ++j) b[d][j] = row[sp == last ? off_last[j] : off[j]];
    };
    const uint32_t *xrow[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) xrow[t] = bits + (size_t)min(r0 + 16 * t + li, R - 1) * W;
    uint32_t xw[RT], xn[RT];
    auto fetch_x = [&](int word) {
#pragma unroll
      for (int t = 0; t < RT; ++t) xn[t] = xrow[t][min(word, W - 1)];
    };
    auto step = [&](int d) {
      double a[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const uint32_t b1 = (xw[t] >> (4 * d + lk)) & 1u;
        a[t] = __hiloint2double(b1 ? 0x3FF00000 : 0, 0);
      }
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int t = 0; t < RT; ++t)
          acc[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[d][j], acc[t][j], 0, 0, 0);
    };
    fetch_x(0);
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(d, d);
    int s0 = 0;
    for (; 4 * (s0 + D) <= n; s0 += D) {
#pragma unroll
      for (int t = 0; t < RT; ++t) xw[t] = xn[t];
      fetch_x((s0 + D) >> 3);
#pragma unroll
      for (int d = 0; d < D; ++d) {
        step(d);
        fetch(d, s0 + D + d);
      }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) xw[t] = xn[t];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s0 + d < steps) {
        if (4 * (s0 + d) + lk >= n) {
#pragma unroll
          for (int j = 0; j < CT; ++j) b[d][j] = 0.0;
        }
        step(d);
      }
    }
  }

  float dmax = 0.0f;
  double diag[CT];
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const int c = min(c0 + 16 * j + li, n - 1);
    diag[j] = q[(size_t)c * n + c];
  }
  uint32_t xs[RT][4];  // bit j: spin c0 + 16 j + li of the state
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t *x = bits + (size_t)min(r0 + 16 * t + lk + 4 * e, R - 1) * W;
      xs[t][e] = 0;
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        const int c = min(c0 + 16 * j + li, n - 1);
        xs[t][e] |= ((x[c >> 5] >> (c & 31)) & 1u) << j;
      }
    }
  if constexpr (kFields) {
    float old[RT][4][CT];  // all requested before the first is replaced
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < CT; ++j)
          old[t][e][j] = fields[(size_t)min(r0 + 16 * t + lk + 4 * e, R - 1) * ldf +
                                min(c0 + 16 * j + li, n - 1)];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = r0 + 16 * t + lk + 4 * e;
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          const int c = c0 + 16 * j + li;
          if (r < R && c < n) {
            const double h = diag[j] + acc[t][j][e] - (xs[t][e] >> j & 1u ? diag[j] : 0.0);
            dmax = fmaxf(dmax, (float)fabs(h - (double)old[t][e][j]));
            fields[(size_t)r * ldf + c] = (float)h;
          }
        }
      }
  }
  // energy terms: the columns' terms of a state are added 16 apart in ascending
  // order, from wave to wave of the WC that share the state
  for (int ph = 0; ph < WC; ++ph) {
    if (ph == wc) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = r0 + 16 * t + lk + 4 * e;
          double s = ph > 0 ? sl[t * 4 + e][lane] : 0.0;
#pragma unroll
          for (int j = 0; j < CT; ++j)
            if (c0 + 16 * j + li < n && (xs[t][e] >> j & 1u)) s += acc[t][j][e] + diag[j];
          if (ph == WC - 1) {
            // reduce s over the 16 lanes sharing this row (fixed shuffle tree)
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 16);
            if (li == 0 && r < R) partial[(size_t)r * ncb + cb] = 0.5 * s;
          } else {
            sl[t * 4 + e][lane] = s;
          }
        }
    }
    __syncthreads();
  }
  if (kFields) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) dmax = fmaxf(dmax, __shfl_xor(dmax, o, 64));
    if (lane == 0) atomicMax(drift_max, __float_as_uint(dmax));
  }
}

__global__ __launch_bounds__(256) void reduce_partials_kernel(const double *__restrict__ partial,
                                                               int R, int ncb,
                                                               double *__restrict__ out) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= R) return;
  double s = 0.0;
  for (int b = 0; b < ncb; ++b) s += partial[(size_t)r * ncb + b];
  out[r] = s;
}

void launch_pack_bytes(hipStream_t st, const uint8_t *bytes, int n, int count, int W,
                       uint32_t *bits) {
  const size_t total = (size_t)count * W;
  if (total == 0) return;
  pack_bytes_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>(bytes, n, count, W, bits);
  OS_HIP_CHECK(hipGetLastError());
}

void launch_unpack_bits(hipStream_t st, const uint32_t *bits, int n, int count, int W,
                        uint8_t *bytes) {
  const size_t total = (size_t)count * n;
  if (total == 0) return;
  unpack_bits_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>(bits, n, count, W, bytes);
  OS_HIP_CHECK(hipGetLastError());
}

size_t energy_scratch_bytes(int n, int count) {
  const int ncb = (n + kTN - 1) / kTN;
  return sizeof(double) * (size_t)count * ncb;
}

// n <= 64, energies only: one thread per state, in the reference's order
// (sa::energy, annealing.hpp:31-40): one FP64 accumulator over the upper
// triangle row by row, q[i][j] * x_i * x_j for every j >= i (zero terms
// included, as the reference's loop has them; the product by x_i x_j is exact,
// so it goes into the addition's fma).  The work-group stages the triangle in
// LDS with zeros elsewhere, so eight columns at a time need no bounds; every
// thread then reads the same addresses (broadcasts).  The chain of additions
// bounds it: n = 60, 1024 states 46 -> 34 us, 262144 states 121 -> 83 us.
__global__ __launch_bounds__(256) void energy_small_kernel(int n, int W, const double *__restrict__ q,
                                                          int count,
                                                          const uint32_t *__restrict__ bits,
                                                          double *__restrict__ out) {
  __shared__ double ql[64][64];
  const int s = blockIdx.y;
  const double *qs = q + (size_t)s * n * n;
  const int n8 = (n + 7) & ~7;
  {
    const int j = threadIdx.x & 63;
#pragma unroll 8
    for (int i = threadIdx.x >> 6; i < n; i += 4) {
      const double v = qs[i * n + min(j, n - 1)];
      ql[i][j] = j >= i && j < n ? v : 0.0;
    }
  }
  __syncthreads();
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= count) return;
  const uint32_t *x = bits + ((size_t)s * count + r) * W;
  const uint32_t x0 = x[0], x1 = W > 1 ? x[1] : 0u;
  double e = 0.0;
  for (int i = 0; i < n; ++i) {
    const uint32_t xi = (i < 32 ? x0 >> i : x1 >> (i - 32)) & 1u ? 0x3FF00000u : 0u;
    for (int j0 = i & ~7; j0 < n8; j0 += 8) {
      const uint32_t xb = (j0 < 32 ? x0 : x1) >> (j0 & 31);
      double row[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) row[j] = ql[i][j0 + j];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t on = (uint32_t)((int)(xb << (31 - j)) >> 31) & xi;
        e = fma(row[j], __hiloint2double((int)on, 0), e);
      }
    }
  }
  out[(size_t)s * count + r] = e;
}

namespace {

// Grid of xq_mfma_kernel for `tiles` tiles of states by ncb blocks of columns:
// work-items along a dimension stay below 2^32, so beyond 2^24 work-groups the
// tiles go over a second one.
struct XqGrid {
  unsigned x, y;
};
constexpr XqGrid xq_grid(size_t ncb, size_t tiles) {
  const size_t along = tiles < 0xFFFFFF / ncb ? tiles : 0xFFFFFF / ncb;
  return {(unsigned)(ncb * along), (unsigned)((tiles + along - 1) / along)};
}
constexpr bool xq_grid_holds(size_t ncb, size_t states, size_t rt) {
  const size_t tiles = (states + 16 * rt - 1) / (16 * rt);
  const XqGrid g = xq_grid(ncb, tiles);
  return (size_t)g.x * 256 < (size_t)1 << 32 && g.x % ncb == 0 && g.y <= 65535 &&
         (size_t)g.x / ncb * g.y >= tiles && (size_t)g.x / ncb * (g.y - 1) < tiles;
}
static_assert(xq_grid_holds(1, 1, 1) && xq_grid_holds(128, 4096, 2), "one tile, and N = 16384");
static_assert(xq_grid_holds(64, 65535 * 128, 2) && xq_grid_holds(65, 65535 * 128, 2) &&
                  xq_grid_holds(65, 65535 * 128, 1) && xq_grid_holds(1024, 65535 * 128, 2) &&
                  xq_grid_holds(8, 0x7FFFFFFF, 1),
              "8.4 million states at any N, 2^31 - 1 at N = 1024");

}  // namespace

void launch_energy_fp64(hipStream_t st, int n, int W, const double *q, int count,
                        const uint32_t *bits, double *out, double *scratch, float *fields, int ldf,
                        unsigned int *drift_max, int num_instances) {
  if (count <= 0 || num_instances <= 0) return;
  if (!fields && n <= 64) {
    energy_small_kernel<<<dim3((count + 255) / 256, num_instances), 256, 0, st>>>(n, W, q, count,
                                                                                bits, out);
    OS_HIP_CHECK(hipGetLastError());
    return;
  }
  const int ncb = (n + kTN - 1) / kTN;
  double *part = ncb == 1 ? out : scratch;  // one block of columns: its sums are the energies
  // 32 states a work-group read Q half as often as 16, once there is a
  // work-group for each of the 256 CUs; fewer states go by 16.  Energies |
  // fields too, us, 16 against 32: 1024 states at N = 1024 (256 groups of 32)
  // 53 | 73 against 56 | 67, 16 instances of 256 at N = 300 (384) 25 | 55
  // against 30 | 40, 4096 at N = 8192 12.1 ms against 9.3; 460 at N = 512 (60)
  // 19 | 25 against 30 | 33, 1024 at N = 60 (32) 5 | 9 against 7 | 10.  Between
  // 32 and 64 states nothing differs by more than 4 % on that side but small
  // counts lose (1024 at N = 1024: 93 | 99 with 64).
  const size_t groups32 = (size_t)ncb * ((count + 31) / 32) * num_instances;
#define OS_XQ(RT)                                                                                \
  do {                                                                                           \
    const XqGrid g = xq_grid(ncb, ((size_t)count + 16 * RT - 1) / (16 * RT));                    \
    const dim3 grid(g.x, g.y, num_instances);                                                    \
    if (fields)                                                                                  \
      xq_mfma_kernel<true, RT><<<grid, 256, 0, st>>>(n, W, q, count, bits, part, ncb, fields,    \
                                                     ldf, drift_max);                            \
    else                                                                                         \
      xq_mfma_kernel<false, RT><<<grid, 256, 0, st>>>(n, W, q, count, bits, part, ncb, nullptr,  \
                                                      0, nullptr);                               \
  } while (0)
  if (groups32 >= 256) OS_XQ(2);
  else OS_XQ(1);
#undef OS_XQ
  OS_HIP_CHECK(hipGetLastError());
  if (ncb == 1) return;
  const int rows = count * num_instances;
  reduce_partials_kernel<<<(rows + 255) / 256, 256, 0, st>>>(scratch, rows, ncb, out);
  OS_HIP_CHECK(hipGetLastError());
}

}  // namespace os
