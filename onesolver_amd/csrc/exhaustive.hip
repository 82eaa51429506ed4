// exhaustive.hip -- the exact QUBO minimum by enumeration of all 2^n states.
//
// Restates exhaustive::solve (include/exhaustive/exhaustive.hpp:29-167):
// E(x) = sum_{i <= j} q[i][j] x_i x_j over the upper triangle of q (diagonal:
// the linear terms), bit i of the state index is variable i, energies are
// FP64 sums in the reference's order (i ascending, then j >= i ascending,
// exhaustive.hpp:113-128), and of equal energies the lowest state index wins
// (each work-item keeps its first minimum, exhaustive.hpp:129-132, and the
// host takes the first minimal work-item, :158-160).
//
// n <= 20: one thread per state computes that literal energy; a minimum over
// (energy, index) pairs follows.
//
// 20 < n <= 40: thread t owns the states whose top n-L bits equal t and walks
// them in Gray-code order in segments of 2^S states, each from its literal
// energy.
//   pass 1: every thread's minimum energy, and the minimum E_w of them (below);
//   pass 2: only the threads whose minimum is near E_w walk again, their states
//           split over 2^K threads each where few blocks hold them; every state
//           whose walk energy is near E_w gets its literal energy, and the
//           (literal energy, index) minimum of those is the answer.
// "Near" is what rounding can make of the walks, which scales with the
// coefficients and not with E_w (large penalties cancel in the minimum).  With
// exact energies E, let e1, e2 and el bound the rounding of pass 1, pass 2 and
// the literal sums, and x a state of lowest literal energy: where E_w is pass
// 1's energy of y, E(x) <= E(y) + 2 el <= E_w + e1 + 2 el, so pass 1 finds x's
// thread within 2 e1 + 2 el of E_w and pass 2 finds x within e1 + e2 + 2 el:
// the literal minimum is always among the candidates and the result equals the
// reference's.  The bounds are walk_bound()'s.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <vector>

#include "../../include/onesolver.h"
#include "os_kernels.h"

namespace os {

namespace {

constexpr int kMaxN = 40;
constexpr int kLiteralMaxN = 20;
constexpr int kLow = 5;       // pass 2: bits flipped in the unrolled order
constexpr int kMinLow = 7;    // pass 1: bits of an unrolled block
constexpr int kSegBits = 12;  // literal restart every 2^kSegBits states
constexpr int kMaxActive = 16;  // blocks with candidates that pass 2 splits
constexpr int kMaxTopBits = 20;
constexpr int kThreads = 256;

__device__ __forceinline__ bool better(double e, uint64_t x, double be, uint64_t bx) {
  return e < be || (e == be && x < bx);
}

// q (n x n, row stride n, upper triangle used) into LDS as a symmetric
// matrix qs[i][j] = q[min][max] with row stride kMaxN.
__device__ void load_q(int n, const double *__restrict__ q, double *qs) {
  for (int k = threadIdx.x; k < n * n; k += blockDim.x) {
    const int i = k / n, j = k % n;
    const int a = min(i, j), b = max(i, j);
    qs[i * kMaxN + j] = q[(size_t)a * n + b];
  }
}

// The reference's per-state energy and summation order (exhaustive.hpp:113-128).
__device__ double literal_energy(int n, const double *qs, uint64_t x) {
  double e = 0.0;
  for (int i = 0; i < n; ++i) {
    if (!((x >> i) & 1u)) continue;
    e += qs[i * kMaxN + i];
    for (int j = i + 1; j < n; ++j)
      if ((x >> j) & 1u) e += qs[i * kMaxN + j];
  }
  return e;
}

// Field of bit b in state x: q_bb + sum_{i != b} q_bi x_i.
__device__ __forceinline__ double field(int n, const double *qs, uint64_t x, int b) {
  double h = qs[b * kMaxN + b];
  for (int i = 0; i < n; ++i)
    if (i != b && ((x >> i) & 1u)) h += qs[b * kMaxN + i];
  return h;
}

// Minimum over the block of (e, x) pairs, lexicographic; thread 0 writes it.
__device__ void block_min(double e, uint64_t x, double *out_e, uint64_t *out_x) {
  __shared__ double se[kThreads];
  __shared__ uint64_t sx[kThreads];
  se[threadIdx.x] = e;
  sx[threadIdx.x] = x;
  __syncthreads();
  for (int s = kThreads / 2; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s && better(se[threadIdx.x + s], sx[threadIdx.x + s], se[threadIdx.x],
                                       sx[threadIdx.x])) {
      se[threadIdx.x] = se[threadIdx.x + s];
      sx[threadIdx.x] = sx[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out_e[blockIdx.x] = se[0];
    out_x[blockIdx.x] = sx[0];
  }
}

}  // namespace

// One thread per state, n <= 30.  An energy that is NaN or not below DBL_MAX
// never wins (the reference's strict comparison against its DBL_MAX start,
// exhaustive.hpp:108-132); state 0 (energy 0) always competes.
__global__ __launch_bounds__(kThreads) void exh_literal_kernel(int n, const double *__restrict__ q,
                                                               double *__restrict__ out_e,
                                                               uint64_t *__restrict__ out_x) {
  __shared__ double qs[kMaxN * kMaxN];
  load_q(n, q, qs);
  __syncthreads();
  const uint64_t x = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  double e = DBL_MAX;
  uint64_t bx = 0;
  if (x < (1ull << n)) {
    const double v = literal_energy(n, qs, x);
    if (v < DBL_MAX) {
      e = v;
      bx = x;
    }
  }
  block_min(e, bx, out_e, out_x);
}

// Pass 1, 20 < n <= 40; L = n - P bits per thread, 2^P threads: writes every
// thread's minimum energy to tmin and per-block minima of them.
//
// FP64 issue bounds it, so a state costs few instructions.  The fields
// h_j = q_jj + sum_{i != j} q_ij x_i of the low kSegBits bits are kept in
// registers.  Bits 0, 1 and 2 are not walked: with them clear and energy e,
//   min over x0, x1, x2 = e + min(g(h0, h1), h2 + g(h0 + q02, h1 + q12)),
//   g(a, b) = min(min(0, a), b + min(0, a + q01)),
// 16 instructions for 8 states.  Bits 3 .. 6 go once round the Gray cycle in an
// unrolled block whose signs are constants and whose couplings are scalars; a
// higher bit flips once per 128 states.  About 3 instructions a state instead
// of 11 (5 FMAs and a minimum, and a field summed from LDS every 32 states).
// Measured: n = 32 2174 -> 579 us; whole calls n = 31 1459 -> 489 us, n = 25
// 281 -> 153, n = 21 127 -> 117.
template <int B>
__device__ __forceinline__ void flip_high(const double *qs, bool set, double &e,
                                          double (&h)[kSegBits]) {
  const double sb = set ? -1.0 : 1.0;
  int row = B * kMaxN;
  asm volatile("" : "+v"(row));  // or every row is kept in registers
  e = fma(sb, h[B], e);
#pragma unroll
  for (int j = 0; j < kSegBits; ++j)
    if (j != B) h[j] = fma(sb, qs[row + j], h[j]);
}

__global__ __launch_bounds__(kThreads) void exh_min_kernel(int n, int L, const double *__restrict__ q,
                                                           double *__restrict__ tmin,
                                                           double *__restrict__ out_e,
                                                           uint64_t *__restrict__ out_x) {
  __shared__ double qs[kMaxN * kMaxN];
  const int S = min(L, kSegBits);
  const uint64_t t = (uint64_t)blockIdx.x * kThreads + threadIdx.x;
  load_q(n, q, qs);
  __syncthreads();
  auto uniform = [](double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
  };
  double ql[kMinLow][kMinLow];  // q_ij, i < j
#pragma unroll
  for (int i = 0; i < kMinLow; ++i)
#pragma unroll
    for (int j = i + 1; j < kMinLow; ++j) ql[i][j] = uniform(qs[i * kMaxN + j]);
  double emin = DBL_MAX;
  const bool active = t < (1ull << (n - L));
  const int segs = active ? 1 << (L - S) : 0;
  const int blocks = 1 << (S - kMinLow);
  for (int seg = 0; seg < segs; ++seg) {
    const uint64_t x0 = (t << L) | ((uint64_t)seg << S);  // low S bits zero
    double e = literal_energy(n, qs, x0);
    double h[kSegBits];
#pragma unroll
    for (int j = 0; j < kSegBits; ++j) h[j] = qs[j * kMaxN + j];
    for (int i = S; i < n; ++i) {  // (fields of bits from S on are not used)
      const double xi = (x0 >> i) & 1u ? 1.0 : 0.0;
#pragma unroll
      for (int j = 0; j < kSegBits; ++j) h[j] = fma(xi, qs[i * kMaxN + j], h[j]);
    }
    for (int blk = 0;;) {
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const double a = fmin(fmin(0.0, h[0]), h[1] + fmin(0.0, h[0] + ql[0][1]));
        const double h0 = h[0] + ql[0][2], h1 = h[1] + ql[1][2];
        const double b = fmin(fmin(0.0, h0), h1 + fmin(0.0, h0 + ql[0][1]));
        emin = fmin(emin, e + fmin(a, h[2] + b));
        // the next bit of the cycle: state k ^ (k >> 1) of bits 3 .. 6 so far
        const int f = k < 15 ? 3 + __builtin_ctz(k + 1) : 6;
        const bool set = ((k ^ (k >> 1)) >> (f - 3)) & 1;
        e = set ? e - h[f] : e + h[f];
#pragma unroll
        for (int j = 0; j < kMinLow; ++j)
          if (j != f) {
            const double c = j < f ? ql[j][f] : ql[f][j];
            h[j] = set ? h[j] - c : h[j] + c;
          }
        __builtin_amdgcn_sched_barrier(0);
      }
      // the fields of the bits above followed none of it: the cycle ends where
      // it began
      if (++blk == blocks) break;
      const int B = kMinLow + __builtin_ctz((unsigned)blk);
      // bit B of the Gray code of blk - 1
      const bool set = (((blk - 1) ^ ((blk - 1) >> 1)) >> (B - kMinLow)) & 1;
      switch (B) {
        case 7: flip_high<7>(qs, set, e, h); break;
        case 8: flip_high<8>(qs, set, e, h); break;
        case 9: flip_high<9>(qs, set, e, h); break;
        case 10: flip_high<10>(qs, set, e, h); break;
        default: flip_high<11>(qs, set, e, h); break;
      }
    }
  }
  static_assert(kSegBits == 12 && kMinLow == 7, "the flips above");
  if (active) tmin[t] = emin;
  block_min(emin, 0, out_e, out_x);
}

// Blocks of pass 1 that hold a candidate.
struct ActiveBlocks {
  int count;
  int id[kMaxActive];
};

// Pass 2: walks the states of the threads of pass 1 with tmin <= thr1 and writes
// per-block (literal energy, index) minima of the candidates e_walk <= thr2.  A
// walk energy that is NaN (sums beyond FP64) is a candidate.  A thread takes
// 2^(L-K) of a pass-1 thread's 2^L states; blocks are those of `act`, 2^K each,
// or all of them where act.count is 0.
__global__ __launch_bounds__(kThreads) void exh_gray_kernel(int n, int L, int K, ActiveBlocks act,
                                                            const double *__restrict__ q,
                                                            double thr1, double thr2,
                                                            const double *__restrict__ tmin,
                                                            double *__restrict__ out_e,
                                                            uint64_t *__restrict__ out_x) {
  __shared__ double qs[kMaxN * kMaxN];
  const uint64_t block =
      act.count ? ((uint64_t)act.id[blockIdx.x >> K] << K) + (blockIdx.x & ((1u << K) - 1u))
                : blockIdx.x;
  const uint64_t t = block * kThreads + threadIdx.x;
  L -= K;
  const int S = min(L, kSegBits);
  bool active = t < (1ull << (n - L));
  if (active) active = !(tmin[t >> K] > thr1);
  if (!__syncthreads_or(active)) {  // no candidate in this block
    if (threadIdx.x == 0) {
      out_e[blockIdx.x] = DBL_MAX;
      out_x[blockIdx.x] = 0;
    }
    return;
  }
  load_q(n, q, qs);
  __syncthreads();
  // the off-diagonal part of the low kLow x kLow block of q in registers:
  // ql[i][j] = q_ij for i < j
  double ql[kLow][kLow];
#pragma unroll
  for (int i = 0; i < kLow; ++i)
#pragma unroll
    for (int j = i + 1; j < kLow; ++j) ql[i][j] = qs[i * kMaxN + j];
  double emin = DBL_MAX;
  uint64_t xmin = 0;
  const int segs = active ? 1 << (L - S) : 0;
  const int blocks = 1 << (S - kLow);
  for (int seg = 0; seg < segs; ++seg) {
    // segment start: low S bits zero
    uint64_t xhi = (t << L) | ((uint64_t)seg << S);
    double e = literal_energy(n, qs, xhi);
    double h[kLow], s[kLow];
#pragma unroll
    for (int j = 0; j < kLow; ++j) {
      h[j] = field(n, qs, xhi, j);
      s[j] = 1.0;  // 1 - 2 x_j
    }
    for (int blk = 0; blk < blocks; ++blk) {
      // low kLow bits at the block start: bit kLow-1 of the Gray code of 2^kLow * blk
      const uint32_t low0 = (blk & 1) ? 1u << (kLow - 1) : 0u;
#pragma unroll
      for (int pos = 0; pos < (1 << kLow); ++pos) {
        if (pos > 0) {
          const int b = __builtin_ctz(pos);
          e = fma(s[b], h[b], e);
#pragma unroll
          for (int j = 0; j < kLow; ++j)
            if (j != b) h[j] = fma(s[b], j < b ? ql[j][b] : ql[b][j], h[j]);
          s[b] = -s[b];
        }
        if (!(e > thr2)) {
          const uint64_t x = xhi | (low0 ^ (uint32_t)(pos ^ (pos >> 1)));
          const double v = literal_energy(n, qs, x);
          if (better(v, x, emin, xmin)) {
            emin = v;
            xmin = x;
          }
        }
      }
      if (blk + 1 < blocks) {
        // the low bits end at low0 ^ 2^(kLow-1); flip bit B
        const int B = kLow + __builtin_ctz((unsigned)(blk + 1));
        const uint64_t x = xhi | (low0 ^ (1u << (kLow - 1)));
        const double sb = ((x >> B) & 1u) ? -1.0 : 1.0;
        e = fma(sb, field(n, qs, x, B), e);
#pragma unroll
        for (int j = 0; j < kLow; ++j) h[j] = fma(sb, qs[j * kMaxN + B], h[j]);
        xhi ^= 1ull << B;
      }
    }
  }
  block_min(emin, xmin, out_e, out_x);
}

int exhaustive_max_n() { return kMaxN; }

// Threads and per-thread bits of the Gray walk for n (20 < n <= 40).
static void gray_shape(int n, int *P, int *L) {
  *P = std::min(n - kMinLow, kMaxTopBits);
  *L = n - *P;
}

namespace {

// What bounds the rounding of energies of the upper triangle of q.
struct Size {
  double sum = 0.0;    // sum of all |q_ij|: no exact energy is larger
  double field = 0.0;  // largest |q_jj| + sum of |q_ij| of a bit: no exact field is
};

Size coefficient_size(int n, const double *q) {
  Size s;
  std::vector<double> f(n, 0.0);
  for (int i = 0; i < n; ++i)
    for (int j = i; j < n; ++j) {
      const double a = std::fabs(q[(size_t)i * n + j]);
      s.sum += a;
      f[i] += a;
      if (j != i) f[j] += a;
    }
  for (double v : f) s.field = std::max(s.field, v);
  return s;
}

// Bound of |walk energy - exact energy| over a segment of `flips` flips, to
// first order in u = 2^-53 and a quarter more for the rest.  The segment starts
// from a literal energy (at most n (n + 1) / 2 additions) and fields of at most
// n additions; each flip adds one rounding to the energy and one to every field,
// and the flipped field's error so far to the energy.  The closed form of pass 1
// adds three fields and a few roundings.  flips = 0: a literal energy.
double walk_bound(int n, int flips, const Size &s) {
  const double fields = (flips * (n + 0.5 * flips) + 3.0 * (n + flips)) * s.field;
  return 1.25 * 0x1p-53 * ((0.5 * n * (n + 1) + flips + 8.0) * s.sum + fields);
}

}  // namespace

void exhaustive_solve(hipStream_t st, int n, const double *q_host, const double *q_dev,
                      double *tmin, double *part_e, uint64_t *part_x, size_t part_cap,
                      double *best_e, uint64_t *best_x) {
  bool finite = true;
  for (int i = 0; i < n; ++i)
    for (int j = i; j < n; ++j) finite = finite && std::isfinite(q_host[(size_t)i * n + j]);
  const Size size = coefficient_size(n, q_host);
  // beyond this, a sum of a walk may leave FP64, which no bound covers
  const bool bounded = size.sum <= 1e300;
  auto reduce = [&](int nb, std::vector<double> *minima) {
    std::vector<double> e(nb);
    std::vector<uint64_t> x(nb);
    OS_HIP_CHECK(hipMemcpyAsync(e.data(), part_e, sizeof(double) * nb, hipMemcpyDeviceToHost, st));
    OS_HIP_CHECK(hipMemcpyAsync(x.data(), part_x, sizeof(uint64_t) * nb, hipMemcpyDeviceToHost, st));
    OS_HIP_CHECK(hipStreamSynchronize(st));
    double be = DBL_MAX;
    uint64_t bx = 0;
    for (int i = 0; i < nb; ++i)
      if (e[i] < be || (e[i] == be && x[i] < bx)) {
        be = e[i];
        bx = x[i];
      }
    *best_e = be;
    *best_x = bx;
    if (minima) minima->swap(e);
  };
  if (n <= kLiteralMaxN || (!bounded && n <= 30)) {
    const int nb = (int)(((1ull << n) + kThreads - 1) / kThreads);
    OS_REQUIRE((size_t)nb <= part_cap, "partials buffer too small");
    exh_literal_kernel<<<nb, kThreads, 0, st>>>(n, q_dev, part_e, part_x);
    OS_HIP_CHECK(hipGetLastError());
    reduce(nb, nullptr);
    return;
  }
  if (!finite)
    throw Error(OS_ERR_UNSUPPORTED, "exhaustive search with non-finite coefficients supports n <= 30");
  OS_REQUIRE(n <= kMaxN, "exhaustive search supports n <= 40");
  int P, L;
  gray_shape(n, &P, &L);
  const int nb = (int)(((1ull << P) + kThreads - 1) / kThreads);
  OS_REQUIRE((size_t)nb <= part_cap, "partials buffer too small");
  exh_min_kernel<<<nb, kThreads, 0, st>>>(n, L, q_dev, tmin, part_e, part_x);
  OS_HIP_CHECK(hipGetLastError());
  std::vector<double> minima;
  reduce(nb, &minima);
  // candidates of pass 1 and, for walks of 2^(L-K) states a thread, of pass 2;
  // every state where nothing is bounded
  const double ew = *best_e;
  const double e1 = walk_bound(n, 17 << (std::min(L, kSegBits) - kMinLow), size);
  const double el = walk_bound(n, 0, size);
  const double thr1 = bounded ? ew + 2.0 * (e1 + el) : INFINITY;
  auto thr2 = [&](int split) {
    const double e2 = walk_bound(n, 1 << std::min(L - split, kSegBits), size);
    return bounded ? ew + e1 + e2 + 2.0 * el : INFINITY;
  };
  // One thread's walk is a serial chain, so its states go to 2^K threads where
  // few blocks hold candidates (most instances: one; n = 32 441 -> 53 us).
  // Instances with many fill the chip by themselves; their threads are split as
  // far as 2^20 threads and walks of 2^kLow states allow (all states tied, n = 26:
  // 5.8 ms undivided, SPLITMS split in two).
  ActiveBlocks act{0, {}};
  int found = 0;
  for (int i = 0; i < nb; ++i)
    if (!(minima[i] > thr1) && found++ < kMaxActive) act.id[act.count++] = i;
  int K = std::min(8, L - kLow);
  if (found > kMaxActive || ((size_t)found << K) > part_cap) {
    K = std::min(n - kLow, kMaxTopBits) - P;
    act.count = 0;
  }
  const int nb2 = (act.count ? found : nb) << K;
  exh_gray_kernel<<<nb2, kThreads, 0, st>>>(n, L, K, act, q_dev, thr1, thr2(K), tmin, part_e,
                                            part_x);
  OS_HIP_CHECK(hipGetLastError());
  reduce(nb2, nullptr);
  if (*best_e == DBL_MAX) throw Error(OS_ERR_INTERNAL, "exhaustive search found no candidate");
}

size_t exhaustive_thread_slots(int n) {
  if (n <= kLiteralMaxN) return 0;
  int P, L;
  gray_shape(std::min(n, kMaxN), &P, &L);
  return (size_t)1 << P;
}

size_t exhaustive_partials(int n) {
  if (n <= 30) return (size_t)(((1ull << std::min(n, 30)) + kThreads - 1) / kThreads);
  return (size_t)1 << (kMaxTopBits - 8);
}

}  // namespace os
