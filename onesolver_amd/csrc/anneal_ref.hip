// anneal_ref.hip -- reference-semantics simulated annealing on the GPU.
//
// Restates the chain of sa::anneal (include/simulated_annealing/annealing.hpp:85-126)
// with O(N) local fields instead of the O(N^2) energy recompute of :104:
//   - one wavefront per replica; its 64 lanes share the replica's fields
//     h_j = Q_jj + sum_{l!=j} Q_jl x_l (FP64, in LDS when they fit);
//   - attempt t: Philox draw -> site s = floor(w0*N/2^32), u = w1*2^-32;
//     dE = (1-2x_s) h_s; accept iff dE < 0 || exp(-dE/beta) > u
//     (annealing.hpp:106-107 with E_cur - E_new = -dE);
//   - an accepted flip updates all fields with row s of Q (coalesced,
//     Q is symmetric), E += dE;
//   - best state copied whenever E < E_best (annealing.hpp:115-121).
// ref_anneal_kernel takes these steps one by one, ref_anneal_window_kernel 64 at
// a time; launch_ref_anneal says which runs.
#include "os_kernels.h"

namespace os {

template <bool kLdsFields>
__global__ __launch_bounds__(64) void ref_anneal_kernel(int n, const double *__restrict__ q,
                                                        const double *__restrict__ beta,
                                                        uint64_t total_attempts, int spb,
                                                        uint32_t k0, uint32_t k1,
                                                        double *__restrict__ gfields,
                                                        uint32_t *__restrict__ best_bits, int W,
                                                        double *__restrict__ best_run) {
  extern __shared__ __align__(16) unsigned char smem[];
  const uint32_t replica = blockIdx.x;
  const int lane = threadIdx.x;
  double *h = kLdsFields ? reinterpret_cast<double *>(smem) : gfields + (size_t)replica * n;
  uint8_t *x = smem + (kLdsFields ? sizeof(double) * (size_t)n : 0);
  uint8_t *best = x + n;

  for (int j = lane; j < n; j += 64) {
    const uint4 o = philox4x32_10(make_uint4((uint32_t)(j >> 7), replica, 0u, TAG_REF_INIT), k0, k1);
    const uint8_t b = (uint8_t)((pick(o, (j >> 5) & 3) >> (j & 31)) & 1u);
    x[j] = b;
    best[j] = b;
    h[j] = q[(size_t)j * n + j];
  }
  __syncthreads();
  // h_j += sum_{l != j, x_l = 1} Q_lj (row l of the symmetric Q, coalesced)
  for (int l = 0; l < n; ++l) {
    if (x[l]) {
      const double *row = q + (size_t)l * n;
      for (int j = lane; j < n; j += 64)
        if (j != l) h[j] += row[j];
    }
  }
  __syncthreads();
  double part = 0.0;
  for (int j = lane; j < n; j += 64)
    if (x[j]) part += 0.5 * (h[j] + q[(size_t)j * n + j]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
  double e_cur = part;
  double e_best = part;

  for (uint64_t t = 0; t < total_attempts; ++t) {
    const double b = beta[t / (uint64_t)spb];
    const uint4 o =
        philox4x32_10(make_uint4((uint32_t)t, replica, (uint32_t)(t >> 32), TAG_REF_STEP), k0, k1);
    const int s = (int)__umulhi(o.x, (uint32_t)n);
    const double u = (double)o.y * 0x1p-32;
    const uint8_t xs = x[s];
    const double hs = h[s];
    const double de = xs ? -hs : hs;
    const bool accept = (de < 0.0) || (exp(-de / b) > u);
    if (accept) {
      const double d = xs ? -1.0 : 1.0;
      const double *row = q + (size_t)s * n;
      for (int j = lane; j < n; j += 64)
        if (j != s) h[j] = fma(row[j], d, h[j]);
      if (lane == 0) x[s] = (uint8_t)(1 - xs);
      e_cur += de;
    }
    __syncthreads();
    if (e_cur < e_best) {
      e_best = e_cur;
      for (int j = lane; j < n; j += 64) best[j] = x[j];
    }
  }
  __syncthreads();
  uint32_t *dst = best_bits + (size_t)replica * W;
  for (int w = lane; w < W; w += 64) {
    uint32_t v = 0;
    for (int bb = 0; bb < 32; ++bb) {
      const int j = w * 32 + bb;
      if (j < n && best[j]) v |= 1u << bb;
    }
    dst[w] = v;
  }
  if (lane == 0) best_run[replica] = e_best;
}

// n <= 1024: the same chain, 64 attempts at a time.  The draws of an attempt do
// not depend on the state, so lane m draws attempt t + m (site, u, threshold)
// and keeps its site's field and spin.  All 64 acceptance tests are taken at
// once; the first accepted attempt (ballot) is the next flip of the chain --
// everything before it is a rejection -- and updates the fields and spins the
// later lanes keep, with the chain's own fma; then the tests of the lanes
// behind it are taken again.  So a rejection costs a 64th of a step and an
// acceptance some forty instructions.  The n fields themselves take the
// window's accepted rows of Q at its end, in order, several requested at once.
// The couplings between the window's sites come from Q staged in LDS (kQLds,
// n <= 64) or are gathered into LDS at its start.
// The state and the best state are bit words, word w in lane w.
//
// The test exp(-dE / b) > u is decided by dE against -b ln u, made once per
// lane and window, where they differ by more than 1e-13 (b + |b ln u|), far
// above the rounding of either side; otherwise, and for b or u outside the
// ordinary, the expression itself is evaluated.  Every FP64 operation that
// reaches the state, energy or best state is the one of ref_anneal_kernel, so
// the chains are the same.
//
// A chain is serial, one wave per try: what bounds it is the instructions per
// acceptance and, for n > 64, the rows of Q read from L2 (8 n bytes per
// acceptance).  Measured on one MI355X: n = 28, 1024 tries x 1000 attempts
// 248 -> 55 us (speculating on all outcomes of six attempts before); n = 512,
// 460 tries x 1000 attempts 1636 -> 428 us (ref_anneal_kernel before: every
// acceptance waited for its row).
// Above 1024 spins 32 fields, as many diagonal entries and two rows of a lane
// no longer fit 256 registers; ref_anneal_kernel takes over there.
constexpr int kRefWindowN = 1024;
// For 64 < n the window's couplings (33 .. 40 KB of LDS) leave four tries a CU,
// 1024 on the chip, where ref_anneal_kernel has up to 32 a CU.  Up to two rounds
// of them the window kernel is never slower, however many attempts are accepted;
// beyond, the other one catches up, first where the schedule is hot, and from 768
// spins on it never does (its rows no longer hide behind one another).  Whole
// calls of 300 attempts, all accepted, ms, ref_anneal_kernel | window: n = 65
// 2048 tries 0.41 | 0.40, 4096 0.58 | 0.72; n = 128 2048 0.41 | 0.38, 4096 0.53 |
// 0.69, 16384 1.46 | 2.53; n = 256 4096 0.85 | 0.87, 16384 2.24 | 3.25; n = 640
// 2048 1.79 | 1.17, 4096 2.04 | 2.06, 16384 5.6 | 7.3; n = 768 2048 2.49 | 1.39,
// 16384 9.5 | 9.0; n = 1024 16384 18.5 | 11.7.
constexpr uint32_t kRefWindowTries = 2048;
constexpr int kRefAlwaysWindowN = 768;
static bool ref_window(int n, uint32_t tries) {
  return n <= 64 || (n <= kRefWindowN && (tries <= kRefWindowTries || n >= kRefAlwaysWindowN));
}

__device__ __forceinline__ double readlane_f64(double v, int l) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// NC: fields per lane (j = lane + 64 c), n <= 64 NC.
template <int NC, bool kQLds>
__global__ __launch_bounds__(64) void ref_anneal_window_kernel(
    int n, const double *__restrict__ q, const double *__restrict__ beta,
    uint64_t total_attempts, int spb, uint32_t k0, uint32_t k1,
    uint32_t *__restrict__ best_bits, int W, double *__restrict__ best_run) {
  extern __shared__ __align__(16) double sm[];
  double *qs = sm;           // kQLds: Q, n x n
  double *pair = sm;         // otherwise: couplings of the window's sites, 64 x 64,
  double *hl = sm + 64 * 64;  // and the fields, n
  const uint32_t replica = blockIdx.x;
  const int lane = threadIdx.x;
  if (kQLds) {
    for (int i = lane; i < n * n; i += 64) qs[i] = q[i];
    __syncthreads();
  }
  // h[j] = fma(Q[s][j], d, h[j]) for j != s, row after row of the list that
  // next(s, d) walks (false behind its end, with any valid s); kBatch rows are
  // requested together, so that a batch and not every row waits for L2.  A
  // lane's fields past n take copies of column n - 1 and are never read.
  constexpr int kBatch = NC <= 8 ? 8 : 64 / NC;
  double qd[NC], h[NC];
  int col[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) col[c] = min(lane + 64 * c, n - 1);
  auto add_rows = [&](auto next) {
    for (bool more = true; more;) {
      int sr[kBatch];
      bool on[kBatch];
      double d[kBatch], r[kBatch][NC];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        on[k] = next(sr[k], d[k]);
#pragma unroll
        for (int c = 0; c < NC; ++c)
          r[k][c] = kQLds ? qs[sr[k] * n + col[c]] : (q + (size_t)sr[k] * n)[(uint32_t)col[c]];
      }
      more = on[kBatch - 1];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        if (!on[k]) break;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const double v = fma(r[k][c], d[k], h[c]);
          h[c] = lane + 64 * c != sr[k] ? v : h[c];
        }
      }
    }
  };
  // start state: word `lane` of the state
  uint32_t word = 0u;
  {
    const uint4 o =
        philox4x32_10(make_uint4((uint32_t)(lane >> 2), replica, 0u, TAG_REF_INIT), k0, k1);
    const int valid = n - 32 * lane;
    const uint32_t v = pick(o, (uint32_t)lane & 3u);
    word = valid >= 32 ? v : valid <= 0 ? 0u : (v & ((1u << valid) - 1u));
  }
  uint32_t best = word;
  // fields: diagonal, then + row l for every set l in ascending order
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    qd[c] = q[(size_t)col[c] * n + col[c]];
    h[c] = qd[c];
  }
  {
    int w = -1;
    uint32_t bits = 0u;
    add_rows([&](int &l, double &d) {  // fma(row, 1, h) is h + row
      l = 0;
      d = 1.0;
      while (bits == 0u) {
        if (++w >= W) return false;
        bits = (uint32_t)__builtin_amdgcn_readlane((int)word, w);
      }
      l = 32 * w + __builtin_ctz(bits);
      bits &= bits - 1u;
      return true;
    });
  }
  double part = 0.0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int j = lane + 64 * c;
    const uint32_t xw =
        (uint32_t)__builtin_amdgcn_ds_bpermute((j >> 5) << 2, (int)word);
    if (j < n && ((xw >> (j & 31)) & 1u)) part += 0.5 * (h[c] + qd[c]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
  double e_cur = part;
  double e_best = part;

  uint32_t bi = 0, bc = 0;  // attempt t is number bc of beta[bi]
  for (uint64_t t = 0; t < total_attempts; t += 64) {
    const int kk = (int)min((uint64_t)64, total_attempts - t);
    const uint64_t tm = t + (uint64_t)lane;
    const uint4 o =
        philox4x32_10(make_uint4((uint32_t)tm, replica, (uint32_t)(tm >> 32), TAG_REF_STEP), k0,
                      k1);
    const int s = (int)__umulhi(o.x, (uint32_t)n);
    const double u = (double)o.y * 0x1p-32;
    const double b = lane < kk ? beta[bi + (bc + (uint32_t)lane) / (uint32_t)spb] : 1.0;
    bi += (bc + 64u) / (uint32_t)spb;
    bc = (bc + 64u) % (uint32_t)spb;
    const double thr = -b * log(u);
    const double tol = 1e-13 * (b + fabs(thr));
    const bool plain = b > 0.0 && b < 1e300 && u > 0.0;
    // dE < lo: accepted for sure (lo >= 0, so dE < 0 is among them); dE > hi:
    // rejected for sure; in between, NaN included: the expression decides
    const double lo = plain ? fmax(thr - tol, 0.0) : 0.0, hi = plain ? thr + tol : INFINITY;
    // this lane's field and spin
    double hm;
    if (NC == 1) {
      const uint64_t hb = (uint64_t)__double_as_longlong(h[0]);
      const uint32_t h0 = (uint32_t)__builtin_amdgcn_ds_bpermute(s << 2, (int)(uint32_t)hb);
      const uint32_t h1 =
          (uint32_t)__builtin_amdgcn_ds_bpermute(s << 2, (int)(uint32_t)(hb >> 32));
      hm = __longlong_as_double((long long)(((uint64_t)h1 << 32) | h0));
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
        if (lane + 64 * c < n) hl[lane + 64 * c] = h[c];
      __syncthreads();
      hm = hl[s];
    }
    uint32_t xb =
        ((uint32_t)__builtin_amdgcn_ds_bpermute((s >> 5) << 2, (int)word) >> (s & 31)) & 1u;
    if (!kQLds) {
      // pair[m][lane] = Q[s_m][s_lane] (read by the lanes behind m)
#pragma unroll 1
      for (int m0 = 0; m0 < 64; m0 += 16) {
        double v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          v[k] = (q + (size_t)__builtin_amdgcn_readlane(s, m0 + k) * n)[(uint32_t)s];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) pair[(m0 + k) * 64 + lane] = v[k];
      }
      __syncthreads();
    }
    uint64_t live = kk == 64 ? ~0ull : (1ull << kk) - 1ull;  // attempts not yet decided
    uint64_t taken = 0ull, down = 0ull;                      // accepted; those flipping 1 -> 0
    double de = xb ? -hm : hm;
    for (;;) {
      const uint64_t cand = __ballot(!(de > hi)) & live;
      if (cand == 0ull) break;
      const int m = __builtin_ctzll(cand);
      live &= (~1ull) << m;
      if (!((__ballot(de < lo) >> m) & 1ull))
        if (!((__ballot(exp(-de / b) > u) >> m) & 1ull)) continue;
      const int sm_ = __builtin_amdgcn_readlane(s, m);
      const uint32_t xm = (uint32_t)__builtin_amdgcn_readlane((int)xb, m);
      const double dem = readlane_f64(de, m);
      const double pv = kQLds ? qs[sm_ * n + s] : pair[m * 64 + lane];
      const double hn = fma(pv, xm ? -1.0 : 1.0, hm);
      const bool same = s == sm_;
      hm = same ? hm : hn;
      xb ^= same ? 1u : 0u;
      de = xb ? -hm : hm;
      word ^= lane == (sm_ >> 5) ? 1u << (sm_ & 31) : 0u;
      e_cur += dem;
      taken |= 1ull << m;
      down |= (uint64_t)xm << m;
      const bool better = e_cur < e_best;
      e_best = better ? e_cur : e_best;
      best = better ? word : best;
    }
    // the window's accepted rows into the fields, in order
    add_rows([&](int &l, double &d) {
      const bool on = taken != 0ull;
      const int m = on ? __builtin_ctzll(taken) : 0;
      taken &= taken - 1ull;
      l = __builtin_amdgcn_readlane(s, m);
      d = (down >> m) & 1ull ? -1.0 : 1.0;
      return on;
    });
  }
  if (lane < W) best_bits[(size_t)replica * W + lane] = best;
  if (lane == 0) best_run[replica] = e_best;
}

int ref_lds_limit() { return 4096; }

size_t ref_lds_bytes(int n) {
  return (n <= ref_lds_limit() ? sizeof(double) * (size_t)n : 0) + 2 * (size_t)n;
}

void launch_ref_anneal(hipStream_t st, int n, const double *q, const double *beta, int num_iter,
                       int spb, uint32_t num_tries, uint64_t seed, double *gfields,
                       uint32_t *best_bits, double *best_run) {
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const uint64_t total = (uint64_t)num_iter * (uint64_t)spb;
  const int W = (n + 31) / 32;
  const size_t lds = (ref_lds_bytes(n) + 15) & ~(size_t)15;
  if (ref_window(n, num_tries)) {
    // fields per lane: the next power of two of n / 64
    const size_t wlds = sizeof(double) * (n <= 64 ? (size_t)n * n : (size_t)64 * 64 + n);
#define OS_WINDOW(NC, QL)                                                           \
  ref_anneal_window_kernel<NC, QL><<<num_tries, 64, wlds, st>>>(n, q, beta, total,   \
                                                                spb, k0, k1, best_bits, W, best_run)
    if (n <= 64) OS_WINDOW(1, true);
    else if (n <= 128) OS_WINDOW(2, false);
    else if (n <= 256) OS_WINDOW(4, false);
    else if (n <= 512) OS_WINDOW(8, false);
    else OS_WINDOW(16, false);
#undef OS_WINDOW
  } else if (n <= ref_lds_limit()) {
    ref_anneal_kernel<true><<<num_tries, 64, lds, st>>>(n, q, beta, total, spb, k0, k1, nullptr,
                                                         best_bits, W, best_run);
  } else {
    ref_anneal_kernel<false><<<num_tries, 64, lds, st>>>(n, q, beta, total, spb, k0, k1, gfields,
                                                          best_bits, W, best_run);
  }
  OS_HIP_CHECK(hipGetLastError());
}

}  // namespace os
