// anneal_dense.hip -- sweep-mode simulated annealing of dense QUBOs with
// delayed field updates on MFMA (gfx950).
//
// Replicas run Metropolis sweeps in a fixed site order j = 0..N-1.  Local
// fields h_rj = Q_jj + sum_{l!=j} Q_jl x_rl live in MFMA accumulators (fp32).
// Spins are decided in blocks of k = 16; after block b the flip deltas D_b
// (replicas x 16, values -1/0/+1, exact in bf16) update every field:
// F += D * Qhi + D * Qlo on v_mfma_f32_32x32x16_bf16 (Q = Qhi + Qlo, both
// bf16, rows 16b .. 16b+15 of Q).
//
// Work-group: 64 replicas (two 32-replica tiles), 4 waves (one per SIMD, so
// each wave has up to the full register file and the fields sit in accumulation
// registers).  Blocks are dealt to the waves round-robin: block b belongs to
// wave b % 4, and wave w holds the columns of its blocks as TPW tiles of 32
// columns (tile t = blocks w + 8t and w + 8t + 4).  A sweep visits nb blocks:
// those with spins, rounded up to a whole turn of the waves (not the padded
// size of the tiles).  Step g of the global block sequence (block b of sweep
// sw) has four roles that pass from wave to wave:
//   * the owner of block b applies D_{g-1} to the one tile holding b (4
//     MFMAs), transposes its half of it through LDS, decides the 16 spins in
//     order (lane = replica; flips inside the block correct the later spins
//     with the fp32 16x16 diagonal sub-block of Q) and publishes D_g as bf16
//     rows in an LDS ring -- this is the chain; only then does it apply
//     D_{g-1} to its tiles and, between those MFMAs, update spins, energies
//     and best states (in block order, by a counter of their own);
//   * the wave that owned the block before applies D_{g-1} to all its tiles
//     with the Philox rounds of its next block's thresholds between the MFMAs;
//   * the one before that does the same with their logarithms;
//   * the next owner only applies D_{g-1} and requests its next step's
//     operands, sub-block rows included.
// So the chain of decisions passes from SIMD to SIMD, and each SIMD's MFMA
// and threshold work runs while the others decide.  Thresholds and sub-block
// rows live in the registers of the wave that will use them.  Q operands
// stream from L2 into registers, each requested again as soon as its products
// are issued; waves synchronise only through LDS counters with bounded waits
// (an expired wait is reported in `status`).
//
// What bounds it: one wave issues an instruction every 4-5 cycles and a taken
// branch costs about 35, so the chain is its instruction count (some 185 for
// the 16 decisions) plus three LDS round trips: about 1800 cycles a step.  Up
// to n = 128 that is the step; above, each wave's four roles together (MFMAs
// 33 cycles each, thresholds about 3000) set it: 0.98 us a step at n = 512,
// 1.27 us at n = 1024 (a third of it MFMAs).  Measured on one MI355X
// against the version with thresholds, sub-block and flip masks in LDS and a
// lookup table for the bf16 rows: n = 60, 64 replicas, 64 sweeps 786 -> 190
// us; 16 x n = 300, 256 sweeps 9.0 -> 4.4 ms; 4 x n = 512 replica exchange,
// 256 sweeps 11.9 -> 7.2 ms; n = 1024, 16384 replicas, 512 sweeps 52.7 ->
// 41.5 ms (40.8 .. 45 in longer runs, depending on the card).
//
// Acceptance: flip iff dE < neg_ln_u(w) * tscale[t] with w the Philox word of
// counter (j>>2, replica, sweep, tag), i.e. with probability
// min(1, exp(-dE / tscale^-1)).  With `tsr` (replica exchange) the scale is
// tsr[row] of the replica instead, for the whole launch.
#include <type_traits>

#include "os_kernels.h"

namespace os {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kWaves = 4;
constexpr int kRT = 64;       // replicas per work-group
constexpr int kRing = 8;      // D blocks kept in LDS
constexpr int kFT = kRT + 4;  // row stride (floats) of the transposed field tile
constexpr int kSpinLimit = 1 << 24;

// The owner of step g writes ring slot g % kRing after it has seen D_{g-1}
// published.  The owners of steps g-4 .. g-1 -- all four waves -- published
// only after reading the rows of those steps, so every wave has read D_{g-5}
// and older; slot g % kRing last held D_{g-kRing}.
static_assert(kRing >= kWaves + 1, "a ring slot is rewritten only after every wave read it");

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Synchronisation between the waves only concerns LDS data written with
// ordinary ds_write instructions.  LDS operations of one wave complete in
// order, so publishing needs only a compiler barrier and a counter written
// behind the data -- not the vmcnt(0) wait that a workgroup release fence
// implies, which would stall on this wave's outstanding operand loads.  The
// counters are accessed by ds instructions in asm, so no memory-model fence
// or atomic lowering adds such a wait either; each asm read waits for its own
// result (lgkmcnt(0)) inside the statement.
__device__ __forceinline__ void lds_writes_done() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt/expcnt unconstrained
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

__device__ __forceinline__ void wave_sync() {
  lds_writes_done();
  __builtin_amdgcn_wave_barrier();
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}

// Publishes v in *p behind all of this wave's earlier LDS writes, which the
// LDS completes in order.
__device__ __forceinline__ void lds_store(int *p, int v) {
  asm volatile("ds_write_b32 %0, %1" : : "v"(lds_addr(p)), "v"(v) : "memory");
}

// Waits until *p >= target and returns the A operands at `row` (replica lc of
// each 32-replica half, 1 KB apart); false once kSpinLimit polls have passed.
// The rows are requested behind the counter in every poll: a wave's LDS reads
// complete in order, so rows read after a counter value that counts them are
// the published ones, and the wait ends one LDS round trip earlier than with
// a separate read.  The loop is scalar and inside the statement: written in
// C++, every wave of every step pays some forty instructions of exec-mask
// bookkeeping for it.  A wave that gives up publishes nothing more, so the
// others run into their own limit.
#define OS_POLL(reads)                                                              \
  "s_mov_b32 %[left], %[limit]\n1:\n\tds_read_b32 %[v], %[p]\n\t" reads              \
  "s_waitcnt lgkmcnt(0)\n\tv_readfirstlane_b32 %[c], %[v]\n\t"                       \
  "s_sub_u32 %[left], %[left], 1\n\ts_cmp_ge_i32 %[c], %[t]\n\ts_cbranch_scc1 2f\n\t" \
  "s_cmp_lg_u32 %[left], 0\n\ts_cbranch_scc1 1b\n2:"
__device__ __forceinline__ int wait_rows(const int *p, int target, const uint4 *row,
                                          bf16x8 (&A)[2]) {
  int v, c, left;
  asm volatile(OS_POLL("ds_read_b128 %[a], %[r]\n\tds_read_b128 %[b], %[r] offset:1024\n\t")
               : [v] "=&v"(v), [a] "=&v"(A[0]), [b] "=&v"(A[1]), [c] "=&s"(c),
                 [left] "=&s"(left)
               : [p] "v"(lds_addr(p)), [r] "v"(lds_addr(row)), [t] "s"(__builtin_amdgcn_readfirstlane(target)),
                 [limit] "i"(kSpinLimit)
               : "memory", "scc");
  return c >= target;
}

// The same for the state word and the energy of a replica.
__device__ __forceinline__ int wait_state(const int *p, int target, const uint32_t *word,
                                           const double *energy, uint32_t &x, double &e) {
  int v, c, left;
  asm volatile(OS_POLL("ds_read_b32 %[x], %[w]\n\tds_read_b64 %[e], %[f]\n\t")
               : [v] "=&v"(v), [x] "=&v"(x), [e] "=&v"(e), [c] "=&s"(c), [left] "=&s"(left)
               : [p] "v"(lds_addr(p)), [w] "v"(lds_addr(word)), [f] "v"(lds_addr(energy)),
                 [t] "s"(__builtin_amdgcn_readfirstlane(target)), [limit] "i"(kSpinLimit)
               : "memory", "scc");
  return c >= target;
}
#undef OS_POLL

// The 16 decisions of a block, lane = replica.  c: the fields on entry, each
// field as its spin was decided on return; d1: the delta +1 / -1 of a flip;
// th: thresholds; q[j]: row j of the fp32 16x16 sub-block, column m in lane m
// of every 16 lanes; d (out): the delta taken, or 0.  Spin j flips iff
// c[j] d1[j] < th[j], after which c[m] += q[j][m] d[j] for m > j: v_fmac_f32
// with its Q operand broadcast from lane m by DPP, so a row costs one register
// and no read.  Step j leaves the corrections of c[j+2..] to step j+1, which
// runs two of them in the two wait states a select needs after its compare
// and the rest behind the select.  Each step is one asm statement: its first
// two instructions are the wait states a DPP read needs should a q register
// have been copied just before it.
#define OS_FM(q, d, m) \
  "v_fmac_f32_dpp %[c" #m "], %[" #q "], %[" #d "] row_newbcast:" #m " row_mask:0xf bank_mask:0xf\n\t"
#define OS_F15(q, d) OS_FM(q, d, 15)
#define OS_F14(q, d) OS_FM(q, d, 14) OS_F15(q, d)
#define OS_F13(q, d) OS_FM(q, d, 13) OS_F14(q, d)
#define OS_F12(q, d) OS_FM(q, d, 12) OS_F13(q, d)
#define OS_F11(q, d) OS_FM(q, d, 11) OS_F12(q, d)
#define OS_F10(q, d) OS_FM(q, d, 10) OS_F11(q, d)
#define OS_F9(q, d) OS_FM(q, d, 9) OS_F10(q, d)
#define OS_F8(q, d) OS_FM(q, d, 8) OS_F9(q, d)
#define OS_F7(q, d) OS_FM(q, d, 7) OS_F8(q, d)
#define OS_F6(q, d) OS_FM(q, d, 6) OS_F7(q, d)
#define OS_F5(q, d) OS_FM(q, d, 5) OS_F6(q, d)
#define OS_F4(q, d) OS_FM(q, d, 4) OS_F5(q, d)
#define OS_O15 [c15] "+v"(c[15])
#define OS_O14 [c14] "+v"(c[14]), OS_O15
#define OS_O13 [c13] "+v"(c[13]), OS_O14
#define OS_O12 [c12] "+v"(c[12]), OS_O13
#define OS_O11 [c11] "+v"(c[11]), OS_O12
#define OS_O10 [c10] "+v"(c[10]), OS_O11
#define OS_O9 [c9] "+v"(c[9]), OS_O10
#define OS_O8 [c8] "+v"(c[8]), OS_O9
#define OS_O7 [c7] "+v"(c[7]), OS_O8
#define OS_O6 [c6] "+v"(c[6]), OS_O7
#define OS_O5 [c5] "+v"(c[5]), OS_O6
#define OS_O4 [c4] "+v"(c[4]), OS_O5
#define OS_O3 [c3] "+v"(c[3]), OS_O4
#define OS_O2 [c2] "+v"(c[2]), OS_O3
// the test of step J, `fill` between the compare and the select
#define OS_TEST(fill)                                  \
  "v_mul_f32_e32 %[t], %[cj], %[s]\n\t"                \
  "v_cmp_lt_f32_e32 vcc, %[t], %[th]\n\t" fill         \
  "v_cndmask_b32_e32 %[d], 0, %[s], vcc\n\t"
#define OS_IN(J) [cj] "v"(c[J]), [s] "v"(d1[J]), [th] "v"(th[J])
// step J (1 .. 14): A, B: the two corrections run as fill, rest: the others of
// row J-1, N = J + 1: the first correction of row J
#define OS_STEP(J, N, fill, rest, outs)                                                     \
  asm volatile(OS_TEST(fill) rest OS_FM(q, d, N)                                            \
               : [d] "=&v"(d[J]), [t] "=&v"(t), outs                                        \
               : OS_IN(J), [p] "v"(q[J - 1]), [e] "v"(d[J - 1]), [q] "v"(q[J])              \
               : "vcc")
__device__ __forceinline__ void decide16(float (&c)[16], const float (&d1)[16],
                                         const float (&th)[16], const float (&q)[16],
                                         float (&d)[16]) {
  float t;
  asm volatile(OS_TEST("s_nop 1\n\t") OS_FM(q, d, 1)
               : [d] "=&v"(d[0]), [t] "=&v"(t), [c1] "+v"(c[1])
               : OS_IN(0), [q] "v"(q[0])
               : "vcc");
  OS_STEP(1, 2, OS_FM(p, e, 2) OS_FM(p, e, 3), OS_F4(p, e), OS_O2);
  OS_STEP(2, 3, OS_FM(p, e, 3) OS_FM(p, e, 4), OS_F5(p, e), OS_O3);
  OS_STEP(3, 4, OS_FM(p, e, 4) OS_FM(p, e, 5), OS_F6(p, e), OS_O4);
  OS_STEP(4, 5, OS_FM(p, e, 5) OS_FM(p, e, 6), OS_F7(p, e), OS_O5);
  OS_STEP(5, 6, OS_FM(p, e, 6) OS_FM(p, e, 7), OS_F8(p, e), OS_O6);
  OS_STEP(6, 7, OS_FM(p, e, 7) OS_FM(p, e, 8), OS_F9(p, e), OS_O7);
  OS_STEP(7, 8, OS_FM(p, e, 8) OS_FM(p, e, 9), OS_F10(p, e), OS_O8);
  OS_STEP(8, 9, OS_FM(p, e, 9) OS_FM(p, e, 10), OS_F11(p, e), OS_O9);
  OS_STEP(9, 10, OS_FM(p, e, 10) OS_FM(p, e, 11), OS_F12(p, e), OS_O10);
  OS_STEP(10, 11, OS_FM(p, e, 11) OS_FM(p, e, 12), OS_F13(p, e), OS_O11);
  OS_STEP(11, 12, OS_FM(p, e, 12) OS_FM(p, e, 13), OS_F14(p, e), OS_O12);
  OS_STEP(12, 13, OS_FM(p, e, 13) OS_FM(p, e, 14), OS_F15(p, e), OS_O13);
  OS_STEP(13, 14, OS_FM(p, e, 14) OS_FM(p, e, 15), "", OS_O14);
  OS_STEP(14, 15, OS_FM(p, e, 15) "s_nop 0\n\t", "", OS_O15);
  asm volatile(OS_TEST("s_nop 1\n\t") : [d] "=&v"(d[15]), [t] "=&v"(t) : OS_IN(15) : "vcc");
}
#undef OS_STEP
#undef OS_IN
#undef OS_TEST

// f(t) with t as a constant of [LO, HI), by a tree of uniform branches.
template <int LO, int HI, class F>
__device__ __forceinline__ void pick_tile(int t, F &&f) {
  if constexpr (HI - LO == 1) {
    f(std::integral_constant<int, LO>{});
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (t < MID)
      pick_tile<LO, MID>(t, f);
    else
      pick_tile<MID, HI>(t, f);
  }
}

// Column of lane lc in tile t of wave w: the tile holds blocks w + 8t (lanes
// 0..15) and w + 8t + 4 (lanes 16..31).
__device__ __forceinline__ int tile_col(int w, int t, int lc) {
  return 16 * (w + 8 * t + 4 * (lc >> 4)) + (lc & 15);
}

}  // namespace

template <int TPW>
__global__ __launch_bounds__(256, TPW <= 3 ? 2 : 1) void dense_sweep_kernel(
    int n, int nb, const uint4 *__restrict__ qpack, const float *__restrict__ qdb,
    const float *__restrict__ tscale, const float *__restrict__ tsr, int sweep0, int nsweeps,
    uint32_t k0, uint32_t k1,
    uint32_t inst_base, int gpi, float *__restrict__ fields, uint32_t *__restrict__ xbits,
    uint32_t *__restrict__ bestbits, double *__restrict__ energy, double *__restrict__ ebest,
    int *__restrict__ status) {
  static_assert(TPW >= 1 && TPW <= 8, "tiles per wave");
  constexpr int NP = kWaves * 32 * TPW;
  constexpr int NBP = NP / 16;  // blocks of the padded size (strides)
  constexpr int NPW = NP / 32;
  // The owner's tile is brought up to date in a copy, and every tile in the
  // branch-free products behind the decisions, wherever 32 accumulators are
  // left for the copy: products into a tile chosen by branches cost two taken
  // branches each.
  constexpr bool kCopyTile = TPW <= 6;
  constexpr int kVm = 0x0F70 | (2 * TPW & 15) | (2 * TPW >> 4 << 14);  // s_waitcnt vmcnt(2 TPW)
  __shared__ __align__(16) uint4 dring[kRing][kRT][2];  // D rows: 16 bf16 of each replica
  __shared__ __align__(16) float fblk[16][kFT];         // the owner's block, column-major
  __shared__ uint32_t xs[kRT][NPW + 1];
  __shared__ double es[kRT];
  __shared__ double ebs[kRT];
  __shared__ int d_count;  // D blocks published
  __shared__ int e_count;  // blocks whose spins and energies are in xs / es
  __shared__ int abort_flag;

  const int tid = threadIdx.x;
  const int w = tid >> 6;
  const int lane = tid & 63;
  const int lc = lane & 31;
  const int kh = lane >> 5;
  // gpi work-groups per instance: this one anneals replicas [rloc, rloc+64)
  // of instance inst, stored at rows [rbase, rbase+64) of the state arrays
  const int inst = blockIdx.x / gpi;
  const uint32_t rbase = blockIdx.x * kRT;
  const uint32_t rloc = (uint32_t)(blockIdx.x % gpi) * kRT;
  const uint32_t tag = ((inst_base + (uint32_t)inst) << 8) | TAG_SWEEP_THR;
  qpack += (size_t)inst * NBP * NP * 4;
  qdb += (size_t)inst * NBP * 256;
  const int G = nsweeps * nb;

  for (int i = tid; i < kRT * NPW; i += 256)
    xs[i / NPW][i % NPW] = xbits[(size_t)(rbase + i / NPW) * NPW + i % NPW];
  if (tid < kRT) {
    es[tid] = energy[rbase + tid];
    ebs[tid] = ebest[rbase + tid];
  }
  if (tid < 2 * kRT) dring[kRing - 1][tid >> 1][tid & 1] = make_uint4(0u, 0u, 0u, 0u);  // D_{-1}
  if (tid == 0) {
    d_count = 0;
    e_count = 0;
    abort_flag = 0;
  }
  // accumulator element i of lane (lc, kh): replica 32m + 8(i/4) + 4kh + i%4,
  // column tile_col(w, tt, lc)
  f32x16 C[2][TPW];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        C[m][tt][i] = fields[(size_t)(rbase + 32 * m + 8 * (i >> 2) + 4 * kh + (i & 3)) * NP +
                             tile_col(w, tt, lc)];
  // this wave's next owner step: the thresholds of replica `lane` and the
  // fp32 16x16 diagonal sub-block of Q, row j in lanes 0..15 of every 16
  const float ts_own = tsr ? tsr[rbase + lane] : 0.0f;
  // (between the two steps that make them, th holds the Philox words)
  float th[16], qr[16];
  // spins beyond n never flip
  auto cut_thresholds = [&](int bn) {
    if (16 * bn + 16 > n) {
#pragma unroll
      for (int u = 0; u < 16; ++u)
        if (16 * bn + u >= n) th[u] = -INFINITY;
    }
  };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4 o = philox4x32_10(make_uint4((uint32_t)(4 * w + i), rloc + (uint32_t)lane,
                                             (uint32_t)sweep0, tag), k0, k1);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      th[4 * i + u] = __uint_as_float(pick(o, u));
      if (w < 2) th[4 * i + u] = neg_ln_u(pick(o, u)) * (tsr ? ts_own : tscale[0]);
    }
  }
  if (w < 2) cut_thresholds(w);  // waves 2 and 3 make theirs in steps 0 and 1
  auto load_rows = [&](int x) {
#pragma unroll
    for (int j = 0; j < 16; ++j) qr[j] = (qdb + x * 256 + j * 16)[(uint32_t)(lane & 15)];
  };
  load_rows(w);
  __syncthreads();

  // B operands (rows of the next D block to apply, all tiles); a uniform base
  // and one 32-bit lane offset.  An operand is requested for the next step as
  // soon as this step's products have used it, so the requests are spread over
  // the products and have the rest of the step to arrive.
  const uint32_t qoff = (uint32_t)(tile_col(w, 0, lc) * 4 + kh);
  uint4 Bn[TPW][2];
  auto load_op = [&](int x, int tt, int p) {
    Bn[tt][p] = (qpack + ((size_t)x * NP + 128 * tt) * 4 + 2 * p)[qoff];
  };
  // step 0 applies nothing: D_{-1} and its operands are zero
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int tt = 0; tt < TPW; ++tt) Bn[tt][p] = make_uint4(0u, 0u, 0u, 0u);
  // operands of the next owner step's tile, fetched a step early
  uint4 Bo[2] = {make_uint4(0u, 0u, 0u, 0u), make_uint4(0u, 0u, 0u, 0u)};

  // `ok` is read back as a scalar at the end of a step, the only way out of the
  // loop: a break inside a role would leave the step counters in vector
  // registers.  A wave whose wait expired finishes its step on stale rows; the
  // launch is reported as aborted.
  int ok = 1;
  int g = 0, b = 0, sw = 0;  // step g is block b of sweep sw
  while (g < G && ok) {
    // no wait: the newest 2 TPW requests are the next operands.  It tells the
    // compiler that most of what the prologue requested is here, so that its
    // waits in the loop are for the loop's own requests.
    __builtin_amdgcn_s_waitcnt(kVm);
    const int b1 = b + 1 < nb ? b + 1 : 0;
    const int role = (w - b) & 3;  // 0: owner of this step, 1: of the next one, ...
    const uint4 *row = &dring[(g + kRing - 1) % kRing][lc][kh];  // D_{g-1}
    bf16x8 A[2];
    if (role == 0) {
      const int k = b >> 2;
      const int t = k >> 1;     // this wave's tile holding block b
      const int half = k & 1;   // its lanes 16*half .. +15
      const int sh = (b & 1) * 16;
      // this block's spins (its half of the state word is written by this
      // wave only) as the deltas +1 / -1 of a flip
      const uint32_t x0 = xs[lane][b >> 1] >> sh;
      float d1[16];
#pragma unroll
      for (int jj = 0; jj < 16; ++jj)
        d1[jj] = __uint_as_float(0x3F800000u | ((x0 << (31 - jj)) & 0x80000000u));
      ok = wait_rows(&d_count, g, row, A);
      // (a) tile t with D_{g-1}, its half with block b transposed
      auto transpose = [&](const f32x16 &t0, const f32x16 &t1) {
        if ((lc >> 4) != half) return;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float *f = &fblk[lc & 15][8 * q + 4 * kh];
          *reinterpret_cast<float4 *>(f) =
              make_float4(t0[4 * q], t0[4 * q + 1], t0[4 * q + 2], t0[4 * q + 3]);
          *reinterpret_cast<float4 *>(f + 32) =
              make_float4(t1[4 * q], t1[4 * q + 1], t1[4 * q + 2], t1[4 * q + 3]);
        }
      };
      if constexpr (kCopyTile) {
        pick_tile<0, TPW>(t, [&](auto tc) {
          constexpr int tt = decltype(tc)::value;
          f32x16 T[2];
#pragma unroll
          for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int m = 0; m < 2; ++m)
              T[m] = mfma32(A[m], as_bf16x8(Bo[p]), p == 0 ? C[m][tt] : T[m]);
          transpose(T[0], T[1]);
        });
      } else {
#pragma unroll
        for (int tt = 0; tt < TPW; ++tt) {
          if (tt != t) continue;
#pragma unroll
          for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int m = 0; m < 2; ++m)
              C[m][tt] = mfma32(A[m], as_bf16x8(Bo[p]), C[m][tt]);
          transpose(C[0][tt], C[1][tt]);
        }
      }
      wave_sync();
      // ---- sequential decisions of block b, lane = replica ----
      float c[16], d[16];
#pragma unroll
      for (int jj = 0; jj < 16; ++jj) c[jj] = fblk[jj][lane];
      decide16(c, d1, th, qr, d);
      // D_g: the deltas as bf16 (their upper halves), published at once
      uint32_t pk[8];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        pk[i] = __builtin_amdgcn_perm(__float_as_uint(d[2 * i + 1]), __float_as_uint(d[2 * i]),
                                      0x07060302u);
      dring[g % kRing][lane][0] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      dring[g % kRing][lane][1] = make_uint4(pk[4], pk[5], pk[6], pk[7]);
      lds_store(&d_count, g + 1);
      // (b) D_{g-1} into the other tiles and, between their MFMAs, off the
      // chain: spins, energies and best states, in block order.  Bit 7 of a
      // delta's bf16 is set iff it is +1 or -1: the flips of the even spins
      // gather in the low half of fl, of the odd ones in the high half.
      // d * h is exact, so desum gains exactly dE on a flip.
      uint32_t fl = 0u;
      float desum = 0.0f;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            if (kCopyTile || tt != t) C[m][tt] = mfma32(A[m], as_bf16x8(Bn[tt][p]), C[m][tt]);
            if (m == 1) load_op(b, tt, p);
            const int slot = (p * TPW + tt) * 2 + m;  // of 4 TPW
#pragma unroll
            for (int u = 0; u < 16; ++u) {
              if ((u * 4 * TPW) / 16 != slot) continue;
              desum = fmaf(d[u], c[u], desum);
              if (u < 8) fl |= (pk[u] & 0x00800080u) << u;
              if (u == 8) fl = (fl >> 7) & 0x00FF00FFu;
              if (u == 9) fl = (fl | (fl << 4)) & 0x0F0F0F0Fu;
              if (u == 10) fl = (fl | (fl << 2)) & 0x33333333u;
              if (u == 11) fl = (fl | (fl << 1)) & 0x55555555u;
              if (u == 12) fl = (fl | (fl >> 15)) & 0xFFFFu;
            }
            __builtin_amdgcn_sched_barrier(0);
          }
      uint32_t word;
      double e_now;
      ok &= wait_state(&e_count, g, &xs[lane][b >> 1], &es[lane], word, e_now);
      xs[lane][b >> 1] = word ^ (fl << sh);
      e_now += (double)desum;
      es[lane] = e_now;
      if (b == nb - 1 && e_now < ebs[lane]) {
        ebs[lane] = e_now;
        uint32_t *dst = bestbits + (size_t)(rbase + lane) * NPW;
        for (int q = 0; q < NPW; ++q) dst[q] = xs[lane][q];
      }
      lds_store(&e_count, g + 1);
    } else {
      ok = wait_rows(&d_count, g, row, A);
      // D_{g-1} into every tile.  The thresholds of this wave's next block
      // (spins 16*bn .. of replica `lane`) are made under the MFMAs: the four
      // Philox calls in the step after it owned a block, the sixteen
      // logarithms in the step after that; the last step before it owns one
      // again is on the chain and does nothing else.
      if (role == 3) {
        const int bn = b + 3 < nb ? b + 3 : b + 3 - nb;
        const int s2 = b + 3 < nb ? sw : sw + 1;
        uint4 ph[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          ph[i] = make_uint4((uint32_t)(4 * bn + i), rloc + (uint32_t)lane,
                             (uint32_t)(sweep0 + s2), tag);
        uint32_t pk0 = k0, pk1 = k1;
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
              C[m][tt] = mfma32(A[m], as_bf16x8(Bn[tt][p]), C[m][tt]);
              if (m == 1) load_op(b, tt, p);
              const int slot = (p * TPW + tt) * 2 + m;
#pragma unroll
              for (int u = 0; u < 20; ++u) {
                if ((u * 4 * TPW) / 20 != slot) continue;
                if (u && u % 2 == 0) {
                  pk0 += kPhiloxW0;
                  pk1 += kPhiloxW1;
                }
                philox_round(ph[2 * (u % 2)], pk0, pk1);
                philox_round(ph[2 * (u % 2) + 1], pk0, pk1);
                __builtin_amdgcn_sched_barrier(0);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
        for (int u = 0; u < 16; ++u) th[u] = __uint_as_float(pick(ph[u / 4], u % 4));
      } else if (role == 2) {
        const int bn = b + 2 < nb ? b + 2 : b + 2 - nb;
        const int s2 = b + 2 < nb ? sw : sw + 1;
        const float ts2 = tsr ? ts_own : tscale[min(s2, nsweeps - 1)];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
            for (int m = 0; m < 2; ++m) {
              C[m][tt] = mfma32(A[m], as_bf16x8(Bn[tt][p]), C[m][tt]);
              if (m == 1) load_op(b, tt, p);
              const int slot = (p * TPW + tt) * 2 + m;
#pragma unroll
              for (int u = 0; u < 16; ++u) {
                if ((u * 4 * TPW) / 16 != slot) continue;
                th[u] = neg_ln_u(__float_as_uint(th[u])) * ts2;
                if (u % 2) __builtin_amdgcn_sched_barrier(0);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
        cut_thresholds(bn);
      } else {
        // next step is this wave's: its tile of block b1 needs D_g (rows of b)
        const int t1 = (b1 >> 2) >> 1;
#pragma unroll
        for (int p = 0; p < 2; ++p)
          Bo[p] = (qpack + ((size_t)b * NP + 128 * t1) * 4 + 2 * p)[qoff];
        load_rows(b1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int tt = 0; tt < TPW; ++tt) {
#pragma unroll
            for (int m = 0; m < 2; ++m)
              C[m][tt] = mfma32(A[m], as_bf16x8(Bn[tt][p]), C[m][tt]);
            load_op(b, tt, p);
            __builtin_amdgcn_sched_barrier(0);
          }
        // Bo and qr, older than the next operands, have arrived by now.  The
        // role branches are divergent to the compiler, which lays the owner
        // branch out after this one; with the requests and this wait in one
        // block, no path to the owner's products and decisions has them
        // outstanding, so it waits for nothing newer there.
        __builtin_amdgcn_s_waitcnt(kVm);
      }
    }
    g = __builtin_amdgcn_readfirstlane(g + 1);
    b = __builtin_amdgcn_readfirstlane(b1);
    sw = __builtin_amdgcn_readfirstlane(b1 == 0 ? sw + 1 : sw);
    ok = __builtin_amdgcn_readfirstlane(ok);
  }
  // drain: D_{G-1} into every tile
  if (ok && G > 0) {
    bf16x8 A[2];
    ok = wait_rows(&d_count, G, &dring[(G - 1) % kRing][lc][kh], A);
    if (ok) {
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
          for (int m = 0; m < 2; ++m)
            C[m][tt] = mfma32(A[m], as_bf16x8(Bn[tt][p]), C[m][tt]);
    }
  }
  if (!ok && lane == 0) lds_store(&abort_flag, 1);
  // the addresses of the stores are computed anew: kept from the loads, they
  // would take 64 registers through the loop
  asm volatile("" : "+s"(fields));
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int tt = 0; tt < TPW; ++tt)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        fields[(size_t)(rbase + 32 * m + 8 * (i >> 2) + 4 * kh + (i & 3)) * NP +
               tile_col(w, tt, lc)] = C[m][tt][i];
  __syncthreads();
  for (int i = tid; i < kRT * NPW; i += 256)
    xbits[(size_t)(rbase + i / NPW) * NPW + i % NPW] = xs[i / NPW][i % NPW];
  if (tid < kRT) {
    energy[rbase + tid] = es[tid];
    ebest[rbase + tid] = ebs[tid];
  }
  if (tid == 0 && abort_flag) atomicOr(status, 1);
}

// Random initial bits of instance i (rows [i*R, (i+1)*R)): spin j of replica
// r from counter (j>>7, r, 0, ((instance + i) << 8) | TAG_SWEEP_INIT).
__global__ __launch_bounds__(256) void sweep_init_kernel(int n, int npw, int R, int I, uint32_t k0,
                                                         uint32_t k1, uint32_t instance,
                                                         uint32_t *__restrict__ xbits) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)I * R * npw) return;
  const size_t row = idx / npw;
  const uint32_t inst = (uint32_t)(row / R);
  const uint32_t r = (uint32_t)(row % R);
  const int wd = (int)(idx % npw);
  const int j0 = wd * 32;
  const uint32_t tag = ((instance + inst) << 8) | TAG_SWEEP_INIT;
  const uint4 o = philox4x32_10(make_uint4((uint32_t)(j0 >> 7), r, 0u, tag), k0, k1);
  uint32_t v = pick(o, (j0 >> 5) & 3);
  const int valid = n - j0;
  if (valid < 32) v = valid <= 0 ? 0u : (v & ((1u << valid) - 1u));
  xbits[idx] = v;
}

// Warm start of instance i: x_j = (u < p[i][j]), u = (w >> 8) * 2^-24 from
// counter (j>>2, r, 0, ((instance + i) << 8) | TAG_WARM).
__global__ __launch_bounds__(256) void warm_init_kernel(int n, int npw, int R, int I, uint32_t k0,
                                                        uint32_t k1, uint32_t instance,
                                                        const float *__restrict__ p,
                                                        uint32_t *__restrict__ xbits) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (size_t)I * R * npw) return;
  const size_t row = idx / npw;
  const uint32_t inst = (uint32_t)(row / R);
  const uint32_t r = (uint32_t)(row % R);
  const int wd = (int)(idx % npw);
  const float *pi = p + (size_t)inst * n;
  const uint32_t tag = ((instance + inst) << 8) | TAG_WARM;
  uint32_t v = 0;
  for (int q = 0; q < 8; ++q) {
    const int j0 = wd * 32 + 4 * q;
    if (j0 >= n) break;
    const uint4 o = philox4x32_10(make_uint4((uint32_t)(j0 >> 2), r, 0u, tag), k0, k1);
    for (int jj = 0; jj < 4; ++jj) {
      const int j = j0 + jj;
      if (j < n && (float)(pick(o, jj) >> 8) * 0x1p-24f < pi[j]) v |= 1u << (4 * q + jj);
    }
  }
  xbits[idx] = v;
}

// Population annealing: row (instance i, r) of the new population is row
// (i, anc[i][r]) of the old one for r < R; thread = (row, column).
__global__ __launch_bounds__(256) void dense_gather_kernel(int Rp, int R, int npw, int np,
                                                           const uint32_t *__restrict__ anc,
                                                           const uint32_t *__restrict__ x,
                                                           const float *__restrict__ f,
                                                           const double *__restrict__ e,
                                                           uint32_t *__restrict__ x2,
                                                           float *__restrict__ f2,
                                                           double *__restrict__ e2) {
  const int row = blockIdx.y;
  const int col = blockIdx.x * 256 + threadIdx.x;
  const int inst = row / Rp, r = row % Rp;
  const int src = r < R ? inst * Rp + (int)anc[(size_t)inst * R + r] : row;
  if (col < np) f2[(size_t)row * np + col] = f[(size_t)src * np + col];
  if (col < npw) x2[(size_t)row * npw + col] = x[(size_t)src * npw + col];
  if (col == 0) e2[row] = e[src];
}

void launch_dense_gather(hipStream_t st, int num_instances, int Rp, int R, int npw, int np,
                         const uint32_t *anc, const uint32_t *x, const float *f, const double *e,
                         uint32_t *x2, float *f2, double *e2) {
  const dim3 grid((unsigned)((np + 255) / 256), (unsigned)(num_instances * Rp));
  dense_gather_kernel<<<grid, 256, 0, st>>>(Rp, R, npw, np, anc, x, f, e, x2, f2, e2);
  OS_HIP_CHECK(hipGetLastError());
}

// Replica exchange round `round` on the GPU, for the dense and the sparse
// paths (replica r of instance i at row i * Rp + r): thread = (instance,
// ladder, pair p); slots k = round % 2 + 2p and k + 1 of the ladder swap
// their replicas a, b iff d = (1/ts_k - 1/ts_{k+1}) (E_a - E_b) >= 0 or
// u < exp(d), u = (w >> 8) 2^-24 from word 0 of Philox counter (k, l, round,
// ((instance_base + i) << 8) | TAG_EXCHANGE); the swapped replicas take their
// new slots' scales in tsr.  The pairs of a round are disjoint.
__global__ __launch_bounds__(64) void exchange_round_kernel(
    int I, int L, int K, int R, int Rp, uint32_t round, uint32_t k0, uint32_t k1,
    uint32_t inst_base, const float *__restrict__ ts_slots, const double *__restrict__ e,
    uint32_t *__restrict__ rep_at, uint32_t *__restrict__ slot_of, float *__restrict__ tsr) {
  const int pairs = K / 2;
  const int idx = blockIdx.x * 64 + threadIdx.x;
  if (idx >= I * L * pairs) return;
  const int i = idx / (L * pairs), l = (idx / pairs) % L, p = idx % pairs;
  const int k = (int)(round & 1u) + 2 * p;
  if (k + 1 >= K) return;
  const size_t ro = (size_t)i * Rp;
  uint32_t *ra = rep_at + (size_t)i * R + (size_t)l * K;
  const uint32_t a = ra[k], b = ra[k + 1];
  const double d =
      (1.0 / (double)ts_slots[k] - 1.0 / (double)ts_slots[k + 1]) * (e[ro + a] - e[ro + b]);
  const uint4 o = philox4x32_10(
      make_uint4((uint32_t)k, (uint32_t)l, round, ((inst_base + (uint32_t)i) << 8) | TAG_EXCHANGE),
      k0, k1);
  const double u = (double)(o.x >> 8) * 0x1p-24;
  if (d >= 0.0 || u < exp(d)) {
    ra[k] = b;
    ra[k + 1] = a;
    slot_of[(size_t)i * R + a] = (uint32_t)(k + 1);
    slot_of[(size_t)i * R + b] = (uint32_t)k;
    tsr[ro + a] = ts_slots[k + 1];
    tsr[ro + b] = ts_slots[k];
  }
}

void launch_exchange_round(hipStream_t st, int I, int L, int K, int R, int Rp, uint32_t round,
                           uint64_t seed, uint32_t inst_base, const float *ts_slots,
                           const double *e, uint32_t *rep_at, uint32_t *slot_of, float *tsr) {
  const int threads = I * L * (K / 2);
  if (threads == 0) return;
  exchange_round_kernel<<<(threads + 63) / 64, 64, 0, st>>>(
      I, L, K, R, Rp, round, (uint32_t)seed, (uint32_t)(seed >> 32), inst_base, ts_slots, e,
      rep_at, slot_of, tsr);
  OS_HIP_CHECK(hipGetLastError());
}

int dense_max_n() { return kWaves * 32 * 8; }

// Column tiles (32 columns) per wave are instantiated for these counts; n is
// padded up to the next one (128 columns per step).
static const int kTpwList[] = {1, 2, 3, 4, 6, 8};

int dense_padded_n(int n) {
  const int need = (n + kWaves * 32 - 1) / (kWaves * 32);
  for (int t : kTpwList)
    if (t >= need) return t * kWaves * 32;
  return -1;
}

void launch_dense_sweeps(hipStream_t st, int n, int np, int num_instances, const uint4 *qpack,
                         const float *qdb, const float *tscale, const float *tsr, int sweep0,
                         int nsweeps, uint64_t seed, uint32_t instance, int R_pad, float *fields,
                         uint32_t *xbits, uint32_t *bestbits, double *energy, double *ebest,
                         int *status) {
  const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
  const int gpi = R_pad / kRT;
  const dim3 grid(num_instances * gpi), block(kWaves * 64);
  // blocks a sweep visits: those with spins, up to a whole turn of the waves
  const int nb = kWaves * ((n + 16 * kWaves - 1) / (16 * kWaves));
  switch (np / (kWaves * 32)) {
#define OS_DENSE_CASE(T)                                                                    \
  case T:                                                                                   \
    dense_sweep_kernel<T><<<grid, block, 0, st>>>(n, nb, qpack, qdb, tscale, tsr, sweep0,     \
                                                  nsweeps, k0, k1, instance, gpi, fields,     \
                                                  xbits, bestbits, energy, ebest, status);    \
    break;
    OS_DENSE_CASE(1)
    OS_DENSE_CASE(2)
    OS_DENSE_CASE(3)
    OS_DENSE_CASE(4)
    OS_DENSE_CASE(6)
    OS_DENSE_CASE(8)
#undef OS_DENSE_CASE
    default:
      throw Error(-3, "dense sweep kernel: unsupported padded size");
  }
  OS_HIP_CHECK(hipGetLastError());
}

void launch_sweep_init(hipStream_t st, int n, int npw, int R, uint64_t seed, uint32_t instance,
                       uint32_t *xbits, int num_instances) {
  const size_t total = (size_t)num_instances * R * npw;
  if (total == 0) return;
  sweep_init_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>(
      n, npw, R, num_instances, (uint32_t)seed, (uint32_t)(seed >> 32), instance, xbits);
  OS_HIP_CHECK(hipGetLastError());
}

void launch_warm_init(hipStream_t st, int n, int npw, int R, uint64_t seed, uint32_t instance,
                      const float *p, uint32_t *xbits, int num_instances) {
  const size_t total = (size_t)num_instances * R * npw;
  if (total == 0) return;
  warm_init_kernel<<<(unsigned)((total + 255) / 256), 256, 0, st>>>(
      n, npw, R, num_instances, (uint32_t)seed, (uint32_t)(seed >> 32), instance, p, xbits);
  OS_HIP_CHECK(hipGetLastError());
}

}  // namespace os
