// Attention contractions: the batched fp16 product of strided or
// channel-blocked operands (with head groups and channel ranges) and the
// blocked channel gather that feeds it.
//
// The product keeps the reference's numerical contract: every output is the
// fp32 sum of its k products taken in reduction order 0, 1, ..., K-1 from a
// zero start, then one round-to-nearest-even cast to fp16.  fp16 x fp16
// products are exact in fp32 (22 significant bits, exponents far from the fp32
// limits), so fma(a, b, acc) rounds exactly like acc + a * b and a per-output
// chain of fmas reproduces the sequential sum bit for bit.  On gfx950
// v_mfma_f32_16x16x4_f32 is such a chain: it adds its four products to the
// accumulator one after the other in ascending k, one fp32 rounding each
// (tests/test_gpu_bmm.py compares every form with the sequential sum, with
// signed zeros, subnormals, infinities and NaN among the operands).  The fp16 matrix instructions are not, and a
// split of the reduction is not either, so the operands are widened to fp32
// and the parallelism is across outputs only.
#include "common.h"

#include <string.h>

#include <algorithm>

namespace thin {
namespace {

// One axis of a logical matrix: index i sits at element offset
// (i / blk) * outer + (i % blk) * inner.
struct Axis {
  FastDiv blk;
  int64_t outer, inner;
  __host__ __device__ __forceinline__ int64_t at(uint32_t i) const {
    const uint32_t q = blk.div(i);
    return (int64_t)q * outer + (int64_t)(i - q * blk.d) * inner;
  }
};

// A logical [batch, rows, cols] matrix over fp16 storage (bmm_flow.cpp:19-33,
// 193-215): element (b, r, c) sits at b * batch + row.at(r + row_origin +
// b * row_group) + col.at(c + col_origin + b * col_group).  Head groups of a
// blocked operand have batch stride 0 and a per-group channel origin.
struct Mat {
  _Float16* p;
  int64_t batch;
  uint32_t row_origin, col_origin, row_group, col_group;
  Axis row, col;
  __device__ __forceinline__ int64_t at(uint32_t b, uint32_t r, uint32_t c) const {
    return (int64_t)b * batch + row.at(r + row_origin + b * row_group) + col.at(c + col_origin + b * col_group);
  }
};

// ---------------------------------------------------------------- matrix-core product
// One operand of the product as the kernels read it: `rows` logical rows, each
// K steps long.
struct Side {
  const _Float16* p;
  int64_t batch;
  int64_t hop;  // bytes from a chunk of steps (bmm_kernel) or a tile of rows (bmm_short_kernel's P) to the next
  uint32_t row_origin, step_origin, row_group, step_group, rows;
  uint32_t last_run;  // first step of the last run of 8 to load: K - 8 on a plain axis, whose memory may end with the
                      // row, the last multiple of 8 below K on a blocked one, whose blocks hold whole runs
  uint32_t last_rows;  // the same of the runs of 8 rows, and what it leaves where rows of a plain axis are no multiple
  uint32_t early;      // of 8: rows by which the last tile starts early, or, of a single tile,
  uint32_t ragged;     // the rows in that run
  bool steps_near;    // the smaller stride is along the steps
  Axis row, step;
};

// The output with the axis that is contiguous in memory as `p` (the matrix
// instruction gives a lane 4 consecutive rows of its tile, so that axis rides
// on the instruction's rows) and the other as `q`.
struct BmmPlan {
  Side P, Q;
  _Float16* y;
  int64_t ybatch;
  uint32_t yp_group;  // p indexes between batch entries (grouped blocked outputs)
  uint32_t y_vec;     // runs of 4 * W outputs along p from multiples of 4 * W are contiguous
  Axis yp, yq;
  uint32_t k;
  uint32_t span;      // bmm_short_kernel: P tiles per block,
  int64_t yhop;       // and output elements from one to the next
  uint32_t ptiles;
  uint32_t walk;      // blocks of an axis do not divide a chunk (a tile): offsets anew for each, no hops
  FastDiv pblocks, qtiles;
};

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h8u __attribute__((ext_vector_type(8), aligned(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

// The last n (1-7) of 8 elements to the front, zeros behind.
__device__ __forceinline__ h8 tail_first(const h8& v, uint32_t n) {
  typedef uint64_t u2 __attribute__((ext_vector_type(2)));
  const u2 d = __builtin_bit_cast(u2, v);
  const uint32_t cut = 16u * (8u - n);
  return __builtin_bit_cast(
      h8, cut < 64u ? (u2){d[0] >> cut | d[1] << (64u - cut), d[1] >> cut} : (u2){d[1] >> (cut - 64u), 0});
}

constexpr uint32_t kBmmThreads = 256;  // 4 waves, 2 x 2 over the block's tile

// The f32 matrix instruction shares its issue with the VALU (each VALU
// instruction between two of them costs about 8 cycles; one takes 32), so the
// loops hold as little else as they can: operands are widened to fp32 once, on
// their way into LDS (widening each lane's operands in the loop instead: 111
// of 140 TFLOP/s in a loop of products alone), the loads take a scalar base
// and a lane offset that stays the same from chunk to chunk, and LDS buffers
// are compile-time offsets.
//
// Staging of one operand's R rows x KD steps.  Every load is a 16-byte run of
// 8 steps of a row or 8 rows of a step (any 2-byte alignment) at an address
// clamped into the operand, with no branch around it, so that all of a chunk's
// loads are in flight at once.
//
// Step-major operands (RF false: the steps of a row are adjacent in memory)
// lie in LDS per 32 steps as [row][8 slots][4 floats]: the instruction's lane
// (i, g) takes step 4s + g of row i in its s-th call, so calls 4h..4h+3 are
// slot (h, g), one 16-byte read.  Slot h is swapped by bit 1 of the row and g
// xored with minus the row's group of four, which puts each 16 lanes that a
// 16-byte read serves at once (0-3, 12-15, 20-27; 4-11, 16-19, 28-31) on
// distinct banks; 32-step groups are one slot apart for the writes.
// Row-major operands (RF true: the rows of a step are adjacent) lie
// [step][row], a lane reading its W adjacent rows of one step at a time; half
// a row group is swapped for alternate steps (W = 2) or step pairs (W = 1),
// so that the four steps of a call lie on distinct banks.
//
// SECOND: an operand of fewer units than threads takes the upper threads.
template <bool RF, int KD, int R, int W, bool SECOND = false>
struct Stage {
  static constexpr uint32_t kGroup = R * 32 + 4;                     // !RF: floats per 32 steps
  static constexpr uint32_t kFloats = RF ? KD * R : KD / 32 * kGroup;
  static constexpr uint32_t kUnits = RF ? KD * R / 8 : KD * R / 16;  // a run of 8 / two runs of 8 steps
  static constexpr uint32_t kPer = kUnits < kBmmThreads ? 1 : kUnits / kBmmThreads;
  static constexpr uint32_t kAcross = RF ? R / 8 : KD / 16;          // units side by side along the memory axis
  static constexpr uint32_t kNext = kBmmThreads / kAcross;           // steps between a thread's units
  static_assert(RF || kPer == 1, "one unit of a step-major operand per thread");
  static constexpr uint32_t kLoads = RF ? kPer : 2;

  uint32_t off[kLoads];            // bytes from the base of the batch entry
  uint32_t to[RF ? 1 : 4];         // LDS position (floats)
  using Regs = h8[kLoads];

  static __device__ __forceinline__ uint32_t tid() {
    return SECOND && kUnits < kBmmThreads ? threadIdx.x ^ (kBmmThreads / 2) : threadIdx.x;
  }
  static __device__ __forceinline__ bool active() { return kUnits >= kBmmThreads || tid() < kUnits; }
  static __device__ __forceinline__ uint32_t across() { return tid() % kAcross; }
  // the row (step) of the thread's unit: 32-step chunks, two units to a row,
  // deal rows 1, 8 and 16 apart to neighbouring threads, whose LDS writes then
  // fall on distinct banks
  static __device__ __forceinline__ uint32_t along() {
    const uint32_t a = tid() / kAcross;
    if (RF || KD != 32) return a;
    return (a & 33u) | (a & 6u) << 2 | (a & 24u) >> 2;
  }
  static __device__ __forceinline__ uint32_t slot(uint32_t row, uint32_t h, uint32_t g) {
    return row * 32u + ((h ^ (row >> 1 & 1u)) * 4u + (g ^ ((0u - row / (4u * W)) & 3u))) * 4u;
  }
  static __device__ __forceinline__ uint32_t swapped(uint32_t step, uint32_t row) {  // RF: place in the step
    return W == 2 ? row ^ (step & 1u) * 32u : row ^ (step >> 1 & 1u) * 16u;
  }

  static __device__ __forceinline__ const char* base(const Side& s, uint32_t bt) {
    return reinterpret_cast<const char*>(s.p + (int64_t)bt * s.batch);
  }

  __device__ __forceinline__ void place() {
    if constexpr (RF) {
      to[0] = along() * R + swapped(along(), across() * 8u);  // kNext is a multiple of 4
    } else {
#pragma unroll
      for (uint32_t g = 0; g < 4; ++g) to[g] = across() / 2 * kGroup + slot(along(), across() & 1u, g);
    }
  }

  // offsets of the tile from row r0 and step k0
  __device__ __forceinline__ void aim(const Side& s, uint32_t bt, uint32_t r0, uint32_t k0, uint32_t K) {
    const uint32_t ro = s.row_origin + bt * s.row_group, so = s.step_origin + bt * s.step_group;
    if constexpr (RF) {
      const int64_t row = s.row.at(ro + min(r0 + across() * 8u, s.last_rows));
#pragma unroll
      for (uint32_t u = 0; u < kPer; ++u)
        off[u] = (uint32_t)(row + s.step.at(so + min(k0 + along() + u * kNext, K - 1u))) * 2u;
    } else {
      const int64_t row = s.row.at(ro + min(r0 + along(), s.rows - 1u));
#pragma unroll
      for (uint32_t h = 0; h < 2; ++h)
        off[h] = (uint32_t)(row + s.step.at(so + min(k0 + across() * 16u + 8u * h, s.last_run))) * 2u;
    }
  }

  __device__ __forceinline__ void load(const char* b, Regs& v) {
#pragma unroll
    for (uint32_t u = 0; u < kLoads; ++u) {
      __asm__("" : "+v"(off[u]));  // keeps the offset 32 bits wide: one scalar base and one register a load
      v[u] = *reinterpret_cast<const h8u*>(b + off[u]);
    }
  }

  // zeroes the steps past the end (a zero product leaves every sum as it is);
  // the run of steps across the end was loaded from last_run on
  __device__ __forceinline__ void trim(const Side& s, uint32_t k0, uint32_t K, Regs& v) const {
    const h8 zero = (h8)(_Float16)0;
#pragma unroll
    for (uint32_t u = 0; u < kLoads; ++u) {
      if constexpr (RF) {
        if (k0 + along() + u * kNext >= K) v[u] = zero;
      } else {
        typedef uint64_t u2 __attribute__((ext_vector_type(2)));
        const uint32_t k = k0 + across() * 16u + 8u * u, c = K & 7u;  // c steps of the run across the end
        if (c && k < K && k + 8u > K) {
          if (s.step.blk.d == 1) {  // they are the last c of the 8
            v[u] = tail_first(v[u], c);
          } else {  // the first c of the 8
            const u2 d = __builtin_bit_cast(u2, v[u]);
            const uint64_t keep = (1ull << 16u * (c & 3u)) - 1u;
            v[u] = __builtin_bit_cast(h8, c < 4u ? (u2){d[0] & keep, 0} : (u2){d[0], d[1] & keep});
          }
        }
        if (k >= K) v[u] = zero;
      }
    }
  }

  template <bool ODD>
  __device__ __forceinline__ void store(const Side& s, float* lds, Regs& v) const {
    if constexpr (RF && ODD) {
      if (s.ragged && across() == s.rows / 8u) {
#pragma unroll
        for (uint32_t u = 0; u < kPer; ++u) v[u] = tail_first(v[u], s.ragged);
      }
    }
    if (!active()) return;
    if constexpr (RF) {
#pragma unroll
      for (uint32_t u = 0; u < kPer; ++u) {
        f4* d = reinterpret_cast<f4*>(lds + to[0] + u * kNext * R);
        d[0] = (f4){(float)v[u][0], (float)v[u][1], (float)v[u][2], (float)v[u][3]};
        d[1] = (f4){(float)v[u][4], (float)v[u][5], (float)v[u][6], (float)v[u][7]};
      }
    } else {
#pragma unroll
      for (uint32_t g = 0; g < 4; ++g)
        *reinterpret_cast<f4*>(lds + to[g]) =
            (f4){(float)v[0][g], (float)v[0][g + 4], (float)v[1][g], (float)v[1][g + 4]};
    }
  }

  // tile row that instruction row i of the wave's tile t holds; the 4 rows a
  // lane gets back, over the W tiles, are 4 * W consecutive ones either way
  static __device__ __forceinline__ uint32_t row_of(uint32_t i, uint32_t t) {
    return RF ? i * W + t : (i >> 2) * (4u * W) + 4u * t + (i & 3u);
  }
  // position of (instruction row r of 4, tile t) in those 4 * W rows
  static __device__ __forceinline__ constexpr uint32_t place_of(uint32_t r, uint32_t t) { return RF ? r * W + t : 4u * t + r; }
};

// A wave's reads of W tiles of an operand, 8 calls (32 steps) at a time.
template <bool RF, int KD, int R, int W>
struct Operand {
  using S = Stage<RF, KD, R, W>;
  typedef float fw __attribute__((ext_vector_type(W)));
  uint32_t at[RF ? 1 : 2 * W];
  struct Group {
    f4 steps[RF ? 1 : W][2];
    fw rows[RF ? 8 : 1];
    __device__ __forceinline__ float value(uint32_t s, uint32_t t) const {
      if constexpr (RF) return rows[s][t];
      else return steps[t][s / 4][s % 4];
    }
  };

  __device__ __forceinline__ void init(uint32_t wave_row, uint32_t lane) {
    const uint32_t i = lane & 15u, g = lane >> 4;
    if constexpr (RF) {
      at[0] = g * R + S::swapped(g, wave_row + i * W);
    } else {
#pragma unroll
      for (uint32_t t = 0; t < W; ++t)
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) at[2 * t + h] = S::slot(wave_row + S::row_of(i, t), h, g);
    }
  }
  __device__ __forceinline__ void read(Group& d, const float* lds, uint32_t c32) const {
    if constexpr (RF) {
#pragma unroll
      for (uint32_t s = 0; s < 8; ++s) d.rows[s] = *reinterpret_cast<const fw*>(lds + at[0] + (c32 * 32u + 4u * s) * R);
    } else {
#pragma unroll
      for (uint32_t t = 0; t < W; ++t)
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h)
          d.steps[t][h] = *reinterpret_cast<const f4*>(lds + at[2 * t + h] + c32 * S::kGroup);
    }
  }
};

// FIRST: from zero sums
template <int W, bool FIRST = false, class GP, class GQ>
__device__ __forceinline__ void bmm_call(f4 (&acc)[W][W], const GP& gp, const GQ& gq, uint32_t s) {
#pragma unroll
  for (int i = 0; i < W; ++i)
#pragma unroll
    for (int j = 0; j < W; ++j)
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(gp.value(s, i), gq.value(s, j),
                                                       FIRST ? (f4){0.f, 0.f, 0.f, 0.f} : acc[i][j], 0, 0, 0);
}

// The wave's outputs: p index pr holds the lane's first, rows below plo / qlo
// belong to another block.
template <int W, class SP, class SQ>
__device__ __forceinline__ void bmm_write(const BmmPlan& p, uint32_t bt, const f4 (&acc)[W][W], uint32_t pr, uint32_t plo,
                                          uint32_t q0, uint32_t qlo, uint32_t lane) {
  _Float16* y = p.y + (int64_t)bt * p.ybatch;
  const uint32_t po = pr + bt * p.yp_group;
#pragma unroll
  for (uint32_t t = 0; t < W; ++t) {
    const uint32_t q = q0 + SQ::row_of(lane & 15u, t);
    if (q >= p.Q.rows || q < qlo) continue;
    typedef _Float16 hv __attribute__((ext_vector_type(4 * W), aligned(2)));
    hv o;
#pragma unroll
    for (uint32_t a = 0; a < W; ++a)
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) o[SP::place_of(r, a)] = (_Float16)acc[a][t][r];
    _Float16* row = y + p.yq.at(q);
    if (p.y_vec && pr >= plo && pr + 4u * W <= p.P.rows) {
      *reinterpret_cast<hv*>(row + p.yp.at(po)) = o;
    } else {
#pragma unroll
      for (uint32_t e = 0; e < 4 * W; ++e)
        if (pr + e >= plo && pr + e < p.P.rows) row[p.yp.at(po + e)] = o[e];
    }
  }
}

// First row of a tile: the last tile of an operand whose rows lie on a plain
// axis and are no multiple of 8 starts up to 7 rows early, so that its rows
// are whole runs (the rows it shares with the tile before are not written).
// The blocks of a blocked axis hold whole runs.
template <bool RF>
__device__ __forceinline__ uint32_t tile_row(const Side& s, uint32_t tile, uint32_t tiles, uint32_t r) {
  return RF && tile + 1u == tiles ? tile * r - s.early : tile * r;
}

template <int B>
struct Const {
  static constexpr int value = B;
};

// y[p, q] = sum_k P[p, k] Q[q, k] for K > 32, a block of 4 waves per 32W x 32W
// outputs, W x W instruction tiles per wave.  Chunks of KD steps alternate
// between two LDS buffers; the loads of the next two chunks are in flight under
// the products of this one (one: 41.2 against 36.4 us for the batched v p^T,
// four: 40.7).
//
// Bound by the issue of the products and of the VALU work beside them: at
// [128,64,400] x [128,400,400] the matrix pipe is busy 41,600 of the 77,700
// cycles that the launch keeps a shader engine busy (54%).  34.3 us back to back
// on the same operands, 37.8 in a kernel trace over changing ones (80.5 with the
// fma chains this replaced), against the 17 us that the products alone take at
// 153 TFLOP/s.
//
// ODD: blocks that do not divide a chunk, or rows of one tile that end in a
// partial run (walk, ragged).  With their tests in every product's loop, v p^T
// of 1600 tokens took 20.7-21.8 us instead of 20.4.
template <int KD, int W, bool PR, bool QR, bool ODD>
__global__ __launch_bounds__(kBmmThreads, W == 2 ? 3 : 2) void bmm_kernel(BmmPlan p) {
  constexpr int R = 32 * W;
  using SP = Stage<PR, KD, R, W>;
  using SQ = Stage<QR, KD, R, W, true>;
  using OP = Operand<PR, KD, R, W>;
  using OQ = Operand<QR, KD, R, W>;
  constexpr int PF = 2;
  constexpr uint32_t kBuf = SP::kFloats + SQ::kFloats;
  __shared__ __attribute__((aligned(16))) float lds[2 * kBuf];
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t rest = p.pblocks.div(blockIdx.x), pt = blockIdx.x - rest * p.pblocks.d;
  const uint32_t bt = p.qtiles.div(rest), qt = rest - bt * p.qtiles.d;
  const uint32_t K = p.k;
  const uint32_t p0 = tile_row<PR>(p.P, pt, p.ptiles, R), q0 = tile_row<QR>(p.Q, qt, p.qtiles.d, R);
  const uint32_t last = (K - 1u) / KD;  // the last chunk, whole or not

  SP sp;
  SQ sq;
  typename SP::Regs vp[PF];
  typename SQ::Regs vq[PF];
  const char* bp = SP::base(p.P, bt);
  const char* bq = SQ::base(p.Q, bt);
  sp.aim(p.P, bt, p0, 0, K);
  sq.aim(p.Q, bt, q0, 0, K);
  uint32_t n = 0;  // the next chunk to load
  // chunk n into register set n % PF; past the last chunk that one again,
  // which nothing stores: a test around the loads would leave the waits
  // without a count of the loads behind the one they wait for
  auto load = [&](int set) __attribute__((always_inline)) {
    if (n == last || (ODD && n < last && p.walk)) {
      sp.aim(p.P, bt, p0, ODD ? n * KD : last * KD, K);
      sq.aim(p.Q, bt, q0, ODD ? n * KD : last * KD, K);
      bp = SP::base(p.P, bt);
      bq = SQ::base(p.Q, bt);
    }
    sp.load(bp, vp[set]);
    sq.load(bq, vq[set]);
    if (n < last) {
      bp += p.P.hop;
      bq += p.Q.hop;
    }
    ++n;
  };
#pragma unroll
  for (int set = 0; set < PF; ++set) load(set);
  sp.place();
  sq.place();
  const uint32_t wp = (wave & 1u) * 16u * W, wq = (wave >> 1) * 16u * W;  // the wave's rows in the tile
  const bool work = p0 + wp < p.P.rows && q0 + wq < p.Q.rows;
  OP op;
  OQ oq;
  op.init(wp, lane);
  oq.init(wq, lane);
  f4 acc[W][W];
#pragma unroll
  for (int a = 0; a < W; ++a)
#pragma unroll
    for (int b = 0; b < W; ++b) acc[a][b] = (f4){0.f, 0.f, 0.f, 0.f};

  typename OP::Group gp[2];
  typename OQ::Group gq[2];
  uint32_t c = 0;  // the chunk to multiply
  auto store = [&](int set, float* to, bool end) __attribute__((always_inline)) {
    if (end) {
      sp.trim(p.P, last * KD, K, vp[set]);
      sq.trim(p.Q, last * KD, K, vq[set]);
    }
    sp.template store<ODD>(p.P, to, vp[set]);
    sq.template store<ODD>(p.Q, to + SP::kFloats, vq[set]);
  };
  // chunk c = S mod PF from its buffer, chunk c + 1 into the other
  auto step = [&](auto S) __attribute__((always_inline)) {
    constexpr int set = decltype(S)::value;
    constexpr uint32_t kFrom = set & 1 ? kBuf : 0, kTo = kBuf - kFrom;
    load(set);
    if (work) {
      op.read(gp[0], lds + kFrom, 0);
      oq.read(gq[0], lds + kFrom + SP::kFloats, 0);
#pragma unroll
      for (uint32_t g = 0; g < KD / 32; ++g) {
        if (g + 1 < KD / 32) {  // the next 32 steps, under the products of these
          op.read(gp[(g + 1) & 1], lds + kFrom, g + 1);
          oq.read(gq[(g + 1) & 1], lds + kFrom + SP::kFloats, g + 1);
        }
#pragma unroll
        for (uint32_t s = 0; s < 8; ++s) bmm_call<W>(acc, gp[g & 1], gq[g & 1], s);
      }
    }
    ++c;
    // every wave was done with that buffer's chunk c - 1 at the last barrier
    store((set + 1) % PF, lds + kTo, c == last);
    __syncthreads();
    return c < last;
  };
  store(0, lds, last == 0);
  __syncthreads();
  if (last) {
    while (step(Const<0>()) && step(Const<1>())) {
    }
  }
  if (!work) return;
  const float* from = lds + (last & 1u ? kBuf : 0u);
  uint32_t calls = (K - last * KD + 3u) / 4u;
  for (uint32_t g = 0; calls; ++g) {
    op.read(gp[0], from, g);
    oq.read(gq[0], from + SP::kFloats, g);
    if (calls >= 8u) {
#pragma unroll
      for (uint32_t s = 0; s < 8; ++s) bmm_call<W>(acc, gp[0], gq[0], s);
      calls -= 8u;
    } else {
#pragma unroll
      for (uint32_t s = 0; s < 7; ++s)
        if (s < calls) bmm_call<W>(acc, gp[0], gq[0], s);
      calls = 0;
    }
  }
  bmm_write<W, SP, SQ>(p, bt, acc, p0 + wp + (lane >> 4) * (4u * W), pt * R, q0 + wq, qt * R, lane);
}

// The same for K <= 32 (one chunk): the block keeps its Q operand in registers
// and walks `span` P tiles, the next tile's loads in flight under the products
// and stores of this one.  At [128,400,32] x [128,32,400] 24.4 us (96.9 with
// the fma chains this replaced): 9 us of it without products and stores, the
// products add 11 and the stores of 41 MB 3 to 4.
template <int W, bool PR, bool QR, bool ODD>
__global__ __launch_bounds__(kBmmThreads) void bmm_short_kernel(BmmPlan p) {
  constexpr int KD = 32, R = 32 * W;
  using SP = Stage<PR, KD, R, W>;
  using SQ = Stage<QR, KD, R, W, true>;
  using OP = Operand<PR, KD, R, W>;
  using OQ = Operand<QR, KD, R, W>;
  __shared__ __attribute__((aligned(16))) float lds[SQ::kFloats + 2 * SP::kFloats];
  const uint32_t lane = threadIdx.x & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t rest = p.pblocks.div(blockIdx.x), pb = blockIdx.x - rest * p.pblocks.d;
  const uint32_t bt = p.qtiles.div(rest), qt = rest - bt * p.qtiles.d;
  const uint32_t K = p.k;
  const uint32_t q0 = tile_row<QR>(p.Q, qt, p.qtiles.d, R);
  uint32_t pt = pb * p.span;
  const uint32_t pend = min(pt + p.span, p.ptiles);

  SP sp;
  SQ sq;
  typename SP::Regs vp;
  typename SQ::Regs vq;
  const char* bp = SP::base(p.P, bt);
  uint32_t p0 = tile_row<PR>(p.P, pt, p.ptiles, R);
  sp.aim(p.P, bt, p0, 0, K);
  sq.aim(p.Q, bt, q0, 0, K);
  sq.load(SQ::base(p.Q, bt), vq);
  sp.load(bp, vp);
  sp.place();
  sq.place();
  const uint32_t wp = (wave & 1u) * 16u * W, wq = (wave >> 1) * 16u * W;
  OP op;
  OQ oq;
  op.init(wp, lane);
  oq.init(wq, lane);
  float* const ldsp = lds + SQ::kFloats;
  if (K < KD) {
    sq.trim(p.Q, 0, K, vq);
    sp.trim(p.P, 0, K, vp);
  }
  sq.template store<ODD>(p.Q, lds, vq);
  sp.template store<ODD>(p.P, ldsp, vp);
  __syncthreads();
  typename OQ::Group gq;
  oq.read(gq, lds, 0);
  const uint32_t calls = (K + 3u) / 4u;
  // the lane's outputs of a whole tile: one run of 4 * W per q row
  typedef _Float16 hv __attribute__((ext_vector_type(4 * W), aligned(2)));
  _Float16* out[W];
  bool mine[W];
#pragma unroll
  for (uint32_t t = 0; t < W; ++t) {
    const uint32_t q = q0 + wq + SQ::row_of(lane & 15u, t);
    mine[t] = q < p.Q.rows && q >= qt * R;
    out[t] = p.y + ((int64_t)bt * p.ybatch + p.yq.at(min(q, p.Q.rows - 1u)) +
                    p.yp.at(pt * R + wp + (lane >> 4) * (4u * W) + bt * p.yp_group));
  }
  auto step = [&](auto B) __attribute__((always_inline)) {  // tile pt from buffer B, the next one into the other
    constexpr uint32_t kFrom = decltype(B)::value ? SP::kFloats : 0, kTo = SP::kFloats - kFrom;
    const bool more = pt + 1u < pend;
    const uint32_t pr = p0 + wp;
    if (more) {
      p0 = tile_row<PR>(p.P, pt + 1u, p.ptiles, R);
      if (pt + 2u == p.ptiles || (ODD && p.walk)) {
        sp.aim(p.P, bt, p0, 0, K);
        bp = SP::base(p.P, bt);
      } else {
        bp += p.P.hop;
      }
      sp.load(bp, vp);
    }
    const bool work = pr < p.P.rows && q0 + wq < p.Q.rows;
    f4 acc[W][W];
    if (work) {
      typename OP::Group gp;
      op.read(gp, ldsp + kFrom, 0);
      bmm_call<W, true>(acc, gp, gq, 0);
      if (calls == 8u) {
#pragma unroll
        for (uint32_t s = 1; s < 8; ++s) bmm_call<W>(acc, gp, gq, s);
      } else {
#pragma unroll
        for (uint32_t s = 1; s < 7; ++s)
          if (s < calls) bmm_call<W>(acc, gp, gq, s);
      }
    }
    // the next tile into LDS before this one's outputs are stored: its loads
    // and the stores are counted together, and a wait for them after the
    // stores waits for the stores as well (24.9 against 23.9 us at
    // [128,400,32] x [128,32,400])
    if (more) {
      if (K < KD) sp.trim(p.P, 0, K, vp);
      sp.template store<ODD>(p.P, ldsp + kTo, vp);
    }
    if (work) {
      if (p.y_vec && pt + 1u < p.ptiles) {
#pragma unroll
        for (uint32_t t = 0; t < W; ++t) {
          hv o;
#pragma unroll
          for (uint32_t a = 0; a < W; ++a)
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r) o[SP::place_of(r, a)] = (_Float16)acc[a][t][r];
          if (mine[t]) *reinterpret_cast<hv*>(out[t]) = o;
          out[t] += p.yhop;
        }
      } else {
        bmm_write<W, SP, SQ>(p, bt, acc, pr + (lane >> 4) * (4u * W), pt * R, q0 + wq, qt * R, lane);
      }
    }
    if (more) __syncthreads();
    ++pt;
  };
  for (;;) {
    step(Const<0>());
    if (pt >= pend) break;
    step(Const<1>());
    if (pt >= pend) break;
  }
}

// Steps per chunk of bmm_kernel, measured on v p^T: the 64 x 64 form, with
// three or four blocks on a compute unit, takes 36.4 us with 32 at
// [128,64,400] x [128,400,400] and 39.2 with 64; the 32 x 32 form, with one or
// two, 21.7 us with 128 at [4,64,1600] x [4,1600,1600] and 23.7 with 64.
constexpr int bmm_depth(int w) { return w == 2 ? 32 : 128; }

// Any strides: the elements are gathered, 32 steps a chunk, into [step][row]
// tiles of RP and RQ rows (RP * RQ = 1024), one 16 x 16 instruction tile per
// wave.  Bound by the element loads and their addresses, so an operand of at
// most 16 rows takes a tile of 16 ([128,8,400] x [128,400,400], both of stride
// 2: 46 us with 32); every load is in range by its clamped index (under a
// test, each waits for the one before: 1.5x), and 64-step chunks measured
// 1.1-1.8x slower.
template <int RP, int RQ>
__global__ __launch_bounds__(kBmmThreads) void bmm_gather_kernel(BmmPlan p) {
  constexpr int KD = 32;
  static_assert(RP * RQ == 1024, "one 16 x 16 tile for each of 4 waves");
  __shared__ float ldsp[KD * (RP + 1)], ldsq[KD * (RQ + 1)];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t rest = p.pblocks.div(blockIdx.x), pt = blockIdx.x - rest * p.pblocks.d;
  const uint32_t bt = p.qtiles.div(rest), qt = rest - bt * p.qtiles.d;
  const uint32_t K = p.k;
  _Float16 vp[RP * KD / kBmmThreads], vq[RQ * KD / kBmmThreads];
  auto load = [&](auto R, const Side& s, uint32_t tile, uint32_t k0, auto& d) __attribute__((always_inline)) {
    const _Float16* src = s.p + (int64_t)bt * s.batch;
#pragma unroll
    for (uint32_t u = 0; u < sizeof(d) / 2; ++u) {
      const uint32_t e = tid + u * kBmmThreads;
      const uint32_t r = s.steps_near ? e / KD : e % R.value, k = s.steps_near ? e % KD : e / R.value;
      d[u] = src[s.row.at(s.row_origin + bt * s.row_group + min(tile * R.value + r, s.rows - 1u)) +
                 s.step.at(s.step_origin + bt * s.step_group + min(k0 + k, K - 1u))];
    }
  };
  auto store = [&](auto R, const Side& s, uint32_t k0, const auto& d, float* to) __attribute__((always_inline)) {
#pragma unroll
    for (uint32_t u = 0; u < sizeof(d) / 2; ++u) {
      const uint32_t e = tid + u * kBmmThreads;
      const uint32_t r = s.steps_near ? e / KD : e % R.value, k = s.steps_near ? e % KD : e / R.value;
      to[k * (R.value + 1) + r] = k0 + k < K ? (float)d[u] : 0.f;  // zero steps past the end leave the sums as they are
    }
  };
  const uint32_t i = lane & 15u, g = lane >> 4, wp = wave % (RP / 16) * 16u, wq = wave / (RP / 16) * 16u;
  f4 acc[1][1] = {{(f4){0.f, 0.f, 0.f, 0.f}}};
  load(Const<RP>(), p.P, pt, 0, vp);
  load(Const<RQ>(), p.Q, qt, 0, vq);
  for (uint32_t k0 = 0; k0 < K; k0 += KD) {
    if (k0) __syncthreads();
    store(Const<RP>(), p.P, k0, vp, ldsp);
    store(Const<RQ>(), p.Q, k0, vq, ldsq);
    __syncthreads();
    if (k0 + KD < K) {
      load(Const<RP>(), p.P, pt, k0 + KD, vp);
      load(Const<RQ>(), p.Q, qt, k0 + KD, vq);
    }
#pragma unroll
    for (uint32_t s = 0; s < KD / 4; ++s)
      acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(ldsp[(4 * s + g) * (RP + 1) + wp + i],
                                                       ldsq[(4 * s + g) * (RQ + 1) + wq + i], acc[0][0], 0, 0, 0);
  }
  using S = Stage<false, 32, 32, 1>;
  bmm_write<1, S, S>(p, bt, acc, pt * RP + wp + g * 4u, pt * RP, qt * RQ + wq, qt * RQ, lane);
}

template <bool SHORT, int W, bool PR, bool QR>
void launch_form(const BmmPlan& p, uint32_t grid, hipStream_t stream) {
  const bool odd = p.walk || p.P.ragged || p.Q.ragged;
  const dim3 g(grid), t(kBmmThreads);
  if constexpr (SHORT) {
    if (odd) hipLaunchKernelGGL((bmm_short_kernel<W, PR, QR, true>), g, t, 0, stream, p);
    else hipLaunchKernelGGL((bmm_short_kernel<W, PR, QR, false>), g, t, 0, stream, p);
  } else {
    if (odd) hipLaunchKernelGGL((bmm_kernel<bmm_depth(W), W, PR, QR, true>), g, t, 0, stream, p);
    else hipLaunchKernelGGL((bmm_kernel<bmm_depth(W), W, PR, QR, false>), g, t, 0, stream, p);
  }
}

template <bool SHORT, int W>
void launch_bmm(const BmmPlan& p, bool pr, bool qr, uint32_t grid, hipStream_t stream) {
  if (pr && qr) launch_form<SHORT, W, true, true>(p, grid, stream);
  else if (pr) launch_form<SHORT, W, true, false>(p, grid, stream);
  else if (qr) launch_form<SHORT, W, false, true>(p, grid, stream);
  else launch_form<SHORT, W, false, false>(p, grid, stream);
}

void launch_gather(const BmmPlan& p, uint32_t rp, uint32_t grid, hipStream_t stream) {
  if (rp == 64) hipLaunchKernelGGL((bmm_gather_kernel<64, 16>), dim3(grid), dim3(kBmmThreads), 0, stream, p);
  else if (rp == 16) hipLaunchKernelGGL((bmm_gather_kernel<16, 64>), dim3(grid), dim3(kBmmThreads), 0, stream, p);
  else hipLaunchKernelGGL((bmm_gather_kernel<32, 32>), dim3(grid), dim3(kBmmThreads), 0, stream, p);
}

// ---------------------------------------------------------------- chains on the VALU
// A chain of fmas per output, a lane to an output column, for products that
// leave the matrix tiles mostly empty (few rows of a, short reductions, many
// batch entries) or that only the gather could load: b's columns must run
// along k in aligned 16-byte vectors.  The dispatch holds both sides'
// measurements.
constexpr uint32_t kChainCols = 64;  // one output column per lane

struct ChainPlan {
  Mat a, b, y;  // a: [batch, m, k], b: [batch, k, n], y: [batch, m, n]
  uint32_t m, n, k;
  uint32_t mtiles, ntiles;
  bool a_kfast;  // stage a along k (its smaller stride is on k)
  // bytes from b.p to the end of its storage, vectors per contiguous run along
  // k (0 = one run) and the byte jump after a run
  uint32_t b_bytes, b_vrun, b_vjump;
  FastDiv div_mt, div_nt;  // block index -> (batch, row tile, column tile)
};

// Lane j owns output column j and streams that column from memory with 16-byte
// loads.  A block is one wave; it stages its RM rows of a in LDS as fp32
// (KS * 64 steps at a time) and each reduction step is RM fmas on LDS
// broadcasts.  The column is read in rounds of RV vectors (8 steps each): the
// first round is issued before the rows of a are staged, each later round
// loads while the previous one is consumed, and a whole round is consumed by
// straight-line code so that the LDS reads of one vector overlap the fmas of
// the previous one.  KS and RV are sized to K so that short reductions issue
// no surplus loads.
template <int RM, int KS, int RV>
__global__ __launch_bounds__(64) void chain_stream_kernel(ChainPlan p) {
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  constexpr uint32_t kDepth = KS * 64;  // steps of a staged per round (a multiple of 8 * RV)
  __shared__ __attribute__((aligned(16))) float As[RM][kDepth];
  const uint32_t lane = threadIdx.x;
  uint32_t t = blockIdx.x;
  const uint32_t q = p.div_nt.div(t), nt = t - q * p.ntiles;  // no integer division sequence
  const uint32_t bt = p.div_mt.div(q), mt = q - bt * p.mtiles;
  const uint32_t i0 = mt * RM, j = nt * kChainCols + lane;
  const _Float16* bcol = p.b.p + (int64_t)bt * p.b.batch +
                         p.b.col.at(min(j, p.n - 1) + p.b.col_origin + bt * p.b.col_group);
  const uint32_t rbase = p.b.row_origin + bt * p.b.row_group;
  // vector v of the column holds steps [8v, 8v + 8).  Loads go through a
  // buffer resource: the lane's column start is the vector offset, the step
  // offset is uniform (a scalar register) and advances by 16 bytes per vector
  // plus the run jump at each run end, so addressing costs a few scalar
  // operations per vector.  Loads past the last whole vector re-read it and
  // are not consumed.
  const uint32_t nvec = p.k / 8;
  const __amdgpu_buffer_rsrc_t brsrc = dev::buffer_rsrc(p.b.p, p.b_bytes);
  const uint32_t bvoff = (uint32_t)(bcol - p.b.p) * 2u;
  uint32_t bsoff = (uint32_t)p.b.row.at(rbase) * 2u;
  uint32_t rpos = p.b_vrun ? (rbase - p.b.row.blk.div(rbase) * p.b.row.blk.d) / 8u : 0u;
  uint32_t vaddr = 0;  // vector whose offset bsoff holds
  auto load_round = [&](h8 (&buf)[RV]) {
#pragma unroll
    for (int v = 0; v < RV; ++v) {
      buf[v] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(brsrc, bvoff, bsoff, 0));
      if (vaddr + 1 < nvec) {
        ++vaddr;
        bsoff += 16u;
        if (p.b_vrun && ++rpos == p.b_vrun) {
          rpos = 0;
          bsoff += p.b_vjump;
        }
      }
    }
  };
  h8 cur[RV], nxt[RV];
  if (nvec) load_round(cur);

  float acc[RM];
#pragma unroll
  for (int r = 0; r < RM; ++r) acc[r] = 0.f;
  typedef float f4 __attribute__((ext_vector_type(4)));
  // rows' steps kk..kk+7 of the staged a
  auto read_a = [&](f4 (&a)[RM][2], uint32_t kk) {
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      a[r][0] = *reinterpret_cast<const f4*>(&As[r][kk]);
      a[r][1] = *reinterpret_cast<const f4*>(&As[r][kk + 4]);
    }
  };
  auto fmas = [&](const f4 (&a)[RM][2], const h8& v) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float bv = (float)v[q];
#pragma unroll
      for (int r = 0; r < RM; ++r) acc[r] = __builtin_fmaf(a[r][q / 4][q % 4], bv, acc[r]);
    }
  };
  auto consume = [&](const h8& v, uint32_t kk) {
    f4 a[RM][2];
    read_a(a, kk);
    fmas(a, v);
  };
  uint32_t vnext = 0;  // first vector not yet consumed (a multiple of RV between rounds)
  for (uint32_t k0 = 0; k0 < p.k; k0 += kDepth) {
    const uint32_t kc = min(kDepth, p.k - k0);
    if (k0) __syncthreads();  // the previous round's rows are no longer read
    {
      // every load of the round in flight at once: clamped addresses, then
      // predicated LDS stores
      int64_t colpart[KS];
#pragma unroll
      for (int s = 0; s < KS; ++s)
        colpart[s] = p.a.col.at(k0 + min(lane + s * 64u, kc - 1) + p.a.col_origin + bt * p.a.col_group);
      _Float16 av[RM][KS];
#pragma unroll
      for (int r = 0; r < RM; ++r) {
        const _Float16* row = p.a.p + (int64_t)bt * p.a.batch +
                              p.a.row.at(min(i0 + r, p.m - 1) + p.a.row_origin + bt * p.a.row_group);
#pragma unroll
        for (int s = 0; s < KS; ++s) av[r][s] = row[colpart[s]];
      }
#pragma unroll
      for (int r = 0; r < RM; ++r)
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (lane + s * 64u < kc) As[r][lane + s * 64] = (float)av[r][s];
    }
    __syncthreads();
    const uint32_t vend = min(nvec, (k0 + kc) / 8);  // whole vectors inside this round
    // whole rounds: straight-line code
    while (vnext + RV <= vend) {
      const bool more = vnext + RV < nvec;
      if (more) load_round(nxt);
      // the a steps of vector v + 1 are read while vector v's fmas run
      f4 a0[RM][2], a1[RM][2];
      const uint32_t kb = vnext * 8 - k0;
      read_a(a0, kb);
#pragma unroll
      for (int v = 0; v < RV; v += 2) {
        read_a(a1, kb + (v + 1) * 8);
        fmas(a0, cur[v]);
        __builtin_amdgcn_sched_barrier(0);
        if (v + 2 < RV) read_a(a0, kb + (v + 2) * 8);
        fmas(a1, cur[v + 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) {
#pragma unroll
        for (int v = 0; v < RV; ++v) cur[v] = nxt[v];
      }
      vnext += RV;
    }
    // the last, partial round
    if (vnext < vend) {
#pragma unroll
      for (int v = 0; v < RV; ++v)
        if (vnext + v < vend) consume(cur[v], (vnext + v) * 8 - k0);
      vnext = vend;
    }
    // steps past the last whole vector
    for (uint32_t kk = max(k0, nvec * 8); kk < k0 + kc; ++kk) {
      const float bv = (float)bcol[p.b.row.at(rbase + kk)];
#pragma unroll
      for (int r = 0; r < RM; ++r) acc[r] = __builtin_fmaf(As[r][kk - k0], bv, acc[r]);
    }
  }
  if (j >= p.n) return;
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    const uint32_t i = i0 + r;
    if (i < p.m) p.y.p[p.y.at(bt, i, j)] = (_Float16)acc[r];
  }
}

// Columns of b at least a cache line apart (the probabilities of v p^T: each
// column is a row of p): a lane that streams its own column touches a
// different line per lane and instruction, which saturates the L1 tag lookups.
// Here a block of 4 waves computes 4 * RM rows x 64 columns and loads b in
// kTileDepth-step chunks with 8 lanes per column (one 128-byte line per 8
// lanes), keeps them in LDS as fp16 step pairs, and each lane reads its column
// two steps at a time.  The next chunk is loaded into registers while the
// current one is consumed.  K % 8 == 0.  A dependent fp32 fma takes about 32
// cycles, which bounds a chain however it is tiled.
constexpr uint32_t kTileDepth = 64;

template <int RM>
__global__ __launch_bounds__(kBmmThreads) void chain_tile_kernel(ChainPlan p) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h8 __attribute__((ext_vector_type(8)));
  constexpr uint32_t TM = 4 * RM;
  constexpr uint32_t kAPitch = TM + 4;
  constexpr uint32_t kBPitch = kChainCols + 1;  // in step pairs
  constexpr uint32_t kAPer = TM * kTileDepth / kBmmThreads;  // a elements per thread per chunk
  __shared__ __attribute__((aligned(16))) float As[kTileDepth][kAPitch];
  __shared__ h2 Bs[kTileDepth / 2][kBPitch];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  uint32_t t = blockIdx.x;
  const uint32_t nt = t % p.ntiles;
  t /= p.ntiles;
  const uint32_t mt = t % p.mtiles;
  const uint32_t bt = t / p.mtiles;
  const uint32_t i0 = mt * TM, j0 = nt * kChainCols;

  // b: thread handles vectors e = tid + 256 s: column jj = e / 8, steps
  // 8 * (e % 8) .. + 8 of the chunk
  const __amdgpu_buffer_rsrc_t brsrc = dev::buffer_rsrc(p.b.p, p.b_bytes);
  const uint32_t rbase = p.b.row_origin + bt * p.b.row_group;
  uint32_t bvoff[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const uint32_t jj = (tid + s * kBmmThreads) / 8u;
    bvoff[s] = (uint32_t)((int64_t)bt * p.b.batch +
                          p.b.col.at(min(j0 + jj, p.n - 1) + p.b.col_origin + bt * p.b.col_group)) * 2u;
  }
  const uint32_t kv = tid % 8u;
  h8 bv[2];
  _Float16 av[kAPer];
  auto load_chunk = [&](uint32_t k0, uint32_t kc) {
    // vectors past the chunk's end re-read its last vector (never consumed)
    const uint32_t kk = k0 + min(kv * 8u, kc - 8u);
    const uint32_t soff = (uint32_t)p.b.row.at(rbase + kk) * 2u;
#pragma unroll
    for (int s = 0; s < 2; ++s)
      bv[s] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(brsrc, bvoff[s] + soff, 0, 0));
#pragma unroll
    for (uint32_t s = 0; s < kAPer; ++s) {
      const uint32_t e = tid + s * kBmmThreads;
      const uint32_t kk2 = p.a_kfast ? e % kTileDepth : e / TM;
      const uint32_t ii = p.a_kfast ? e / kTileDepth : e % TM;
      av[s] = p.a.p[p.a.at(bt, min(i0 + ii, p.m - 1), k0 + min(kk2, kc - 1))];
    }
  };
  auto store_chunk = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t jj = (tid + s * kBmmThreads) / 8u;
#pragma unroll
      for (int q = 0; q < 4; ++q) Bs[kv * 4 + q][jj] = (h2){bv[s][2 * q], bv[s][2 * q + 1]};
    }
#pragma unroll
    for (uint32_t s = 0; s < kAPer; ++s) {
      const uint32_t e = tid + s * kBmmThreads;
      const uint32_t kk2 = p.a_kfast ? e % kTileDepth : e / TM;
      const uint32_t ii = p.a_kfast ? e / kTileDepth : e % TM;
      As[kk2][ii] = (float)av[s];
    }
  };

  float acc[RM];
#pragma unroll
  for (int r = 0; r < RM; ++r) acc[r] = 0.f;
  load_chunk(0, min(kTileDepth, p.k));
  for (uint32_t k0 = 0; k0 < p.k; k0 += kTileDepth) {
    const uint32_t kc = min(kTileDepth, p.k - k0);
    store_chunk();
    __syncthreads();
    if (k0 + kTileDepth < p.k) load_chunk(k0 + kTileDepth, min(kTileDepth, p.k - k0 - kTileDepth));
#pragma unroll 4
    for (uint32_t k2 = 0; k2 < kc / 2; ++k2) {
      const h2 b = Bs[k2][lane];
      const float b0 = (float)b[0], b1 = (float)b[1];
#pragma unroll
      for (int r = 0; r < RM; ++r) acc[r] = __builtin_fmaf(As[2 * k2][wave * RM + r], b0, acc[r]);
#pragma unroll
      for (int r = 0; r < RM; ++r) acc[r] = __builtin_fmaf(As[2 * k2 + 1][wave * RM + r], b1, acc[r]);
    }
    __syncthreads();
  }
  const uint32_t j = j0 + lane;
  if (j >= p.n) return;
#pragma unroll
  for (int r = 0; r < RM; ++r) {
    const uint32_t i = i0 + wave * RM + r;
    if (i < p.m) p.y.p[p.y.at(bt, i, j)] = (_Float16)acc[r];
  }
}

// ---------------------------------------------------------------- host

// b's columns run contiguously along k in 16-byte aligned groups of 8: unit
// step along k (a plain axis of stride 1, or a blocked axis of in-block stride
// 1 whose block is a multiple of 8 and whose block stride keeps 8-alignment),
// 8-aligned column, batch and group offsets, a 16-byte aligned base.
bool streamable_b(const Mat& b) {
  const Axis& k = b.row;
  const bool unit = (k.blk.d == 1 && k.outer == 1) || (k.blk.d % 8 == 0 && k.inner == 1 && k.outer % 8 == 0);
  const bool cols = b.col.outer % 8 == 0 && (b.col.blk.d == 1 || b.col.inner % 8 == 0);
  return unit && cols && reinterpret_cast<uintptr_t>(b.p) % 16 == 0 && b.batch % 8 == 0 && b.row_origin % 8 == 0 &&
         b.row_group % 8 == 0;
}

// Runs of `n` consecutive indexes from multiples of n are adjacent in memory:
// a plain axis of stride 1, or a blocked axis of in-block stride 1 whose
// blocks, origin and per-batch origin hold whole runs.
bool runs_of(const Axis& x, uint32_t origin, uint32_t group, uint32_t n) {
  if (x.blk.d == 1) return x.outer == 1;
  return x.inner == 1 && x.blk.d % n == 0 && origin % n == 0 && group % n == 0;
}

// Rows and columns of an operand before transposition (bmm_flow.cpp:280-281).
int64_t rows_of(const thin_desc* d) { return d->sizes[1] * (d->rank == 4 ? d->sizes[3] : 1); }

struct BmmShape {
  int64_t batch, m, k, n;
};

thin_status plan_shape(const thin_desc* a, const thin_desc* b, const thin_bmm_layout* L, BmmShape& s,
                       int64_t& a_rows, int64_t& b_rows) {
  THIN_REQUIRE(a && b && L && desc_valid(a) && desc_valid(b), THIN_ERR_INVALID, "bmm: invalid descriptor");
  THIN_REQUIRE(a->dtype == THIN_F16 && b->dtype == THIN_F16 && (a->rank == 3 || a->rank == 4) &&
                   (b->rank == 3 || b->rank == 4),
               THIN_ERR_INVALID, "bmm requires inference-only same-device FP16 rank-3 or channel-blocked rank-4 tensors");
  int64_t ar = rows_of(a), ac = a->sizes[2], br = rows_of(b), bc = b->sizes[2];
  THIN_REQUIRE(L->groups >= 0 && L->a_offset >= 0 && L->b_offset >= 0, THIN_ERR_INVALID, "invalid channel grouping");
  int64_t abatch = a->sizes[0], bbatch = b->sizes[0];
  for (int o = 0; o < 2; ++o) {
    const thin_desc* x = o ? b : a;
    int64_t& rows = o ? br : ar;
    int64_t& batches = o ? bbatch : abatch;
    if (L->groups && x->rank == 4) {
      THIN_REQUIRE(x->sizes[0] == 1 && rows % L->groups == 0, THIN_ERR_INVALID,
                   "grouped blocked operand requires N=1 and divisible channels");
      rows /= L->groups;
      batches = L->groups;
    }
  }
  const int64_t a_channels = L->a_channels < 0 ? ar - L->a_offset : L->a_channels;
  const int64_t b_channels = L->b_channels < 0 ? br - L->b_offset : L->b_channels;
  THIN_REQUIRE(a_channels > 0 && b_channels > 0 && L->a_offset + a_channels <= ar && L->b_offset + b_channels <= br,
               THIN_ERR_INVALID, "channel selection exceeds its group");
  a_rows = ar;
  b_rows = br;
  s.batch = abatch;
  s.m = L->transpose_a ? ac : a_channels;
  s.k = L->transpose_a ? a_channels : ac;
  const int64_t bk = L->transpose_b ? bc : b_channels;
  s.n = L->transpose_b ? b_channels : bc;
  THIN_REQUIRE(s.batch == bbatch && s.k == bk && s.batch > 0 && s.m > 0 && s.k > 0 && s.n > 0, THIN_ERR_INVALID,
               "bmm dimensions do not match or are empty");
  const int64_t np = (s.n + 15) / 16 * 16;
  THIN_REQUIRE(s.batch <= INT32_MAX && s.m <= INT32_MAX && s.k <= INT32_MAX && np <= INT32_MAX, THIN_ERR_INVALID,
               "bmm dimensions exceed kernel index range");
  THIN_REQUIRE(!L->blocked_output || (L->groups ? s.batch * s.m : s.m) % 16 == 0, THIN_ERR_INVALID,
               "blocked output requires C0-aligned channels");
  return THIN_OK;
}

Axis make_axis(int64_t blk, int64_t outer, int64_t inner) {
  Axis x;
  x.blk = FastDiv::make((uint32_t)blk);
  x.outer = outer;
  x.inner = inner;
  return x;
}

// Logical matrix of an input operand (bmm_flow.cpp:193-215): channels are the
// rows of a blocked operand, tokens its columns; groups split the channels of
// an N=1 blocked operand into heads; origin selects a channel range.
Mat make_input(const thin_desc* x, bool transpose, int64_t groups, int64_t origin) {
  Mat d;
  memset(&d, 0, sizeof d);
  d.p = static_cast<_Float16*>(x->data);
  d.batch = x->strides[0];
  const bool blocked = x->rank == 4;
  d.row = make_axis(blocked ? x->sizes[3] : 1, x->strides[1], blocked ? x->strides[3] : 0);
  d.col = make_axis(1, x->strides[2], 0);
  d.row_origin = (uint32_t)origin;
  if (groups > 0 && blocked) {
    d.batch = 0;
    d.row_group = (uint32_t)(x->sizes[1] * x->sizes[3] / groups);
  }
  if (transpose) {
    const Axis r = d.row;
    d.row = d.col;
    d.col = r;
    d.col_origin = d.row_origin;
    d.row_origin = 0;
    d.col_group = d.row_group;
    d.row_group = 0;
  }
  return d;
}

// Smallest element step along an axis (the in-block stride of a blocked axis).
int64_t unit_step(const Axis& x) { return x.blk.d > 1 ? x.inner : x.outer; }

thin_status check_out(const thin_desc* out, const BmmShape& s, const thin_bmm_layout* L) {
  THIN_REQUIRE(out && desc_valid(out) && out->dtype == THIN_F16, THIN_ERR_INVALID, "bmm: out must be float16");
  if (!L->blocked_output) {
    THIN_REQUIRE(out->rank == 3 && out->sizes[0] == s.batch && out->sizes[1] == s.m && out->sizes[2] == s.n,
                 THIN_ERR_INVALID, "bmm: out must be [%lld, %lld, %lld]", (long long)s.batch, (long long)s.m,
                 (long long)s.n);
  } else {
    const int64_t lead = L->groups ? 1 : s.batch, c1 = (L->groups ? s.batch * s.m : s.m) / 16;
    THIN_REQUIRE(out->rank == 4 && out->sizes[0] == lead && out->sizes[1] == c1 && out->sizes[2] == s.n &&
                     out->sizes[3] == 16,
                 THIN_ERR_INVALID, "bmm: blocked out must be [%lld, %lld, %lld, 16]", (long long)lead,
                 (long long)c1, (long long)s.n);
  }
  return THIN_OK;
}

template <int RM>
void launch_stream_rows(const ChainPlan& p, uint32_t grid, hipStream_t stream) {
  if (p.k <= 32)
    hipLaunchKernelGGL((chain_stream_kernel<RM, 1, 4>), dim3(grid), dim3(64), 0, stream, p);
  else if (p.k <= 64)
    hipLaunchKernelGGL((chain_stream_kernel<RM, 1, 8>), dim3(grid), dim3(64), 0, stream, p);
  else
    hipLaunchKernelGGL((chain_stream_kernel<RM, 8, 8>), dim3(grid), dim3(64), 0, stream, p);
}

void launch_stream(const ChainPlan& p, int rm, uint32_t grid, hipStream_t stream) {
  if (rm == 4) launch_stream_rows<4>(p, grid, stream);
  else if (rm == 2) launch_stream_rows<2>(p, grid, stream);
  else launch_stream_rows<1>(p, grid, stream);
}

void launch_tile(const ChainPlan& p, int rm, uint32_t grid, hipStream_t stream) {
  if (rm == 4) hipLaunchKernelGGL(chain_tile_kernel<4>, dim3(grid), dim3(kBmmThreads), 0, stream, p);
  else if (rm == 2) hipLaunchKernelGGL(chain_tile_kernel<2>, dim3(grid), dim3(kBmmThreads), 0, stream, p);
  else hipLaunchKernelGGL(chain_tile_kernel<1>, dim3(grid), dim3(kBmmThreads), 0, stream, p);
}

// Entries of the batch that one launch takes: a launch holds fewer than 2^32
// threads (it wraps beyond, without an error), and parts in multiples of 16
// begin at whole channel blocks of a grouped output.  0: not even 16 fit.
int64_t batch_part(int64_t batch, uint64_t blocks, uint32_t threads) {
  const int64_t most = (int64_t)(UINT32_MAX / threads / blocks);
  return most >= batch ? batch : most & ~(int64_t)15;
}

// The product as chains; a and b as in thin_layout_bmm, b streamable and of
// b_extent elements.
thin_status launch_chains(const Mat& a, const Mat& b, int64_t b_extent, const BmmShape& s, const thin_desc* out,
                          const thin_bmm_layout* L, hipStream_t stream) {
  ChainPlan p;
  memset(&p, 0, sizeof p);
  p.a = a;
  p.b = b;
  Mat& y = p.y;
  y.p = static_cast<_Float16*>(out->data);
  y.batch = L->blocked_output && L->groups ? 0 : out->strides[0];
  y.row = L->blocked_output ? make_axis(16, out->strides[1], out->strides[3]) : make_axis(1, out->strides[1], 0);
  y.col = make_axis(1, out->strides[2], 0);
  y.row_group = L->blocked_output && L->groups ? (uint32_t)s.m : 0u;  // head b's channels are packed from b * m on
  p.m = (uint32_t)s.m;
  p.n = (uint32_t)s.n;
  p.k = (uint32_t)s.k;
  p.a_kfast = unit_step(a.col) <= unit_step(a.row);
  p.ntiles = (uint32_t)((s.n + kChainCols - 1) / kChainCols);
  p.b_bytes = (uint32_t)(b_extent * 2);
  p.b_vrun = b.row.blk.d == 1 ? 0u : b.row.blk.d / 8u;
  p.b_vjump = b.row.blk.d == 1 ? 0u : (uint32_t)((b.row.outer - b.row.blk.d) * 2);
  const bool tile = p.k % 8 == 0 && b.col.blk.d == 1 && b.col.outer >= 64;
  const int unit = tile ? 4 : 1;  // rows of a block for RM = 1
  auto tiles = [&](int rm) { return (uint64_t)((s.m + unit * rm - 1) / (unit * rm)) * p.ntiles; };  // of one entry
  auto waves = [&](int rm) { return (uint64_t)s.batch * tiles(rm) * (uint64_t)unit; };
  // tile: the tallest that leaves every SIMD about a wave.  Stream: two rows a
  // wave; one when that leaves under half a wave per SIMD, four when it would
  // queue more than 8 waves per SIMD
  const int rm = tile ? (waves(4) >= 1024 ? 4 : waves(2) >= 1024 ? 2 : 1) : waves(2) < 512 ? 1 : waves(2) > 8192 ? 4 : 2;
  p.mtiles = (uint32_t)(tiles(rm) / p.ntiles);
  p.div_mt = FastDiv::make(p.mtiles);
  p.div_nt = FastDiv::make(p.ntiles);
  const int64_t part = batch_part(s.batch, tiles(rm), tile ? kBmmThreads : 64u);
  THIN_REQUIRE(part > 0, THIN_ERR_UNSUPPORTED, "bmm: too many output tiles");
  for (int64_t b0 = 0; b0 < s.batch; b0 += part) {
    const uint32_t grid = (uint32_t)(std::min(part, s.batch - b0) * (int64_t)tiles(rm));
    if (tile) launch_tile(p, rm, grid, stream);
    else launch_stream(p, rm, grid, stream);
    THIN_LAUNCH_CHECK("chain_kernel");
    for (Mat* x : {&p.a, &p.b, &p.y}) {
      x->p += part * x->batch;
      x->row_origin += (uint32_t)part * x->row_group;
      x->col_origin += (uint32_t)part * x->col_group;
    }
    p.b_bytes -= (uint32_t)(part * b.batch * 2);
  }
  return THIN_OK;
}

}  // namespace
}  // namespace thin

using namespace thin;

extern "C" thin_status thin_layout_bmm_shape(const thin_desc* a, const thin_desc* b, const thin_bmm_layout* layout,
                                             int32_t* out_rank, int64_t* out_sizes) {
  clear_error();
  BmmShape s;
  int64_t ar, br;
  thin_status st = plan_shape(a, b, layout, s, ar, br);
  if (st != THIN_OK) return st;
  THIN_REQUIRE(out_rank && out_sizes, THIN_ERR_INVALID, "bmm: null output shape pointer");
  if (!layout->blocked_output) {
    *out_rank = 3;
    out_sizes[0] = s.batch;
    out_sizes[1] = s.m;
    out_sizes[2] = s.n;
  } else {
    *out_rank = 4;
    out_sizes[0] = layout->groups ? 1 : s.batch;
    out_sizes[1] = (layout->groups ? s.batch * s.m : s.m) / 16;
    out_sizes[2] = s.n;
    out_sizes[3] = 16;
  }
  return THIN_OK;
}

extern "C" thin_status thin_layout_bmm(const thin_desc* a, const thin_desc* b, const thin_bmm_layout* layout,
                                       const thin_desc* out, hipStream_t stream) {
  clear_error();
  BmmShape s;
  int64_t ar, br;
  thin_status st = plan_shape(a, b, layout, s, ar, br);
  if (st != THIN_OK) return st;
  st = check_out(out, s, layout);
  if (st != THIN_OK) return st;
  // every logical index the kernel forms (origin + group offset + index)
  // stays below the operand's own row / column count
  for (const thin_desc* x : {a, b, out})
    THIN_REQUIRE(x->sizes[1] * (x->rank == 4 ? x->sizes[3] : 1) < ((int64_t)1 << 31) &&
                     x->sizes[2] < ((int64_t)1 << 31),
                 THIN_ERR_UNSUPPORTED, "bmm: operand dimensions exceed the kernel index range");

  const Mat am = make_input(a, layout->transpose_a, layout->groups, layout->a_offset);
  const Mat bm = make_input(b, layout->transpose_b, layout->groups, layout->b_offset);
  // k is the column axis of a and the row axis of b
  Side sa, sb;
  memset(&sa, 0, sizeof sa);
  memset(&sb, 0, sizeof sb);
  sa.p = am.p;
  sa.batch = am.batch;
  sa.row = am.row;
  sa.step = am.col;
  sa.row_origin = am.row_origin;
  sa.row_group = am.row_group;
  sa.step_origin = am.col_origin;
  sa.step_group = am.col_group;
  sa.rows = (uint32_t)s.m;
  sb.p = bm.p;
  sb.batch = bm.batch;
  sb.row = bm.col;
  sb.step = bm.row;
  sb.row_origin = bm.col_origin;
  sb.row_group = bm.col_group;
  sb.step_origin = bm.row_origin;
  sb.step_group = bm.row_group;
  sb.rows = (uint32_t)s.n;

  BmmPlan p;
  memset(&p, 0, sizeof p);
  p.y = static_cast<_Float16*>(out->data);
  p.k = (uint32_t)s.k;
  const Axis cols = make_axis(1, out->strides[2], 0);
  if (!layout->blocked_output) {
    // rows of n outputs: p is b's columns
    p.P = sb;
    p.Q = sa;
    p.ybatch = out->strides[0];
    p.yp = cols;
    p.yq = make_axis(1, out->strides[1], 0);
  } else {
    // channel r of batch b is packed channel b * m + r of [lead, C1, n, 16]
    // (grouped), or channel r of image b (ungrouped; the two agree when the
    // ungrouped tensor is contiguous); p is the channels
    p.P = sa;
    p.Q = sb;
    p.yp = make_axis(16, out->strides[1], out->strides[3]);
    p.yq = cols;
    if (layout->groups) p.yp_group = (uint32_t)s.m;
    else p.ybatch = out->strides[0];
  }
  // 64 x 64 blocks (four matrix products per operand pair read) where they
  // give every compute unit two, else 32 x 32 ones, which spread the work
  // over four times as many waves
  auto blocks = [&](uint64_t r) { return (uint64_t)s.batch * ((p.P.rows + r - 1) / r) * ((p.Q.rows + r - 1) / r); };
  uint32_t w = blocks(64) >= 512 ? 2 : 1;
  // 16-byte runs along the steps, else along the rows; the kernels' lane
  // offsets are 32-bit
  auto steps_runs = [&](const Side& x) { return s.k >= 8 && runs_of(x.step, x.step_origin, x.step_group, 8); };
  auto rows_runs = [&](const Side& x) {
    return runs_of(x.row, x.row_origin, x.row_group, 8) && (x.row.blk.d != 1 || x.rows >= 8);
  };
  auto near = [](const thin_desc* d) {
    int64_t extent = 0;
    for (int i = 1; i < d->rank; ++i) extent += (d->sizes[i] - 1) * d->strides[i];
    return extent < ((int64_t)1 << 30);
  };
  const bool fast =
      (steps_runs(p.P) || rows_runs(p.P)) && (steps_runs(p.Q) || rows_runs(p.Q)) && near(a) && near(b);
  // Where b's columns come in aligned vectors, the chains on the VALU take what
  // only the gather could load (v p^T of 32 channels in blocks of 4, 1600
  // tokens: 25 us against 49) and products that leave the matrix tiles empty:
  // - short reductions with few rows ([8000,2,8] x [8000,8,4]: 5.9 us against
  //   20) or few tiles ([16,32,8] x [16,8,96]: 3.0 against 3.5; the two meet
  //   at about 128 tiles);
  // - up to 16 rows, half a tile, in enough blocks that throughput counts
  //   ([1500,16,64] x [1500,64,48]: 1.4x; [256,16,64] x [256,64,48], 512
  //   blocks: 0.9x), longer reductions only where columns leave tiles partly
  //   empty too ([1500,16,136]: n = 32 0.92x, n = 48 1.2x).
  // From 24 rows on the matrix tiles are faster or as fast (at worst
  // [256,40,64] x [256,64,64], 7.1 us against 6.5).
  const uint64_t tiles = blocks(32);
  auto sparse = [&] {
    if (s.k <= 32) return s.m <= 8 || tiles < 128;
    return s.m <= 16 && tiles >= 640 && (s.k <= 64 || (s.n > 32 && s.k <= 512));
  };
  int64_t b_extent = 1;  // elements from b's data pointer to its last element, + 1
  for (int d = 0; d < b->rank; ++d) b_extent += (b->sizes[d] - 1) * b->strides[d];
  if (streamable_b(bm) && b_extent * 2 < ((int64_t)1 << 31) && (!fast || sparse()))
    return launch_chains(am, bm, b_extent, s, out, layout, stream);
  if (!fast) w = 1;
  const bool one = s.k <= 32;  // one chunk of steps
  const uint32_t r = 32 * w, kd = (uint32_t)bmm_depth((int)w);
  const bool pr = !steps_runs(p.P), qr = !steps_runs(p.Q);
  for (Side* x : {&p.P, &p.Q}) {  // (of operands with K >= 8 steps, or with 8 or more rows, in runs)
    x->last_run = x->step.blk.d == 1 ? (uint32_t)s.k - 8u : ((uint32_t)s.k - 1u) & ~7u;
    x->last_rows = x->row.blk.d == 1 ? x->rows - 8u : (x->rows - 1u) & ~7u;
    const uint32_t part = x->row.blk.d == 1 ? x->rows & 7u : 0u;
    if (x->rows > r) x->early = part ? 8u - part : 0u;
    else x->ragged = x == &p.P ? (pr ? part : 0u) : (qr ? part : 0u);
  }
  p.P.steps_near = unit_step(p.P.step) <= unit_step(p.P.row);
  p.Q.steps_near = unit_step(p.Q.step) <= unit_step(p.Q.row);
  const uint32_t rp = fast ? r : p.Q.rows <= 16 ? 64 : p.P.rows <= 16 ? 16 : 32, rq = fast ? r : 1024 / rp;
  p.ptiles = (p.P.rows + rp - 1) / rp;
  p.qtiles = FastDiv::make((p.Q.rows + rq - 1) / rq);
  p.y_vec = runs_of(p.yp, 0, p.yp_group, 4 * w) ? 1u : 0u;
  p.span = 1;
  if (fast && one) {
    // as many P tiles a block as leave a block or two a compute unit, in even
    // shares: a wave's fixed work is then spread over more products (q^T k
    // [128,400,32] x [128,32,400] 23.8 us with all seven tiles a block, 25.1
    // with two; [4,1600,32] x [4,32,1600] 12.2 us with five, 13.2 with three,
    // 13.5 with one)
    const uint64_t share = blocks(r) / 400;
    const uint32_t most = share < 1 ? 1u : share > 8 ? 8u : (uint32_t)share;
    const uint32_t parts = (p.ptiles + most - 1) / most;
    p.span = (p.ptiles + parts - 1) / parts;
    p.walk = r % p.P.row.blk.d != 0;
    p.P.hop = (int64_t)(r / p.P.row.blk.d) * p.P.row.outer * 2;
    p.yhop = (int64_t)(r / p.yp.blk.d) * p.yp.outer;
  } else if (fast) {
    p.walk = kd % p.P.step.blk.d != 0 || kd % p.Q.step.blk.d != 0;
    p.P.hop = (int64_t)(kd / p.P.step.blk.d) * p.P.step.outer * 2;
    p.Q.hop = (int64_t)(kd / p.Q.step.blk.d) * p.Q.step.outer * 2;
  }
  p.pblocks = FastDiv::make((p.ptiles + p.span - 1) / p.span);
  const uint64_t per = (uint64_t)p.qtiles.d * p.pblocks.d;  // blocks of an entry
  const int64_t part = batch_part(s.batch, per, kBmmThreads);
  THIN_REQUIRE(part > 0, THIN_ERR_UNSUPPORTED, "bmm: too many output tiles");
  for (int64_t b0 = 0; b0 < s.batch; b0 += part) {
    const uint32_t grid = (uint32_t)(std::min(part, s.batch - b0) * (int64_t)per);
    if (!fast) launch_gather(p, rp, grid, stream);
    else if (one && w == 2) launch_bmm<true, 2>(p, pr, qr, grid, stream);
    else if (one) launch_bmm<true, 1>(p, pr, qr, grid, stream);
    else if (w == 2) launch_bmm<false, 2>(p, pr, qr, grid, stream);
    else launch_bmm<false, 1>(p, pr, qr, grid, stream);
    THIN_LAUNCH_CHECK("bmm_kernel");
    for (Side* x : {&p.P, &p.Q}) {
      x->p += part * x->batch;
      x->row_origin += (uint32_t)part * x->row_group;
      x->step_origin += (uint32_t)part * x->step_group;
    }
    p.y += part * p.ybatch;
    if (p.yp_group && b0 + part < s.batch) p.y += p.yp.at((uint32_t)part * p.yp_group);
  }
  return THIN_OK;
}

// ---------------------------------------------------------------- channel select

namespace thin {
namespace {

// out channel c of [1, C1o, T, 16] = x channel (c / count) * group + begin +
// c % count of [1, C1, T, 16] (bmm_flow.cpp:217-251); one thread per output
// element.
struct SelectPlan {
  const _Float16* x;
  _Float16* y;
  int64_t xs1, xs2, xs3, ys1, ys2, ys3;
  FastDiv tokens, count;
  uint32_t group, begin;
  uint64_t total;  // C1o * T * 16
};

__global__ __launch_bounds__(256) void channel_select_kernel(SelectPlan p) {
  // the plan in registers before the loop's bounds test: one round of scalar
  // loads (one asm statement: each is a scheduling boundary)
  __asm__ volatile("" ::"s"(p.x), "s"(p.y), "s"(p.xs1), "s"(p.xs2), "s"(p.xs3), "s"(p.ys1), "s"(p.ys2), "s"(p.ys3),
                   "s"(p.tokens.d), "s"(p.tokens.mul), "s"(p.tokens.shr), "s"(p.count.d), "s"(p.count.mul),
                   "s"(p.count.shr), "s"(p.group), "s"(p.begin), "s"(p.total));
  for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < p.total; e += (uint64_t)gridDim.x * 256) {
    const uint32_t lane = (uint32_t)(e & 15u);
    const uint32_t rest = (uint32_t)(e >> 4);  // cb * T + t
    const uint32_t cb = p.tokens.div(rest), t = rest - cb * p.tokens.d;
    const uint32_t c = cb * 16u + lane;
    const uint32_t g = p.count.div(c);
    const uint32_t sc = g * p.group + p.begin + (c - g * p.count.d);
    const _Float16 v = p.x[(int64_t)(sc >> 4) * p.xs1 + (int64_t)t * p.xs2 + (int64_t)(sc & 15u) * p.xs3];
    p.y[(int64_t)cb * p.ys1 + (int64_t)t * p.ys2 + (int64_t)lane * p.ys3] = v;
  }
}

thin_status select_shape(const thin_desc* x, int64_t groups, int64_t begin, int64_t count, int64_t* sizes) {
  THIN_REQUIRE(x && desc_valid(x) && x->dtype == THIN_F16 && x->rank == 4 && x->sizes[0] == 1 && x->sizes[3] == 16,
               THIN_ERR_INVALID, "channel_select expects aligned N=1 FP16 blocked input");
  const int64_t channels = x->sizes[1] * 16;
  THIN_REQUIRE(groups > 0 && channels % groups == 0 && begin >= 0 && count > 0 && begin + count <= channels / groups &&
                   groups * count % 16 == 0,
               THIN_ERR_INVALID, "channel_select requires valid equal groups and C0-aligned total output channels");
  sizes[0] = 1;
  sizes[1] = groups * count / 16;
  sizes[2] = x->sizes[2];
  sizes[3] = 16;
  return THIN_OK;
}

}  // namespace
}  // namespace thin

extern "C" thin_status thin_channel_select_shape(const thin_desc* x, int64_t groups, int64_t begin, int64_t count,
                                                 int64_t* out_sizes) {
  clear_error();
  THIN_REQUIRE(out_sizes, THIN_ERR_INVALID, "channel_select: null output shape pointer");
  return select_shape(x, groups, begin, count, out_sizes);
}

extern "C" thin_status thin_channel_select(const thin_desc* x, int64_t groups, int64_t begin, int64_t count,
                                           const thin_desc* out, hipStream_t stream) {
  clear_error();
  int64_t sizes[4];
  thin_status st = select_shape(x, groups, begin, count, sizes);
  if (st != THIN_OK) return st;
  THIN_REQUIRE(out && desc_valid(out) && out->dtype == THIN_F16 && out->rank == 4 && out->sizes[0] == 1 &&
                   out->sizes[1] == sizes[1] && out->sizes[2] == sizes[2] && out->sizes[3] == 16,
               THIN_ERR_INVALID, "channel_select: out must be [1, %lld, %lld, 16] float16", (long long)sizes[1],
               (long long)sizes[2]);
  THIN_REQUIRE(x->sizes[1] * 16 < ((int64_t)1 << 31) && x->sizes[2] < ((int64_t)1 << 31) &&
                   sizes[1] * sizes[2] < ((int64_t)1 << 27),
               THIN_ERR_UNSUPPORTED, "channel_select: tensor too large");
  SelectPlan p;
  memset(&p, 0, sizeof p);
  p.x = static_cast<const _Float16*>(x->data);
  p.y = static_cast<_Float16*>(out->data);
  p.xs1 = x->strides[1];
  p.xs2 = x->strides[2];
  p.xs3 = x->strides[3];
  p.ys1 = out->strides[1];
  p.ys2 = out->strides[2];
  p.ys3 = out->strides[3];
  p.tokens = FastDiv::make((uint32_t)sizes[2]);
  p.count = FastDiv::make((uint32_t)count);
  p.group = (uint32_t)(x->sizes[1] * 16 / groups);
  p.begin = (uint32_t)begin;
  p.total = (uint64_t)sizes[1] * (uint64_t)sizes[2] * 16u;
  if (p.total == 0) return THIN_OK;
  hipLaunchKernelGGL(channel_select_kernel, dim3(grid_for(p.total, 256)), dim3(256), 0, stream, p);
  THIN_LAUNCH_CHECK("channel_select_kernel");
  return THIN_OK;
}
