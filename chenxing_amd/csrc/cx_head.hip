// cx_head.hip -- the LM-head projection with the greedy draw fused, for
// gfx950 (reference chenxing/model/transformer.py:102-104, the last
// hidden state times out_w.T, then chenxing/core/sampler.py:114-115, the
// argmax of the row): the [B, V] logits are never written to HBM.
//
// logits[b, v] = sum_k hidden[b, k] * W[v, k], with bf16 hidden states and
// head weights (row-major [B, D] and [V, D]) and fp32 accumulation on
// MFMA (v_mfma_f32_16x16x32_bf16: A = 16 vocab rows x 32 k, B = 32 k x 16
// batch rows, C = 16 x 16 fp32).  Two stream-ordered launches:
//
//   1. head_wide or  one workgroup per (vocab tile, batch tile of up to 256
//      head_tall    rows): the projection, reduced in registers and LDS to
//                   one 64-bit key per (vocab tile, batch row): the orderable
//                   logit above the complement of the vocab id, so the
//                   largest key is the largest logit with the lowest id on
//                   ties, and a NaN logit (key above +inf) the first NaN --
//                   numpy's argmax.
//   2. head_merge   one workgroup per batch row: the largest of its keys.
//
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>

#include "cx_device.hpp"
#include "cx_internal.hpp"
#include "cx_sampler.h"
#include "cx_timing.hpp"

namespace cx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int HEAD_WG = 256;                 // merge workgroup
constexpr int HEAD_KB = 128;                 // D is a multiple of this

struct HeadArgs {
  const uint16_t* hidden;   // [B, ldh] bf16 bits
  const uint16_t* weight;   // [V, ldw] bf16 bits
  int64_t ldh, ldw;
  int B, D, V;
  uint64_t* part;           // [B, nvt] keys
  int nvt;                  // vocab tiles
  int32_t* out_id;
  float* out_max;           // nullable [B]
  float* out_logits;        // nullable [B, V] (verification)
};

// 16 bytes of head weights: a plain load (the non-temporal form measured
// 0.5 us slower over the 1 GB at B=16)
__device__ __forceinline__ u32x4 ld16(const uint16_t* p) {
  return *(const u32x4*)p;
}

// The 64-bit argmax key of logit x at vocab id v.
__device__ __forceinline__ uint64_t head_key(float x, int v) {
  const uint32_t k = x != x ? 0xFFFFFFFFu : f2key(x);
  return ((uint64_t)k << 32) | (uint32_t)~(uint32_t)v;
}

// A workgroup's keys: lane (g, c) of a wave holds the logits of vocab rows
// v0 + 16 m + 4 g + j (j < 4) at batch rows b0 + 16 n + c.
template <int NT, int MT, int NW>
__device__ __forceinline__ void head_keys(const HeadArgs& A, const f32x4 (&acc)[MT][NT], int v0,
                                          int b0, int vt, uint64_t (&s_key)[NW][16 * NT]) {
  const int w = wave_id(), l = lane_id();
  const int g = l >> 4, c = l & 15;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int b = b0 + 16 * n + c;
    uint64_t key = 0;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int v = v0 + 16 * m + 4 * g + j;
        const float x = acc[m][n][j];
        if (v < A.V) {
          const uint64_t k = head_key(x, v);
          key = k > key ? k : key;
          if (A.out_logits && b < A.B) A.out_logits[(size_t)b * A.V + v] = x;
        }
      }
    uint64_t o = __shfl_xor(key, 16);
    key = o > key ? o : key;
    o = __shfl_xor(key, 32);
    key = o > key ? o : key;
    if (g == 0) s_key[w][16 * n + c] = key;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < 16 * NT && b0 + t < A.B; t += NW * 64) {
    uint64_t key = s_key[0][t];
#pragma unroll
    for (int k = 1; k < NW; ++k) key = s_key[k][t] > key ? s_key[k][t] : key;
    A.part[(size_t)(b0 + t) * A.nvt + vt] = key;
  }
}

// A wave owns 16 MT vocab rows and all the workgroup's 16 NT batch rows, so
// every weight element is loaded by one lane, straight into registers, and
// the weights are read once for up to 256 batch rows; the hidden states (2 MB
// at B = 256, D = 4096: the L2 holds them) pass through LDS in stages of 64 k.
//
//  * Bound: HBM (1.05 GB of weights at V = 128256, D = 4096: 146 us at the
//    rate a large read reaches here) up to B = 256, where the MFMA time
//    is 108 us at the dense peak.
//  * Both operands are requested WIDE_AHEAD stages before they are used: the
//    weights into a register ring, the hidden states by loads that write LDS
//    directly (no registers held, and in issue order with the weights, so
//    waiting for a stage's hidden states leaves the later stages' weights in
//    flight; staged through registers, that wait drains the weight ring).
//    One barrier per stage: after it every wave's share of the stage is in
//    LDS, and every wave is done with the stage before, whose buffer the
//    next request then overwrites.
//  * LDS layout: a stage row is 64 k = 8 chunks of 16 bytes; chunk c of row r
//    is at position c ^ (r & 7), so the 8 rows an operand read touches at a
//    time fall in different banks.  The permutation is in the global address
//    each lane loads from (a direct-to-LDS load writes lane order).
//  * Order of k (NSEG = 4): with rows a multiple of 4096 bytes apart, every
//    workgroup that walks k from 0 asks the same few memory channels at a
//    time.  The workgroups therefore start at different quarters of k and
//    wrap around.  Each quarter has its own accumulators and the four sums
//    are added in one fixed order, so a weight row gives the same logit
//    wherever it lies (equal rows still tie); batches of more than 64 rows,
//    and other pitches, add one sum in k order.  Measured at V = 128256,
//    D = 4096: B = 32 213 -> 189 us, B = 64 228 -> 195 us (with rows padded
//    by 128 bytes: 184 and 195 us); two starts instead of four give nothing,
//    and for larger batches four sets of accumulators do not fit.
//  * Measured (a call, without a profiler), B = 256, V = 128256, D = 4096: 292
//    to 297 us, 905 to 921 TFLOP/s (1416 us with 32 batch rows per pass over
//    the weights); 24 dispatches back to back under the profiler 282 to 395
//    us, the middle ones longest.  B = 128 241 us (was 704 us);
//    B = 16, V = 32000 50 us (131 us with 512 vocab rows a workgroup, which
//    left 193 of the 256 CUs without one).
constexpr int WIDE_SK = 64;                  // k per stage
constexpr int WIDE_AHEAD = 3;                // stages requested ahead
constexpr int WIDE_RING = WIDE_AHEAD + 1;    // stage buffers

template <int MT>
struct WideStage {
  u32x4 w[MT][2];                            // 16 rows x 32 k per operand
};

// s_waitcnt vmcnt(n) alone (gfx9 encoding: vmcnt in bits 3:0 and 15:14;
// expcnt and lgkmcnt at their "no wait" values).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

template <int NT, int MT, int NW, int NSEG>
__global__ __launch_bounds__(NW * 64, 1) void head_wide(HeadArgs A) {
  constexpr int ROWS = 16 * NT;
  constexpr int NH = 2 * NT / NW;            // direct-to-LDS loads a wave issues per stage
  static_assert(2 * NT % NW == 0, "a stage's rows divide over the waves");
  // one array per stage buffer: the compiler then knows that a read of one
  // does not wait for the loads that write another
  __shared__ __align__(16) uint16_t s_h0[ROWS * WIDE_SK];
  __shared__ __align__(16) uint16_t s_h1[ROWS * WIDE_SK];
  __shared__ __align__(16) uint16_t s_h2[ROWS * WIDE_SK];
  __shared__ __align__(16) uint16_t s_h3[ROWS * WIDE_SK];
  __shared__ uint64_t s_key[NW][ROWS];
  const int w = wave_id(), l = lane_id();
  const int g = l >> 4, c = l & 15;
  const int nby = (A.B + ROWS - 1) / ROWS;
  // batch tiles of one vocab tile are neighbours in the dispatch order, so
  // they find the weights in the Infinity Cache
  const int vt = blockIdx.x / nby;
  const int b0 = (int)(blockIdx.x - (unsigned)vt * nby) * ROWS;
  const int v0 = (vt * NW + w) * 16 * MT;
  const int S = A.D / WIDE_SK;
  const uint16_t* wp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
    wp[m] = A.weight + (size_t)min(v0 + 16 * m + c, A.V - 1) * A.ldw + 8 * g;
  // direct-to-LDS load j of this wave: rows (j NW + w) 8 .. + 7
  const uint16_t* hp[NH];
#pragma unroll
  for (int j = 0; j < NH; ++j) {
    const int r = (j * NW + w) * 8 + (l >> 3);
    hp[j] = A.hidden + (size_t)min(b0 + r, A.B - 1) * A.ldh + 8 * ((l & 7) ^ (l >> 3));
  }
  // this workgroup's first segment; neighbours in time and on an XCD differ
  const int phase = __builtin_amdgcn_readfirstlane((vt + (vt >> 3)) % NSEG);
  const int rot = phase * (S / NSEG);
  f32x4 acc[NSEG][MT][NT];
#pragma unroll
  for (int j = 0; j < NSEG; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[j][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  WideStage<MT> ring[WIDE_RING];

  // Request the s-th stage in this workgroup's order (clamped to the last
  // one, so every turn of the loop issues the same number of loads and its
  // counted waits hold to its end).  The hidden states come first: a wait
  // that leaves the later stages' loads outstanding covers them whatever the
  // compiler does with the weights, whose own uses wait for them.
  auto request = [&](int s, uint16_t* buf, WideStage<MT>& x) {
    int ks = min(s, S - 1) + rot;
    if (NSEG > 1 && ks >= S) ks -= S;
    const int k = ks * WIDE_SK;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NH; ++j)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(hp[j] + k),
                                       to_lds(buf + (j * NW + w) * 8 * WIDE_SK), 16, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < 2; ++t) x.w[m][t] = ld16(wp[m] + k + 32 * t);
    __builtin_amdgcn_sched_barrier(0);
  };
  // this lane's operand chunk in a stage buffer: row c of tile 0, slice 0
  const int lofs = c * WIDE_SK + 8 * (g ^ (c & 7));
  auto multiply = [&](const uint16_t* buf, const WideStage<MT>& x, f32x4 (&acc)[MT][NT]) {
    // four operand reads ahead of their MFMAs, kept in that order (two reads
    // and a wait, as the scheduler places them: 303 instead of 291 us at
    // B = 256, V = 128256, D = 4096)
    constexpr int OPS = 2 * NT, AHEAD = 4;
    auto operand = [&](int i) {
      return *(const CX_LDS u32x4*)(to_lds((uint16_t*)buf) + (lofs ^ (32 * (i / NT))) +
                                    (i % NT) * 16 * WIDE_SK);
    };
    u32x4 h[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) h[i] = operand(i);
#pragma unroll
    for (int i = 0; i < OPS; ++i) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        acc[m][i % NT] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8, x.w[m][i / NT]), __builtin_bit_cast(bf16x8, h[i % AHEAD]),
            acc[m][i % NT], 0, 0, 0);
      if (i + AHEAD < OPS) h[i % AHEAD] = operand(i + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Stage s has arrived once at most the later stages' loads are outstanding.
  auto step = [&](int s, uint16_t* cur, const WideStage<MT>& x, uint16_t* nxt, WideStage<MT>& y,
                  f32x4 (&acc)[MT][NT]) {
    wait_vm<(WIDE_AHEAD - 1) * (NH + 2 * MT)>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    request(s + WIDE_AHEAD, nxt, y);
    multiply(cur, x, acc);
    asm volatile("" ::: "memory");
  };

  request(0, s_h0, ring[0]);
  request(1, s_h1, ring[1]);
  request(2, s_h2, ring[2]);
  int s = 0;
#pragma unroll
  for (int j = 0; j < NSEG; ++j) {
    const int end = NSEG == 1 ? S : (j + 1) * (S / NSEG);
    for (; s + WIDE_RING <= end; s += WIDE_RING) {
      step(s, s_h0, ring[0], s_h3, ring[3], acc[j]);
      step(s + 1, s_h1, ring[1], s_h0, ring[0], acc[j]);
      step(s + 2, s_h2, ring[2], s_h1, ring[1], acc[j]);
      step(s + 3, s_h3, ring[3], s_h2, ring[2], acc[j]);
    }
  }
  wait_vm<0>();                              // the last requests write LDS: end them first
  if (NSEG == 1 && s < S) {                  // S is even: two stages left, both requested
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(s_h0, ring[0], acc[0]);
    multiply(s_h1, ring[1], acc[0]);
  }
  // the segments' sums, added in the order of k whatever order they came in
  // (acc[j] is segment (phase + j) % NSEG)
  if (NSEG > 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int p = 0; p < NSEG; ++p)
          if (phase == p)
            sum = (acc[(NSEG - p) % NSEG][m][n] + acc[(NSEG - p + 1) % NSEG][m][n]) +
                  (acc[(NSEG - p + 2) % NSEG][m][n] + acc[(NSEG - p + 3) % NSEG][m][n]);
        acc[0][m][n] = sum;
      }
  }
  head_keys<NT, MT, NW>(A, acc[0], v0, b0, vt, s_key);
}

// Batches of up to 32 rows over a vocabulary whose tiles of 512 rows nearly
// fill the CUs once (head_plan): one workgroup of 16 waves per tile, each
// wave with 32 vocab rows.  The hidden states are staged in LDS a chunk of k
// at a time (4736 k for 16 batch rows, 2304 for 32), so a wave runs its k loop
// without barriers, its weights through a register ring of DEPTH blocks of
// 128 k.  head_wide spends a barrier per 64 k and starts 2004 workgroups at
// V = 128256, which shows where k is short or its walk starts at 0 everywhere:
// B = 32, D = 512 36 against 31 us, D = 1536 85 against 75 us.
constexpr int TALL_NW = 16, TALL_MT = 2;
constexpr int TALL_VT = TALL_NW * TALL_MT * 16;
constexpr int TALL_LDS = 152 * 1024;         // the staged chunk at most
template <int NB>
constexpr int tall_chunk() { return (TALL_LDS / (16 * NB * 2) - 8) / HEAD_KB * HEAD_KB; }

template <int NB, int DEPTH>
__global__ __launch_bounds__(TALL_NW * 64) void head_tall(HeadArgs A) {
  extern __shared__ __align__(16) unsigned char head_lds[];
  __shared__ uint64_t s_key[TALL_NW][16 * NB];
  const int l = lane_id(), g = l >> 4, c = l & 15;
  const int v0 = (int)blockIdx.x * TALL_VT + wave_id() * TALL_MT * 16;
  const int KC = min(A.D, tall_chunk<NB>());
  const int stride = KC + 8;                 // padded: the 16 rows of an operand in different banks
  CX_LDS uint16_t* const hs = to_lds((uint16_t*)head_lds);
  const CX_LDS uint16_t* const hl = hs + c * stride + 8 * g;
  const uint16_t* wp[TALL_MT];
#pragma unroll
  for (int m = 0; m < TALL_MT; ++m)
    wp[m] = A.weight + (size_t)min(v0 + 16 * m + c, A.V - 1) * A.ldw + 8 * g;
  f32x4 acc[TALL_MT][NB];
#pragma unroll
  for (int m = 0; m < TALL_MT; ++m)
#pragma unroll
    for (int n = 0; n < NB; ++n) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 ring[DEPTH][TALL_MT][4];
  auto load = [&](u32x4 (&x)[TALL_MT][4], int k) {
#pragma unroll
    for (int m = 0; m < TALL_MT; ++m)
#pragma unroll
      for (int s = 0; s < 4; ++s) x[m][s] = ld16(wp[m] + k + 32 * s);
  };
  auto multiply = [&](const u32x4 (&x)[TALL_MT][4], int k) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4 h[NB];
#pragma unroll
      for (int n = 0; n < NB; ++n)
        h[n] = *(const CX_LDS u32x4*)(hl + 16 * n * stride + k + 32 * s);
#pragma unroll
      for (int m = 0; m < TALL_MT; ++m)
#pragma unroll
        for (int n = 0; n < NB; ++n)
          acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8, x[m][s]), __builtin_bit_cast(bf16x8, h[n]), acc[m][n],
              0, 0, 0);
    }
  };
  for (int k0 = 0; k0 < A.D; k0 += KC) {
    const int kn = min(KC, A.D - k0);
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (d * HEAD_KB < kn) load(ring[d], k0 + d * HEAD_KB);
    if (k0 > 0) __syncthreads();             // every wave is done with the last chunk
    for (int i = threadIdx.x; i < 16 * NB * (kn / 8); i += TALL_NW * 64) {
      const int r = i / (kn / 8), e = i % (kn / 8) * 8;
      *(CX_LDS u32x4*)(hs + r * stride + e) =
          *(const u32x4*)(A.hidden + (size_t)min(r, A.B - 1) * A.ldh + k0 + e);
    }
    __syncthreads();
    for (int kb = 0; kb < kn; kb += DEPTH * HEAD_KB) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        const int k = kb + d * HEAD_KB;
        if (k >= kn) break;
        const int kx = k + (DEPTH - 1) * HEAD_KB;
        if (kx < kn) load(ring[(d + DEPTH - 1) % DEPTH], k0 + kx);
        multiply(ring[d], k);
      }
    }
  }
  head_keys<NB, TALL_MT, TALL_NW>(A, acc, v0, 0, blockIdx.x, s_key);
}

// One workgroup per batch row: the largest key of its workgroups, four
// loads per thread in flight together.
__global__ __launch_bounds__(HEAD_WG) void head_merge(HeadArgs A) {
  __shared__ uint64_t s_red[HEAD_WG / 64];
  const int b = blockIdx.x;
  const uint64_t* p = A.part + (size_t)b * A.nvt;
  uint64_t key = 0;
  for (int i0 = 0; i0 < A.nvt; i0 += 4 * HEAD_WG) {
    uint64_t k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = i0 + j * HEAD_WG + (int)threadIdx.x;
      k[j] = i < A.nvt ? p[i] : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) key = k[j] > key ? k[j] : key;
  }
  key = wave_reduce(key, OpMax());
  if (lane_id() == 0) s_red[wave_id()] = key;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int j = 1; j < HEAD_WG / 64; ++j) key = s_red[j] > key ? s_red[j] : key;
    A.out_id[b] = (int32_t)~(uint32_t)key;
    if (A.out_max) {
      const uint32_t k = (uint32_t)(key >> 32);
      A.out_max[b] = k == 0xFFFFFFFFu ? __builtin_nanf("") : key2f(k);
    }
  }
}

constexpr int HEAD_VT_MIN = 64;              // the smallest vocab tile of a plan
static int vocab_tiles(int V, int vt) { return (int)(((int64_t)V + vt - 1) / vt); }

// The launch of a batch of B rows over V vocab rows: batch tiles of 32, 64,
// 128 or 256 rows, and workgroups of 64 (4 waves), 128 or 256 vocab rows (8
// waves of 16 or 32), or of 512 (16 waves, head_tall).
struct HeadPlan {
  int nt;            // index of the batch tile: 32 << nt rows
  int vt;            // vocab rows per workgroup
  int nby;           // batch tiles
  bool seg;          // four starting points in k
};
static HeadPlan head_plan(int B, int D, int V, int64_t ldw) {
  HeadPlan p;
  // weight rows a multiple of 4096 bytes apart: four starting points in k
  // (each quarter a whole number of ring turns), for up to 64 batch rows
  p.seg = B <= 64 && ldw % 2048 == 0 && D % (4 * WIDE_RING * WIDE_SK) == 0;
  p.nt = B <= 32 ? 0 : B <= 64 ? 1 : B <= 128 ? 2 : 3;
  p.nby = (B + (32 << p.nt) - 1) / (32 << p.nt);
  if (p.nt == 0) {
    // small workgroups balance best at every V: 120 against 134 us for 128
    // vocab rows at V = 80000, 11 against 15 us at V = 4080
    p.vt = HEAD_VT_MIN;
    // head_tall where its tiles fill the CUs in one round and k either is
    // short or starts at 0 everywhere (B = 32, us, tall against wide: 251
    // tiles D = 256 17 and 22, 3072 141 and 155; 196 tiles D = 1536 65 and
    // 72; 167 tiles D = 768 35 and 38, 1536 63 and 63; 147 tiles D = 512 21
    // and 21, 768 34 and 32; 128 tiles D = 512 22 and 18)
    const int t = vocab_tiles(V, TALL_VT);
    if (!p.seg && (D <= 256 ? t >= 144
                            : t <= 256 && (t >= 192 || (t >= 160 && D <= 768) ||
                                           (t >= 144 && D <= 512))))
      p.vt = TALL_VT;
  } else if (p.nt < 3) {
    // 128 vocab rows (B = 64: 57 against 62 us at V = 32000) once they fill
    // most of the CUs; below, 64 (18 against 24 us at V = 16000)
    p.vt = V > 128 * 160 ? 128 : 64;
  } else {
    // one workgroup per CU at a time: the fewest rounds over the 256 CUs,
    // each weighted by its measured time in us (D = 4096)
    const int vts[3] = {256, 128, 64}, us[3] = {150, 92, 67};
    long best = 0;
    for (int i = 0; i < 3; ++i) {
      const long wg = (long)((V + vts[i] - 1) / vts[i]) * p.nby;
      const long cost = (wg + 255) / 256 * us[i];
      if (i == 0 || cost < best) { best = cost; p.vt = vts[i]; }
    }
  }
  return p;
}

int launch_head(const HeadArgs& A0, hipStream_t s) {
  HeadArgs A = A0;
  const HeadPlan p = head_plan(A.B, A.D, A.V, A.ldw);
  A.nvt = vocab_tiles(A.V, p.vt);
  const bool seg = p.seg;
  using K = void (*)(HeadArgs);
  if (p.vt == TALL_VT) {
    const int v = A.B > 16;
    static const K tall[2] = {head_tall<1, 3>, head_tall<2, 2>};
    const int kc = min(A.D, v ? tall_chunk<2>() : tall_chunk<1>());
    // the dynamic-LDS limit raised once per variant to the most any launch takes
    static std::once_flag once[2];
    hipError_t err = hipSuccess;
    std::call_once(once[v], [&] {
      err = hipFuncSetAttribute((const void*)tall[v], hipFuncAttributeMaxDynamicSharedMemorySize,
                                TALL_LDS);
    });
    if (err != hipSuccess) return (int)err;
    timed_launch(CX_KERNEL_LMHEAD, tall[v], dim3((unsigned)A.nvt), dim3(TALL_NW * 64),
                 (uint32_t)(16 * (v + 1) * (kc + 8) * 2), s, A);
    timed_launch(CX_KERNEL_LMHEAD_MERGE, head_merge, dim3(A.B), dim3(HEAD_WG), 0, s, A);
    return (int)hipGetLastError();
  }
  K k;
  switch (p.nt) {
    case 0: k = seg ? head_wide<2, 1, 4, 4> : head_wide<2, 1, 4, 1>; break;
    case 1:
      k = p.vt == 64 ? (seg ? head_wide<4, 1, 4, 4> : head_wide<4, 1, 4, 1>)
                     : (seg ? head_wide<4, 1, 8, 4> : head_wide<4, 1, 8, 1>);
      break;
    case 2: k = p.vt == 64 ? head_wide<8, 1, 4, 1> : head_wide<8, 1, 8, 1>; break;
    default:
      k = p.vt == 64 ? head_wide<16, 1, 4, 1>
                     : p.vt == 128 ? head_wide<16, 1, 8, 1> : head_wide<16, 2, 8, 1>;
  }
  timed_launch(CX_KERNEL_LMHEAD, k, dim3((unsigned)(A.nvt * p.nby)), dim3(p.vt == 64 ? 256 : 512),
               0, s, A);
  timed_launch(CX_KERNEL_LMHEAD_MERGE, head_merge, dim3(A.B), dim3(HEAD_WG), 0, s, A);
  return (int)hipGetLastError();
}

}  // namespace cx

extern "C" {

// The keys of the smallest vocab tile any plan takes: the size grows with B
// and with V, though the plan's own tile does not, so a workspace of the
// largest call serves every smaller one (B = 256, V = 128256: 4.1 MB, of
// which that plan writes 1.0).
size_t cx_lmhead_workspace_bytes(int32_t B, int32_t V) {
  if (B <= 0 || V <= 0) return 256;
  return ((size_t)B * cx::vocab_tiles(V, cx::HEAD_VT_MIN) * 8 + 255) & ~(size_t)255;
}

int cx_lmhead_argmax_bf16(const uint16_t* hidden, int64_t ldh, const uint16_t* weight,
                          int64_t ldw, int32_t B, int32_t D, int32_t V, int32_t* out_id,
                          float* out_max, float* out_logits, void* workspace, size_t ws_bytes,
                          void* stream) {
  if (B < 0 || V < 1 || D < 1 || ldh < D || ldw < D)
    return cx::api_fail(CX_EINVAL, "bad shape");
  if (B == 0) return CX_OK;
  if (D % cx::HEAD_KB != 0)
    return cx::api_fail(CX_EINVAL, "D (%d) must be a multiple of %d", D, cx::HEAD_KB);
  if (!hidden || !weight || !out_id || !workspace)
    return cx::api_fail(CX_EINVAL, "null pointer argument");
  if ((((uintptr_t)hidden | (uintptr_t)weight) & 15) || ((ldh | ldw) & 7))
    return cx::api_fail(CX_EINVAL, "hidden and weight rows must be 16-byte aligned");
  const size_t need = (size_t)B * cx::vocab_tiles(V, cx::head_plan(B, D, V, ldw).vt) * 8;
  if (ws_bytes < need)
    return cx::api_fail(CX_ENOSPACE, "workspace holds %zu bytes, needs %zu", ws_bytes, need);
  cx::HeadArgs A;
  A.hidden = hidden; A.weight = weight; A.ldh = ldh; A.ldw = ldw;
  A.B = B; A.D = D; A.V = V;
  A.part = (uint64_t*)workspace;
  A.out_id = out_id; A.out_max = out_max; A.out_logits = out_logits;
  const int e = cx::launch_head(A, (hipStream_t)stream);
  if (e != 0) return cx::api_fail(CX_EHIP, "lm-head launch: %s", hipGetErrorString((hipError_t)e));
  return CX_OK;
}

}  // extern "C"
