// cx_deep.hpp -- rows whose nucleus is deeper than any region (reference
// chenxing/core/sampler.py:81-93 and :117-127): top-p and min-p rows with no
// top-k, no typical-p and no penalty window, which the fused kernel leaves
// pending because their kept set outgrows its region; and typical-p rows with
// no other filter.  One workgroup per row; two passes over the row (three
// with min-p) and two short ones, in place of the multi-pass path's eight or
// more:
//
//   pass 1  where the cut lies: a histogram of the terms exp((x - M) / T) (M
//           the row maximum) over DNB value buckets linear in (M - x) / T on
//           [0, DSPAN), the terms in fp32 rounded to integers of 11 bits or
//           more in a scale of their bucket, and from it the buckets the
//           running sum can reach top_p in, the roundings allowed for:
//           usually one
//   pass 2  in fp64, every term e = exp((x - M) / T) <= 1 (table-driven exp):
//           the row's sum S and, per wave range (the row split into NWAVE
//           contiguous id ranges), the sum above those buckets, in registers;
//           the elements of the buckets themselves are gathered.
//   cut     the gathered elements sorted by value (descending) and id
//           (ascending) and scanned on from the sum above them
//           (sampler.py:82-85: cumsum of the sorted probabilities,
//           searchsorted, one past the index): the cut element; of the cut
//           value's group the survivors spread over its ids (spread_kept,
//           cx_device.hpp).  Each range's kept mass is its sum above plus its
//           kept gathered elements.  (With min-p, pass 3 instead sums each
//           range's kept terms again, testing e >= min_p per element,
//           sampler.py:91-93.)
//   draw    the range holding u * Z (Z the kept total), then its sixteenth
//           (each wave sums one); one wave scans that sixteenth in id order
//           (sampler.py:126-127: choice == searchsorted(cumsum, u, 'right'))
//
// Bound: pass 1 by the LDS additions (about 23 cycles a wave), pass 2 by the
// fp64 VALU (a table exp per element), one CU per row.  An exact fixed-point
// histogram in pass 1 instead (64-bit additions, per-range copies, and a
// second pass that took another exponential for the elements between the
// copies' boundary and the cut) took 59 + 46 us at V = 128256 fp32; fp32 LDS
// additions in pass 1 take 164 us, eight times the 32-bit integer ones.
//
// On bf16 rows a term is the product of three LDS table entries, one per
// part of the value's bits (sign, exponent and the top three mantissa bits;
// the next two; the last two: x = xh + xm + xl exactly), each exp of its
// part (exp((xh - M) / T), exp(xm / T), exp(xl / T)), built once per row:
// no fp64 exp per element.  (Rows whose |x| / T could reach 7000 use the
// exp per element, so no table entry can overflow.)
//
// Each thread reads 32 bytes per pass step (8 fp32 or 16 bf16 values).  On
// rows that start at whole dwords (SampleArgs::vec_ok) these are two
// range-checked buffer loads, issued three steps ahead and unpacked only
// where used, so the loads stay in flight; other rows (bf16 rows at odd
// addresses, and fp32 rows of a pointer off a dword address) load value by
// value.
//
// The sums that decide run in a fixed order in fp64.  Each term is within
// 1 ulp (2.5 ulp for the table product), fp64 sums of at most 2^20 terms
// within 2^20 ulp, and the reference's own cumulative sums within 4e-11 (relative)
// of exact: a decision closer to its threshold than 5e-11 of the total
// returns false and the row takes the multi-pass path, as do NaN rows, cuts
// below the bucket span and cut buckets of more elements than the gather
// holds.
#pragma once
#include "cx_device.hpp"
#include "cx_internal.hpp"

namespace cx {

constexpr int DNB = 4096;                     // value buckets
constexpr float DSPAN = 40.0f;                // bucket span below M, units of T (exp(-40) ~ 4e-18)
constexpr float DSCALE = DNB / DSPAN;         // buckets per unit
constexpr double DTOL = 5e-11;                // relative decision margin
constexpr int DCAP = 4 * WG;                  // gather capacity, fp32 rows (block_sort<4>)
constexpr int DCAP16 = 2 * WG;                // gather capacity, bf16 rows
constexpr int DW = 8;                         // 32-bit words per thread per step
constexpr int DNV = 16;                       // most values per thread per step (bf16)
// dynamic LDS: h[2 DNB] u32 | ab[NWAVE][NWAVE] f64 | X, where X
// holds the gather (gk u64 | gi i32 | ga i32, DCAP entries) on fp32 rows and
// the three term tables (4096 + 2048 + 2048 f64) on bf16 rows, whose gather
// (DCAP16 entries) takes h's place once the cut's buckets are known
constexpr int DEEP_OFF_AB = DCAP16 * 16;
constexpr int DEEP_OFF_X = DEEP_OFF_AB + NWAVE * NWAVE * 8;
constexpr int DEEP_LDS = DEEP_OFF_X + DCAP * 16;
static_assert(2 * DNB * 4 <= DEEP_OFF_AB && (4096 + 2048 + 2048) * 8 <= DCAP * 16 &&
              DCAP16 >= 2 * WG, "deep LDS layout");

// 16 bytes (vector_size, so host builds of this header compile too)
typedef uint32_t deep_u32x4 __attribute__((vector_size(16)));

// The row as the passes read it.  nv values per thread per step (8 fp32 or
// 16 bf16, 32 bytes), a step covering nv * WG ids.
struct DeepRow {
  __amdgpu_buffer_rsrc_t rs;  // the row, rounded up to 4 bytes (rows of whole dwords)
  const void* p;
  int V, nv, step;
  bool bf16;
};

// The 32 bytes holding values [e0, e0 + nv) (e0 a multiple of nv).  Rows of
// whole dwords: two range-checked 16-byte loads (zeros past the row, no branch), so
// the compiler can keep them in flight; other rows: value by value, zero
// past V.
template <bool VEC>
__device__ __forceinline__ void deep_fetch(const DeepRow& R, int e0, uint32_t (&w)[DW]) {
  if constexpr (VEC) {
    const int off = e0 * (R.bf16 ? 2 : 4);
    const deep_u32x4 a =
        __builtin_bit_cast(deep_u32x4, __builtin_amdgcn_raw_buffer_load_b128(R.rs, off, 0, 0));
    const deep_u32x4 b =
        __builtin_bit_cast(deep_u32x4, __builtin_amdgcn_raw_buffer_load_b128(R.rs, off + 16, 0, 0));
#pragma unroll
    for (int k = 0; k < 4; ++k) { w[k] = a[k]; w[4 + k] = b[k]; }
  } else if (R.bf16) {
    const uint16_t* p = (const uint16_t*)R.p;
#pragma unroll
    for (int k = 0; k < DW; ++k) {
      const uint32_t lo = e0 + 2 * k < R.V ? p[e0 + 2 * k] : 0u;
      const uint32_t hi = e0 + 2 * k + 1 < R.V ? p[e0 + 2 * k + 1] : 0u;
      w[k] = lo | (hi << 16);
    }
  } else {
    const float* p = (const float*)R.p;
#pragma unroll
    for (int k = 0; k < DW; ++k) w[k] = e0 + k < R.V ? __float_as_uint(p[e0 + k]) : 0u;
  }
}
// bf16 code of value j of a fetch (bf16 rows).
__device__ __forceinline__ uint32_t deep_code(const uint32_t (&w)[DW], int j) {
  return (j & 1) ? (w[j >> 1] >> 16) : (w[j >> 1] & 0xFFFFu);
}
// Word j / 2 (bf16) or j (fp32) of a fetch for a j known only at run time:
// selected, not indexed, so the fetch stays in registers.
__device__ __forceinline__ uint32_t deep_word(const uint32_t (&w)[DW], int k) {
  uint32_t r = 0u;
#pragma unroll
  for (int i = 0; i < DW; ++i) r |= k == i ? w[i] : 0u;
  return r;
}
// Value j of a fetch.
__device__ __forceinline__ float deep_val(const DeepRow& R, const uint32_t (&w)[DW], int j) {
  if (R.bf16) return __uint_as_float((j & 1) ? (w[j >> 1] & 0xFFFF0000u) : (w[j >> 1] << 16));
  return __uint_as_float(w[j < DW ? j : 0]);
}

// Value bucket of x, or -1 below the span (and for NaN): fp32 arithmetic,
// the same expression in every pass, so an element lands in the same
// bucket each time.
__device__ __forceinline__ int deep_bucket(float x, float Mf, float invTf) {
  const float d = (Mf - x) * invTf;
  return d < DSPAN ? (int)(d * DSCALE) : -1;
}
__device__ __forceinline__ double deep_term(float x, double M, double invT, const double* tab) {
  return exp64_neg(((double)x - M) * invT, tab);
}

// bf16 term tables: ta over code >> 4, tb and tc over (code >> 7) << 2 with
// mantissa bits 3..2, resp. 1..0, of the bf16 code.
__device__ __forceinline__ float bf16_of(uint32_t code) { return __uint_as_float(code << 16); }
__device__ inline void deep_build_tables(double* ta, double* tb, double* tc, double M, double invT,
                                         const double* tab) {
  // (entries of infinite or NaN codes, which no in-span value uses, are 0)
  auto fin = [](double v) { return v == v && v < __builtin_inf() ? v : 0.0; };
  for (int i = threadIdx.x; i < 4096; i += WG)
    ta[i] = fin(exp64(((double)bf16_of((uint32_t)i << 4) - M) * invT, tab));
  for (int i = threadIdx.x; i < 2048; i += WG) {
    const uint32_t hi = (uint32_t)(i >> 2) << 7, lo = (uint32_t)(i & 3);
    // exact differences of bf16 values sharing sign and exponent
    tb[i] = fin(exp64(((double)bf16_of(hi | (lo << 2)) - (double)bf16_of(hi)) * invT, tab));
    tc[i] = fin(exp64(((double)bf16_of(hi | lo) - (double)bf16_of(hi)) * invT, tab));
  }
}
__device__ __forceinline__ double deep_term16(uint32_t code, const double* ta, const double* tb,
                                              const double* tc) {
  const uint32_t se = (code >> 7) << 2;
  return ta[code >> 4] * tb[se | ((code >> 2) & 3u)] * tc[se | (code & 3u)];
}

// Exclusive prefix sum of one fp64 per thread across the workgroup, in a
// fixed order.  scratch: 2 * NWAVE slots.
__device__ __forceinline__ double block_excl_scan_d(double v, double* scratch) {
  double inc = v;
  for (int o = 1; o < 64; o <<= 1) {
    const double w = __shfl_up(inc, o);
    if (lane_id() >= o) inc += w;
  }
  if (lane_id() == 63) scratch[wave_id()] = inc;
  __syncthreads();
  if (threadIdx.x < 64) {
    const double w = threadIdx.x < NWAVE ? scratch[threadIdx.x] : 0.0;
    double y = w;
    for (int o = 1; o < 64; o <<= 1) {
      const double z = __shfl_up(y, o);
      if (lane_id() >= o) y += z;
    }
    if (threadIdx.x < NWAVE) scratch[NWAVE + threadIdx.x] = y - w;
  }
  __syncthreads();
  const double r = scratch[NWAVE + wave_id()] + (inc - v);
  __syncthreads();
  return r;
}

template <bool B>
struct DeepFlag {
  static constexpr bool value = B;
};

// f(k, w) for every step k < n of a pass over ids from lo on (this
// thread's fetch w from id lo + k * stride + nv * idx on), with the next
// three steps' loads in flight.
template <bool VEC, class F>
__device__ __forceinline__ void deep_stream(const DeepRow& R, int lo, int stride, int idx, int n,
                                            F&& f) {
  const int e = lo + R.nv * idx;
  uint32_t b0[DW], b1[DW], b2[DW], b3[DW];
  deep_fetch<VEC>(R, e, b0);
  deep_fetch<VEC>(R, e + stride, b1);
  deep_fetch<VEC>(R, e + 2 * stride, b2);
  for (int k = 0; k < n; k += 4) {
    deep_fetch<VEC>(R, e + (k + 3) * stride, b3);
    f(k, b0);
    if (k + 1 >= n) break;
    deep_fetch<VEC>(R, e + (k + 4) * stride, b0);
    f(k + 1, b1);
    if (k + 2 >= n) break;
    deep_fetch<VEC>(R, e + (k + 5) * stride, b1);
    f(k + 2, b2);
    if (k + 3 >= n) break;
    deep_fetch<VEC>(R, e + (k + 6) * stride, b2);
    f(k + 3, b3);
  }
}

// Does the row qualify, and its maximum M (from the fused kernel's slice
// records: exact, the raw values being unpenalised).
// (the conditions on the call and the row's parameters alone; a top-k
// bound only where the caller's path applies it: the counted bf16 path)
__device__ inline bool deep_candidate(const SampleArgs& A, int row, const cx_row_params& P,
                                      bool topk_ok = false) {
  if (A.all_slow || A.out_probs) return false;
  if (!(P.temperature > 0.0) || P.typical_p < 1.0) return false;
  if (P.top_k > 0 && P.top_k < A.V && !topk_ok) return false;
  if (A.logV * (1.0 / P.temperature) > 740.0) return false;       // P**(1/T) may underflow
  if (A.ldh > 0 && A.hist_len[row] > 0 &&
      (P.repetition_penalty != 1.0 || P.presence_penalty != 0.0 || P.frequency_penalty != 0.0))
    return false;
  return true;
}
__device__ inline bool deep_eligible(const SampleArgs& A, int row, const cx_row_params& P,
                                     double& M, bool topk_ok = false) {
  if (!deep_candidate(A, row, P, topk_ok)) return false;
  double m = -__builtin_inf();
  for (int s = 0; s < A.nsplit; ++s) {
    const double v = A.stats[(size_t)row * A.nsplit + s].m;
    m = v > m ? v : m;
  }
  M = m;
  return m > -__builtin_inf() && m < __builtin_inf();
}

// ---------------------------------------------------------------- whole rows
// Rows with no top-k, top-p or min-p and no penalty window: the draw (or,
// with typical-p, the order's entropy) takes every element, so no candidate
// region helps.  The fused kernel reads such a row once (whole_slice) and
// keeps, per 1024-element chunk, the chunk's maximum and its fp64 sums
// against it; slow_kernel's workgroup of the row then has the normaliser and
// every chunk's place in the cumulative sum from one scan of at most ~1040
// records, and the draw reads a single chunk (whole_finish).
//
// Bound: the fused kernel's slices are fp64-VALU work (one table exp per
// element, ~25 instructions; HBM would allow 5 us for 64 rows of 128256
// fp32) on all CUs; the finish is a chain of barriers on one CU per row.
// Before, the row was streamed for a region it then outgrew and summed,
// bucketed and drawn by one workgroup: 64 rows of 128256 fp32, no filter,
// 108 us a call, now 24.6; typical-p 0.95 on the multi-pass path, 1230 us, now
// 117 (deep_row below).
struct WholePart {
  double s;          // sum of exp((x - m) / T) over the chunk (NaN: a NaN or +inf element)
  double sd;         // sum of exp((x - m) / T) (x - m) / T
  float m;           // the chunk's maximum
  int32_t pad;
};
constexpr int WCH = 1024;                     // elements per chunk
static_assert((SLICE_MAX / WCH + 2) * sizeof(WholePart) <= CAPS * sizeof(Cand),
              "a slice's records fit its region");

// (a row without a penalty window; ln V / T > 740: P**(1/T) may underflow)
__device__ __forceinline__ bool whole_row(const SampleArgs& A, const cx_row_params& P) {
  return !(P.top_k > 0 && P.top_k < A.V) && !(P.top_p < 1.0) && !(P.min_p > 0.0) &&
         P.temperature > 0.0 && !A.out_probs && A.logV <= 740.0 * P.temperature;
}

// A slice's chunks: nvc of whole vectors from lo, then nsc over the rest
// [s0, hi) (everything, on bf16 rows at odd addresses), 1024 ids each but the last of
// either kind.
struct WholeSlice {
  int lo, s0, hi, nvc, nsc;
  __device__ int first(int i) const { return i < nvc ? lo + i * WCH : s0 + (i - nvc) * WCH; }
  __device__ int end(int i) const { return min(first(i) + WCH, i < nvc ? s0 : hi); }
};
__device__ __forceinline__ WholeSlice whole_slice_of(const SampleArgs& A, int split) {
  WholeSlice w;
  const int ne = A.bf16 ? 8 : 4;
  w.lo = split * A.split_len;
  w.hi = min(A.V, w.lo + A.split_len);
  w.s0 = (A.vec_ok & VEC_STREAM) && w.hi > w.lo ? w.lo + (w.hi - w.lo) / ne * ne : w.lo;
  w.nvc = (w.s0 - w.lo + WCH - 1) / WCH;
  w.nsc = w.hi > w.s0 ? (w.hi - w.s0 + WCH - 1) / WCH : 0;
  return w;
}

// One chunk's record, by one wave: 16 values per lane, -inf where absent.
__device__ __forceinline__ void whole_chunk(const float (&x)[16], double invT, const double* tab,
                                            WholePart* out) {
  float m = x[0];
  bool bad = false;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    m = fmaxf(m, x[j]);
    bad = bad || !(x[j] < __builtin_inff());
  }
  m = wave_reduce(m, OpMax());
  double s = 0.0, sd = 0.0;
  if (m > -__builtin_inff()) {
    double sa[4] = {0.0, 0.0, 0.0, 0.0}, da[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      // (-inf: the exponential's clamp, so 0 * inf never arises)
      const double d = fmax(((double)x[j] - (double)m) * invT, -745.2);
      const double e = exp64_neg(d, tab);
      sa[j & 3] += e;
      da[j & 3] += e * d;
    }
    s = wave_reduce((sa[0] + sa[1]) + (sa[2] + sa[3]), OpAdd());
    sd = wave_reduce((da[0] + da[1]) + (da[2] + da[3]), OpAdd());
  }
  if (ballot(bad)) s = __builtin_nan("");
  if (lane_id() == 0) {
    out->s = s;
    out->sd = sd;
    out->m = m;
  }
}

// Outcomes of whole_finish.
constexpr int WHOLE_OPEN = 0;      // degenerate or too near a step: the exact path
constexpr int WHOLE_DONE = 1;      // drawn
constexpr int WHOLE_TYP = 2;       // typical-p row: Z holds its sums for deep_row
struct WholeSums {
  double M;          // row maximum
  double c;          // -sum P d, d = (x - M) / T: the entropy less log of sum exp(d)
};

// All threads of the workgroup; every thread gets the same result.  The
// typical order's distance |log P + H| (sampler.py:97-98) is |d + c|.
__device__ inline int whole_finish(const SampleArgs& A, int row, const cx_row_params& P,
                                   double* red_d, int* red_i, WholeSums& Z) {
  __shared__ double tab[64];
  __shared__ double s_w[2 * NWAVE + 4];
  __shared__ double s_off;
  __shared__ int s_ok;
  const int t = threadIdx.x;
  const double invT = 1.0 / P.temperature;
  load_exp64_tab(tab);
  // records 2t and 2t + 1, slice by slice (V < 2^20: at most 1040 in all)
  double ps[2] = {0.0, 0.0}, pd[2] = {0.0, 0.0};
  float pm[2] = {-__builtin_inff(), -__builtin_inff()};
  {
    int base = 0;
    for (int sl = 0; sl < A.nsplit; ++sl) {
      const WholeSlice W = whole_slice_of(A, sl);
      const int n = W.nvc + W.nsc;
      const WholePart* q = (const WholePart*)(A.cands + ((size_t)row * A.nsplit + sl) * CAPS);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int i = 2 * t + j - base;
        if (i >= 0 && i < n) { ps[j] = q[i].s; pd[j] = q[i].sd; pm[j] = q[i].m; }
      }
      base += n;
    }
  }
  const float Mf = block_max(fmaxf(pm[0], pm[1]), (float*)red_i, -__builtin_inff());
  const double M = (double)Mf;
  double dsum = 0.0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (pm[j] > -__builtin_inff()) {
      const double dm = ((double)pm[j] - M) * invT;
      const double f = exp64_neg(dm, tab);
      dsum += f * (pd[j] + ps[j] * dm);
      ps[j] *= f;
    }
  }
  const double S = block_sum(ps[0] + ps[1], red_d);
  if (!(Mf > -__builtin_inff() && Mf < __builtin_inff() && S > 0.0 && S < __builtin_inf()))
    return WHOLE_OPEN;
  if (P.typical_p < 1.0) {
    Z.M = M;
    Z.c = -block_sum(dsum, red_d) / S;
    return Z.c >= 0.0 ? WHOLE_TYP : WHOLE_OPEN;
  }
  // the chunk holding u * S (sampler.py:126-127), then the element in it
  const double t2 = A.u[row] * S, tolS = DTOL * S;
  const double before = block_excl_scan_d(ps[0] + ps[1], s_w);
  const int mine = before + ps[0] > t2 ? 2 * t
                   : before + ps[0] + ps[1] > t2 ? 2 * t + 1 : INT_MAX;
  const int ci = block_min(mine, red_i, INT_MAX);
  if (ci == INT_MAX) return WHOLE_OPEN;
  if (mine == ci) s_off = (ci & 1) ? before + ps[0] : before;
  int lo = 0, hi = 0;
  {
    int base = 0;
    for (int sl = 0; sl < A.nsplit; ++sl) {
      const WholeSlice W = whole_slice_of(A, sl);
      const int n = W.nvc + W.nsc;
      if (ci >= base && ci < base + n) { lo = W.first(ci - base); hi = W.end(ci - base); }
      base += n;
    }
  }
  double e = 0.0;
  if (lo + t < hi) {
    const char* rowp = (const char*)A.logits + (size_t)row * (size_t)A.ld * (A.bf16 ? 2 : 4);
    const float x = A.bf16 ? __uint_as_float((uint32_t)((const uint16_t*)rowp)[lo + t] << 16)
                           : ((const float*)rowp)[lo + t];
    e = exp64_neg(((double)x - M) * invT, tab);
  }
  const double r = block_excl_scan_d(e, s_w) + s_off;      // (its barriers publish s_off)
  const int hit = block_min(r + e > t2 ? t : INT_MAX, red_i, INT_MAX);
  if (hit == INT_MAX) return WHOLE_OPEN;
  if (t == hit) s_ok = r + e > t2 + tolS && r < t2 - tolS ? 1 : 0;
  __syncthreads();
  if (!s_ok) return WHOLE_OPEN;
  if (t == 0) {
    A.out_id[row] = lo + hit;
    A.row_status[row] = CX_ROW_OK;
  }
  return WHOLE_DONE;
}

// TYP: a typical-p row with no other filter (sampler.py:95-105).  The same
// passes in the typical order, ascending |d + c| with d = (x - M) / T and
// c = -sum P d (whole_finish): the buckets are linear in that distance, in
// fp64, so the two sides of the order compare exactly.  A cut beside an
// element of the other side whose distance differs by less than 1e-11 is
// left to the multi-pass path.
template <bool VEC, bool TYP>
__device__ __forceinline__ bool deep_row_impl(const SampleArgs& A, int row, const cx_row_params& P,
                                     double M, unsigned char* dyn, double* red_d, int* red_i,
                                     double c) {
  __shared__ double tab[64];
  __shared__ double s_d[2 * NWAVE + 4];
  __shared__ double s_wm[NWAVE];                     // kept mass per wave range / sixteenth
  __shared__ int s_i[4];
  __shared__ int s_g[2];
  const int t = threadIdx.x, l = lane_id(), w = wave_id();
  M = lane_read(M, 0);                               // uniform: into scalar registers
  c = lane_read(c, 0);
  DeepRow R;
  R.V = A.V;
  R.bf16 = A.bf16 != 0;
  R.nv = R.bf16 ? 16 : 8;
  R.step = R.nv * WG;
  R.p = (const char*)A.logits + (size_t)row * (size_t)A.ld * (R.bf16 ? 2 : 4);
  R.rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(R.p), (short)0,
                                           (R.V * (R.bf16 ? 2 : 4) + 3) & ~3, 0x00020000);
  const int V = R.V, nv = R.nv;
  const double invT = 1.0 / P.temperature;
  const float Mf = (float)M, invTf = (float)invT;
  uint32_t* h = (uint32_t*)dyn;                      // TYP: the upper side's from DNB on
  double* ab = (double*)(dyn + DEEP_OFF_AB);         // ab[r * NWAVE + w]: range r's sum above, wave w's
  double* ta = (double*)(dyn + DEEP_OFF_X);
  double* tb = ta + 4096;
  double* tc = tb + 2048;
  // the term tables: bf16 rows of whole dwords whose |x| / T stays below
  // 7000 (others take the exponential itself: one pass for both is enough
  // where every load is a single value)
  const bool use_tab = VEC && R.bf16 && (fabs(M) + 40.0 * P.temperature) * invT < 7000.0;
  const int cap = R.bf16 ? DCAP16 : DCAP;
  unsigned char* gbase = R.bf16 ? dyn : dyn + DEEP_OFF_X;
  uint64_t* gk = (uint64_t*)gbase;
  int32_t* gi = (int32_t*)(gbase + cap * 8);
  int32_t* ga = (int32_t*)(gbase + cap * 12);        // the value's bits
  // wave ranges: NWAVE contiguous id ranges of L ids, L a multiple of the
  // step, so each workgroup step lies in one range
  const int L = ((V + NWAVE * R.step - 1) / (NWAVE * R.step)) * R.step;
  const int nsteps = (V + R.step - 1) / R.step, spr = L / R.step;
  int range = 0, left = spr;                         // pass 2's range, and its steps left
  // the typical order's distance of value x; the bucket of x (-1 past the
  // span): the same expression in every pass
  auto dist = [&](float x) { return fabs(((double)x - M) * invT + c); };
  auto bucket = [&](float x) -> int {
    if constexpr (!TYP) return deep_bucket(x, Mf, invTf);
    const double v = dist(x) * (double)DSCALE;
    return v < (double)DNB ? (int)v : -1;
  };
  // pass 1's integers: 2^s brings the bucket's largest term (of the typical
  // order's upper side, d + c > 0, where the terms grow with the distance)
  // into (2^(wbits - 2), 2^(wbits - 1)], so V of them, the fp32 error
  // included, stay below 2^32.  Rounding one of them to an integer changes it
  // by at most 1.02 * 2^(1 - wbits) of itself (a bucket's smallest is 0.99 of
  // its largest), the fp32 term by 2e-5: eps bounds the relative error of any
  // sum of them.
  const int wbits = __clz(V);
  const double eps = 1.02 * __builtin_ldexp(2.0, -wbits) + 2e-5;
  constexpr float LOG2E = 1.44269504f;
  const float cf = (float)c;
  auto weight_scale = [&](int b, bool up) -> int {
    const float top = up ? (float)(b + 1) * (1.0f / DSCALE) - cf : (float)b * (-1.0f / DSCALE) - cf;
    return wbits - 1 - (int)__builtin_ceilf(top * LOG2E);
  };
  const bool cut = TYP || P.top_p < 1.0;
  // (below, the decision margin, relative to the whole row's sum, is wide
  // beside the kept mass: the multi-pass path)
  if (TYP && !(P.typical_p >= 0.02)) return false;
  for (int b = t; b < 2 * DNB; b += WG) h[b] = 0u;
  for (int b = t; b < NWAVE * NWAVE; b += WG) ab[b] = 0.0;
  if (t == 0) { s_i[0] = 0; s_i[2] = 0; }
  load_exp64_tab(tab);                               // its barrier also orders the clears

  // ---- pass 1: the buckets [blo, bhi] that hold the cut
  int blo = DNB, bhi = DNB;                          // no cut: every bucket above it
  if (cut) {
    deep_stream<VEC>(R, 0, R.step, t, nsteps, [&](int k, const uint32_t (&wd)[DW]) {
      const int e0 = k * R.step + nv * t;
#pragma unroll
      for (int j = 0; j < DNV; ++j) {
        if (j >= nv) break;
        const float x = e0 + j < V ? deep_val(R, wd, j) : -__builtin_inff();
        const int b = bucket(x);
        const bool up = TYP && ((double)x - M) * invT + c > 0.0;
        const float lg = (x - Mf) * invTf * LOG2E + (float)weight_scale(b, up);
        if (b >= 0)
          atomicAdd(h + (up ? DNB : 0) + b, (uint32_t)(__builtin_amdgcn_exp2f(lg) + 0.5f));
      }
    });
    __syncthreads();
    double vb[4];
    double c4 = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int b = 4 * t + j;
      vb[j] = __builtin_ldexp((double)h[b], -weight_scale(b, false));
      if (TYP) vb[j] += __builtin_ldexp((double)h[DNB + b], -weight_scale(b, true));
      c4 += vb[j];
    }
    const double Sa = block_sum(c4, s_d);
    const double p = TYP ? P.typical_p : P.top_p;
    double incl = block_excl_scan_d(c4, s_d);
    // The mass up to a bucket's end against the mass past it, a : r, each
    // within eps: blo is the first bucket that can reach p, bhi the first
    // that must.  (Against the whole row's sum, top_p within eps of 1 would
    // have no upper bucket.)  slack: the mass below the span, at most
    // V exp(-40), and the rounding of r.
    const double slack = 5e-12 * Sa;
    int b0 = INT_MAX, b1 = INT_MAX;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      incl += vb[j];
      const double a = incl * (1.0 - p), r = (Sa - incl) * p;
      if (b0 == INT_MAX && vb[j] != 0.0 && a * (1.0 + eps) >= r * (1.0 - eps) - slack)
        b0 = 4 * t + j;
      if (b1 == INT_MAX && vb[j] != 0.0 && a * (1.0 - eps) >= r * (1.0 + eps) + slack * p)
        b1 = 4 * t + j;
    }
    // (uniform values, here and below, into scalar registers)
    blo = __builtin_amdgcn_readfirstlane(block_min(b0, red_i, INT_MAX));
    bhi = __builtin_amdgcn_readfirstlane(block_min(b1, red_i, INT_MAX));
    if (bhi == INT_MAX) return false;                // NaN sums, or p within 6e-12 of 1
  }
  if (use_tab) {
    deep_build_tables(ta, tb, tc, M, invT, tab);
    __syncthreads();
  }

  // ---- pass 2: S, the sums above the cut's buckets, and their elements
  double s = 0.0, above = 0.0;
  int bad = 0;
  auto pass2 = [&](auto tables) __attribute__((always_inline)) {
  deep_stream<VEC>(R, 0, R.step, t, nsteps, [&](int k, const uint32_t (&wd)[DW]) {
    constexpr bool TAB = decltype(tables)::value;
    const int e0 = k * R.step + nv * t;
    uint32_t mg = 0u;
#pragma unroll
    for (int j = 0; j < DNV; ++j) {
      if (j >= nv) break;
      const float x = e0 + j < V ? deep_val(R, wd, j) : -__builtin_inff();
      const int b = bucket(x);
      // (the tables leave out terms below the span: at most V exp(-40) in all)
      const double e = !TAB ? deep_term(x, M, invT, tab)
                            : (b >= 0 ? deep_term16(deep_code(wd, j), ta, tb, tc) : 0.0);
      if (!(x <= Mf)) bad = 1;
      s += e;
      above += (uint32_t)b < (uint32_t)blo ? e : 0.0;
      if ((uint32_t)(b - blo) <= (uint32_t)(bhi - blo)) mg |= 1u << j;
      // the sums so far: left to the end of the step, the selects keep every
      // term of it in a register
      if ((j & 3) == 3) __asm__ volatile("" : "+v"(s), "+v"(above), "+v"(mg), "+v"(bad));
    }
    // the lane's elements of the cut's buckets, one by one (few lanes have any)
    while (mg) {
      const int j = __builtin_ctz(mg);
      mg &= mg - 1u;
      const uint32_t wj = deep_word(wd, R.bf16 ? j >> 1 : j);
      const float x = __uint_as_float(!R.bf16 ? wj : (j & 1) ? (wj & 0xFFFF0000u) : (wj << 16));
      const int pos = atomicAdd(s_i, 1);
      if (pos < cap) {
        gk[pos] = d2key(TYP ? -dist(x) : (double)x);
        gi[pos] = e0 + j;
        ga[pos] = (int32_t)__float_as_uint(x);
      }
    }
    if (--left == 0 || k + 1 == nsteps) {
      const double m = wave_reduce(above, OpAdd());
      if (l == 0) ab[range * NWAVE + w] = m;
      above = 0.0;
      ++range;
      left = spr;
    }
  });
  };
  // (a branch per element would leave each wave waiting for its own table
  // read: 51 us at V = 128256 fp32)
  if (use_tab) pass2(DeepFlag<VEC>());
  else pass2(DeepFlag<false>());
  const double S = lane_read(block_sum(s, s_d), 0);
  if (block_max(bad, red_i, 0)) return false;        // NaN (or a value above M)
  const double tolS = DTOL * S;

  float xcut = -__builtin_inff();
  double dcut = 0.0;                                 // TYP: the cut distance
  int g0 = 0, gn = 0, gj = 0;                        // the cut value's group: none
  double kept = 0.0;                                 // range w's kept gathered terms, lane l's part
  if (cut) {
    const double tgt = (TYP ? P.typical_p : P.top_p) * S;
    const double total = lane_read(block_sum(t < NWAVE * NWAVE ? ab[t] : 0.0, s_d), 0);
    const int ng = __builtin_amdgcn_readfirstlane(s_i[0]);
    __syncthreads();
    if (ng > cap || ng == 0) return false;
    // key descending, id ascending: a few entries by counting the ones
    // before each, the count split over the threads left.  Every wave reads
    // every entry of its share from LDS, ng^2 / 64 reads in all, so larger
    // gathers take the bitonic sort, up to 14 us (64 rows of 128256, N(0, 2)
    // logits, top-p 0.5 at temperature 4, near 1000 entries: 225 against
    // 154 us a call; at temperature 2, 300 to 500 of them, 159 against 145).
    if (ng <= WG / 4) {
      int* rank = (int*)(gk + WG);
      const int np = max(64, 1 << (32 - __clz(max(ng, 2) - 1)));
      const int parts = WG / np, e = t & (np - 1), pt = t / np;
      rank[t] = 0;
      __syncthreads();
      const uint64_t ke = e < ng ? gk[e] : 0ull;
      const int32_t ie = e < ng ? gi[e] : 0, ae = e < ng ? ga[e] : 0;
      const int j0 = pt * ng / parts, j1 = (pt + 1) * ng / parts;
      int before = 0, same = e >= j0 && e < j1 ? -1 : 0;
#pragma unroll 4
      for (int j = j0; j < j1; ++j) {
        const uint64_t kj = gk[j];
        before += kj > ke ? 1 : 0;
        same += kj == ke ? 1 : 0;
      }
      // equal keys by id (fp32 rows: hardly ever any)
      if (ballot(e < ng && same > 0))
        for (int j = j0; j < j1; ++j) before += gk[j] == ke && gi[j] < ie ? 1 : 0;
      if (e < ng && before > 0) atomicAdd(rank + e, before);
      __syncthreads();
      const int re = rank[e];
      if (pt == 0 && e < ng) { gk[re] = ke; gi[re] = ie; ga[re] = ae; }
      __syncthreads();
    } else {
      block_sort<4>(gk, gi, ga, ng);
    }
    // thread t: sorted entries 4t .. 4t+3, their terms and running sums
    double qv[4];
    double s4 = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = 4 * t + j;
      qv[j] = e < ng ? deep_term(__uint_as_float((uint32_t)ga[e]), M, invT, tab) : 0.0;
      s4 += qv[j];
    }
    double run = total + block_excl_scan_d(s4, s_d);
    int jstar = INT_MAX;
    double cprev = 0.0, cstar = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = 4 * t + j;
      const double incl = run + qv[j];
      if (jstar == INT_MAX && e < ng && incl >= tgt) {
        jstar = e;
        cprev = run;
        cstar = incl;
      }
      run = incl;
    }
    const int js = __builtin_amdgcn_readfirstlane(block_min(jstar, red_i, INT_MAX));
    if (js == INT_MAX) return false;
    if (jstar == js) {
      // robust: this element's running sum clearly reaches the target and
      // the one before clearly does not (the first element is always kept)
      const bool first = !TYP && total == 0.0 && js == 0;
      const bool ok = cstar >= tgt + tolS && (first || cprev < tgt - tolS);
      s_i[1] = ok ? 1 : 0;
      s_g[0] = js;
      s_g[1] = js + 1;
      red_d[2 * NWAVE + 2] = key2d(gk[js]);
    }
    __syncthreads();
    if (!s_i[1]) return false;
    // the cut value's group: sorted positions [g0, g1), ascending ids
    {
      const uint64_t kj = gk[js];
      auto diff = [&](int e) { return (double)__uint_as_float((uint32_t)ga[e]) - M; };
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = 4 * t + j;
        if (e < ng && gk[e] == kj) { atomicMin(&s_g[0], e); atomicMax(&s_g[1], e + 1); }
        // another d at the very same distance, the order's other side as a
        // rule (+0 and -0, or values that x - M rounds together, are one d;
        // its own flag, since waves behind this one still read s_i[1] above)
        if (TYP && e < ng && gk[e] == kj && diff(e) != diff(js)) s_i[2] = 1;
      }
    }
    __syncthreads();
    if constexpr (TYP) {
      if (t == 0) {
        const double kd = key2d(gk[js]);
        const double fr = -kd * (double)DSCALE;
        const bool near = (s_g[0] > 0 && key2d(gk[s_g[0] - 1]) - kd < 1e-11) ||
                          (s_g[1] < ng && kd - key2d(gk[s_g[1]]) < 1e-11) ||
                          fabs(fr - __builtin_rint(fr)) < 1e-8;   // beside the next bucket
        if (near || s_i[2]) s_i[1] = 0;
      }
      __syncthreads();
      if (!s_i[1]) return false;
    }
    if constexpr (TYP) dcut = lane_read(-red_d[2 * NWAVE + 2], 0);
    else xcut = (float)lane_read(red_d[2 * NWAVE + 2], 0);
    g0 = __builtin_amdgcn_readfirstlane(s_g[0]);
    gn = __builtin_amdgcn_readfirstlane(s_g[1]) - g0;
    gj = js + 1 - g0;
    // the kept part of the gathered elements, the entries above the cut value
    // and the group's survivors, in the keys' place (done with); wave w sums
    // range w's in their order
    if (P.min_p <= 0.0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = 4 * t + j;
        const bool k = e < g0 || (e < g0 + gn && spread_keeps(e - g0, gj, gn, V <= TIE_NET));
        if (e < ng) gk[e] = (uint64_t)__double_as_longlong(k ? qv[j] : 0.0);
      }
      __syncthreads();
      for (int e = l; e < g0 + gn; e += 64)
        kept += (uint32_t)(gi[e] - w * L) < (uint32_t)L ? __longlong_as_double((long long)gk[e]) : 0.0;
    }
  }

  // kept: above the cut value, or in its group among the survivors (the
  // group's member of a given id found by bisection of its sorted ids);
  // with min-p, e >= min_p
  const double minp = P.min_p;
  const double minp_tol = 1e-12 * minp;
  const uint32_t kcut = f2key(xcut);
  auto in_group = [&](int id) -> bool {
    if (gj >= gn) return true;
    int lo = g0, hi = g0 + gn;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (gi[mid] < id) lo = mid + 1; else hi = mid;
    }
    return spread_keeps(lo - g0, gj, gn, V <= TIE_NET);
  };
  auto kept_e = [&](float x, int id, int& amb) __attribute__((always_inline)) -> double {
    if constexpr (TYP) {
      const double v = dist(x);
      if (!(v < dcut || (v == dcut && in_group(id)))) return 0.0;
    } else {
      const uint32_t kx = f2key(x);
      if (!(kx > kcut || (kx == kcut && in_group(id)))) return 0.0;
    }
    const double ev = deep_term(x, M, invT, tab);
    if (minp > 0.0) {
      if (fabs(ev - minp) <= minp_tol) amb = 1;
      if (ev < minp) return 0.0;
    }
    return ev;
  };
  int amb = 0;
  // kept mass of ids [lo, hi) by one wave (hi - lo a multiple of 64 nv), in
  // a fixed order
  auto wave_mass = [&](int lo, int hi) __attribute__((always_inline)) -> double {
    double m = 0.0;
    const int n = hi > lo ? (hi - lo) / (64 * nv) : 0;
    deep_stream<VEC>(R, lo, 64 * nv, l, n, [&](int k, const uint32_t (&wd)[DW]) {
      const int e0 = lo + k * 64 * nv + nv * l;
#pragma unroll
      for (int j = 0; j < DNV; ++j) {
        if (j >= nv) break;
        if (e0 + j < V) m += kept_e(deep_val(R, wd, j), e0 + j, amb);
      }
    });
    return wave_sum(m);
  };

  // ---- each range's kept mass: its sums above the cut's buckets and its
  // kept gathered terms (no min-p), or pass 3
  if (minp <= 0.0) {
    double m = (l < NWAVE ? ab[w * NWAVE + l] : 0.0) + kept;
    m = wave_reduce(m, OpAdd());
    if (l == 0) s_wm[w] = m;
    __syncthreads();
  } else {
    const double m = wave_mass(w * L, w * L + L);
    if (l == 0) s_wm[w] = m;
    if (block_max(amb, red_i, 0)) return false;      // an element at the min-p floor
  }
  double Z = 0.0;
  for (int k = 0; k < NWAVE; ++k) Z += s_wm[k];
  if (!(Z > 0.0)) return false;
  const double tolZ = DTOL * Z;
  const double t2 = lane_read(A.u[row] * Z, 0);
  // the wave range holding t2
  int wr = -1;
  double off = 0.0;
  {
    double o = 0.0;
    for (int k = 0; k < NWAVE && wr < 0; ++k) {
      if (o + s_wm[k] > t2) { wr = k; off = o; }
      o += s_wm[k];
    }
  }
  __syncthreads();
  if (wr < 0) return false;
  // its sixteenth held by each wave
  const int SL = L / NWAVE;
  {
    const double m = wave_mass(wr * L + w * SL, wr * L + (w + 1) * SL);
    if (l == 0) s_wm[w] = m;
  }
  __syncthreads();
  int sr = -1;
  {
    double o = off;
    for (int k = 0; k < NWAVE && sr < 0; ++k) {
      if (o + s_wm[k] > t2) { sr = k; off = o; }
      o += s_wm[k];
    }
  }
  // one wave scans the sixteenth in id order: the first element whose
  // running sum exceeds t2
  if (w == 0) {
    int found = INT_MAX;
    bool ok = false;
    if (sr >= 0) {
      const int lo = wr * L + sr * SL;
      double runw = off;
      for (int base = lo; base < lo + SL && found == INT_MAX; base += 64 * nv) {
        const int e0 = base + nv * l;
        uint32_t wd[DW];
        deep_fetch<VEC>(R, e0, wd);
        double q[DNV];
        double ls = 0.0;
#pragma unroll
        for (int j = 0; j < DNV; ++j) {
          q[j] = j < nv && e0 + j < V ? kept_e(deep_val(R, wd, j), e0 + j, amb) : 0.0;
          ls += q[j];
        }
        double incl = ls;
        for (int o = 1; o < 64; o <<= 1) {
          const double y = __shfl_up(incl, o);
          if (l >= o) incl += y;
        }
        double r = runw + (incl - ls);               // running sum before this lane's elements
        int hit = INT_MAX;
        bool hok = false;
#pragma unroll
        for (int j = 0; j < DNV; ++j) {
          const double ri = r + q[j];
          if (hit == INT_MAX && ri > t2) {
            hit = e0 + j;
            hok = ri > t2 + tolZ && r < t2 - tolZ;
          }
          r = ri;
        }
        found = wave_min(hit);
        if (found != INT_MAX) ok = ballot(hit == found && hok) != 0ull;
        runw += lane_read(incl, 63);
      }
    }
    if (l == 0) s_i[3] = (found != INT_MAX && ok) ? found : -1;
  }
  __syncthreads();
  const int tok = s_i[3];
  if (block_max(amb, red_i, 0) || tok < 0) return false;
  if (t == 0) {
    A.out_id[row] = tok;
    A.row_status[row] = CX_ROW_OK | CX_ROW_FLAG_SLOW | CX_ROW_FLAG_DEEP;
  }
  return true;
}

// The exact normaliser sum over the row's ids [lo, hi) (lo a multiple of
// 16384; the whole row by default) of exp((x - M) / T), in fp64 with the
// table-driven exp, for a row without a penalty window: the passes' stream
// (loads three steps ahead) instead of one load round trip per eight
// elements.  The same value on every thread.
template <bool VEC>
__device__ inline double deep_exact_sum_impl(const SampleArgs& A, int row, double M, double invT,
                                             double* red_d, int lo, int hi) {
  __shared__ double etab[64];
  load_exp64_tab(etab);
  // the row as far as hi: the loads the stream issues past hi return zeros
  // and read nothing (not the next share's logits)
  hi = min(hi, A.V);
  DeepRow R;
  R.V = hi;
  R.bf16 = A.bf16 != 0;
  R.nv = R.bf16 ? 16 : 8;
  R.step = R.nv * WG;
  R.p = (const char*)A.logits + (size_t)row * (size_t)A.ld * (R.bf16 ? 2 : 4);
  R.rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(R.p), (short)0,
                                           (R.V * (R.bf16 ? 2 : 4) + 3) & ~3, 0x00020000);
  const int t = threadIdx.x;
  // per step, the fetch's values as straight-line code (a loop bounded by
  // R.nv, with a break at hi, ran its exps one after another): four
  // accumulators, element j into j % 4, values at or past hi selected away
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  deep_stream<VEC>(R, lo, R.step, t, (hi - lo + R.step - 1) / R.step,
                   [&](int k, const uint32_t (&wd)[DW]) {
    const int e0 = lo + k * R.step + R.nv * t;
    if (R.bf16) {
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float x = __uint_as_float((j & 1) ? (wd[j >> 1] & 0xFFFF0000u) : (wd[j >> 1] << 16));
        const double e = exp64_neg(((double)x - M) * invT, etab);
        s[j & 3] += e0 + j < hi ? e : 0.0;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const double e = exp64_neg(((double)__uint_as_float(wd[j]) - M) * invT, etab);
        s[j & 3] += e0 + j < hi ? e : 0.0;
      }
    }
  });
  return block_sum((s[0] + s[1]) + (s[2] + s[3]), red_d);
}
__device__ inline double deep_exact_sum(const SampleArgs& A, int row, double M, double invT,
                                        double* red_d, int lo = 0, int hi = INT_MAX) {
  return A.vec_ok ? deep_exact_sum_impl<true>(A, row, M, invT, red_d, lo, hi)
                  : deep_exact_sum_impl<false>(A, row, M, invT, red_d, lo, hi);
}

// Samples the row and returns true, or returns false with nothing written
// (the caller runs the multi-pass path).  All threads of the workgroup call
// it and get the same result.  dyn: DEEP_LDS bytes; red_d, red_i: >= 2 *
// NWAVE + 4 slots.  Z: a typical-p row's sums (whole_finish), else null.
__device__ __forceinline__ bool deep_row(const SampleArgs& A, int row, unsigned char* dyn, double* red_d,
                                int* red_i, const WholeSums* Z = nullptr) {
  const cx_row_params P = A.prm[row];
  if (Z)             // (bf16 rows at odd addresses: the multi-pass path)
    return A.vec_ok && deep_row_impl<true, true>(A, row, P, Z->M, dyn, red_d, red_i, Z->c);
  double M = 0.0;
  if (!deep_eligible(A, row, P, M)) return false;
  return A.vec_ok ? deep_row_impl<true, false>(A, row, P, M, dyn, red_d, red_i, 0.0)
                  : deep_row_impl<false, false>(A, row, P, M, dyn, red_d, red_i, 0.0);
}

}  // namespace cx
