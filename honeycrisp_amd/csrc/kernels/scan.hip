// Running sums / products and argsort along the middle axis of an [outer, reduce, inner] view.
//
// cumulativeSum / cumulativeProd (BackendCPU.swift:922-998): out[k] = x[0] (op) ... (op) x[k]
// (or up to x[k-1] when exclusive), optionally from the far end. Rows (inner == 1): a workgroup per row, or, for
// short ones, one wave that walks it in tiles of 64 x 4 elements (in-lane scan, wave scan of the lane totals
// by DPP, running carry); floats are combined in tree order, so they differ from the
// sequential CPU loop by rounding only; int64 is exact. Columns (inner > 1): one lane per
// column, sequential along the axis, lanes coalesced along inner. When there are too few lines
// to fill the chip (rows: and they are long), the axis is cut into segments: totals per segment, a small scan of the
// totals, then the segments are scanned starting from what precedes them.
//
// argsort (BackendCPU.swift:888-920): one block per (outer, inner) pair merge-sorts (key, index)
// pairs in LDS, up to 4096 elements; longer axes are sorted in runs of
// 4096 that are then merged 2, 4 or 8 at a time (every entry counts what goes before it in the other runs). Keys are mapped to unsigned
// integers that order like the values (-0 counts as +0), inverted for descending order; the
// source index breaks ties, so the sort is stable, which the reference's `stable` flag
// asks for and its unstable variant permits.
#include "common.hip.h"

enum { SCAN_SUM = 0, SCAN_PROD = 1 };

template <int OP, typename C> __device__ __forceinline__ C scan_identity() { return OP == SCAN_SUM ? (C)0 : (C)1; }
template <int OP, typename C> __device__ __forceinline__ C scan_combine(C a, C b) {
  return OP == SCAN_SUM ? a + b : a * b;
}

// v of another lane by DPP (`identity` where there is none), a cross-lane move of the vector ALU: no LDS, unlike a shuffle.
template <int CTRL, int ROWS, typename C> __device__ __forceinline__ C lane_move(C v, C identity) {
  if constexpr (sizeof(C) == 8) {
    const uint64_t x = (uint64_t)v, i = (uint64_t)identity;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)i, (int)x, CTRL, ROWS, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(i >> 32), (int)(x >> 32), CTRL, ROWS, 0xf, false);
    return (C)((uint64_t)hi << 32 | lo);
  } else {
    return __builtin_bit_cast(C, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, identity), __builtin_bit_cast(int, v), CTRL, ROWS, 0xf, false));
  }
}
// Inclusive scan over the lanes of a wave: within rows of 16 lanes, then from row to row.
template <int OP, typename C> __device__ __forceinline__ C wave_scan(C v) {
  constexpr C id = OP == SCAN_SUM ? (C)0 : (C)1;
  v = scan_combine<OP, C>(lane_move<0x111, 0xf>(v, id), v);   // row_shr:1, 2, 4, 8
  v = scan_combine<OP, C>(lane_move<0x112, 0xf>(v, id), v);
  v = scan_combine<OP, C>(lane_move<0x114, 0xf>(v, id), v);
  v = scan_combine<OP, C>(lane_move<0x118, 0xf>(v, id), v);
  v = scan_combine<OP, C>(lane_move<0x142, 0xa>(v, id), v);   // row_bcast:15 into rows 1 and 3
  v = scan_combine<OP, C>(lane_move<0x143, 0xc>(v, id), v);   // row_bcast:31 into rows 2 and 3
  return v;
}
// What is in the lanes below: the inclusive scan of the lane before (wave_shr:1).
template <int OP, typename C> __device__ __forceinline__ C wave_before(C incl) { return lane_move<0x138, 0xf>(incl, OP == SCAN_SUM ? (C)0 : (C)1); }

// v of lane `l` (the same in every lane)
template <typename C> __device__ __forceinline__ C lane_value(C v, uint32_t l) {
  if constexpr (sizeof(C) == 8) {
    const uint64_t x = (uint64_t)v;
    return (C)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), l) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)x, l));
  } else {
    return __builtin_bit_cast(C, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
  }
}

// What precedes segment `seg` of a row, from the totals of all of them, in the order of cumulative_carry_impl (same bits).
// A row of up to 256 segments does with this, four rounds at most in every wave, and saves the launch between
// the totals and the scan (2.8 us for [8, 50257] fp32 cut into segments).
template <typename C, int OP>
__device__ __forceinline__ C carry_before(const C* totals, uint32_t segs, uint32_t seg, uint32_t lane) {
  C run = scan_identity<OP, C>();
  for (uint32_t s0 = 0;; s0 += 64) {
    const C incl = wave_scan<OP, C>(s0 + lane < segs ? totals[s0 + lane] : scan_identity<OP, C>());
    if (seg < s0 + 64) {   // (the same in every lane)
      const C before = __shfl(incl, (int)((seg - s0 - 1) & 63), 64);
      return scan_combine<OP, C>(run, seg == s0 ? scan_identity<OP, C>() : before);
    }
    run = scan_combine<OP, C>(run, __shfl(incl, 63, 64));
  }
}

// PHASE 0: the scan itself (of whole lines, or of segments that start from their carry);
// PHASE 1: only the segments' totals, into p.carry.
template <typename T, int OP, int PHASE> __device__ __forceinline__ void cumulative_rows_impl(const hck_scan_args& p) {
  typedef typename Arith<T>::type C;
  constexpr int E = 4;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t segs = p.segs > 1 ? p.segs : 1;
  const uint32_t unit = blockIdx.x * (HCK_BLOCK / 64) + (threadIdx.x >> 6);  // (row, segment)
  if (unit >= p.outer * segs) return;
  const uint32_t row = unit / segs, seg = unit - row * segs;
  const uint32_t n = p.reduce;
  const uint32_t lo = segs > 1 ? seg * p.seg_len : 0;
  const uint32_t hi = segs > 1 ? (lo + p.seg_len < n ? lo + p.seg_len : n) : n;
  const T* in = (const T*)p.in + (size_t)row * n;
  T* out = (T*)p.out + (size_t)row * n;
  C carry = scan_identity<OP, C>();
  if (PHASE == 0 && segs > 1) {
    if (p.totals) carry = carry_before<C, OP>((const C*)p.carry + (size_t)row * segs, segs, seg, lane);
    else carry = ((const C*)p.carry)[unit];
  }
  for (uint32_t base = lo; base < hi; base += 64 * E) {
    // logical positions t (in scan order) of this lane; the element sits at n-1-t when reversed
    C x[E], run = scan_identity<OP, C>();
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t t = base + lane * E + e;
      x[e] = t < hi ? to_arith(in[p.reverse ? n - 1 - t : t]) : scan_identity<OP, C>();
      run = scan_combine<OP, C>(run, x[e]);
    }
    if (PHASE == 1) {
      carry = scan_combine<OP, C>(carry, run);  // per lane; combined across the wave at the end
      continue;
    }
    // inclusive scan of the lane totals across the wave
    const C incl = wave_scan<OP, C>(run);
    C acc = scan_combine<OP, C>(carry, wave_before<OP, C>(incl));
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t t = base + lane * E + e;
      const C next = scan_combine<OP, C>(acc, x[e]);
      if (t < hi) out[p.reverse ? n - 1 - t : t] = from_arith<T>(p.exclusive ? acc : next);
      acc = next;
    }
    carry = scan_combine<OP, C>(carry, __shfl(incl, 63, 64));
  }
  if (PHASE == 1) {
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) carry = scan_combine<OP, C>(carry, __shfl_down(carry, d, 64));
    if (lane == 0) ((C*)p.carry)[unit] = carry;
  }
}

// A workgroup per row, one launch (the host's rule and figures: hc_cumulative). BLOCK lanes take tiles of 4 elements each, GROUP tiles at a time: all
// loads of a group are out before the first is waited for, and its waves' totals meet in LDS once. Bound by the vector ALU of the row's one
// unit, about 3.5 us per 32768 fp32. What it depends on is that lanes exchange by DPP: with shuffles, which go through LDS, rows of 4096 took 5.8 us
// on 256 lanes and 7.3 on 1024 (now 3.9 and 3.1), and with every lane reading all 16 totals of a tile [8, 50257] 10.1 (8.4).
template <typename T, int OP, uint32_t BLOCK> __device__ __forceinline__ void cumulative_rowblock_impl(const hck_scan_args& p) {
  typedef typename Arith<T>::type C;
  constexpr uint32_t E = 4, GROUP = sizeof(C) == 8 ? 4 : 8, WAVES = BLOCK / 64;
  __shared__ C totals[2][GROUP][WAVES];
  const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = p.reduce;
  const T* in = (const T*)p.in + (size_t)blockIdx.x * n;
  T* out = (T*)p.out + (size_t)blockIdx.x * n;
  C carry = scan_identity<OP, C>();
  uint32_t half = 0;   // (totals of neighbouring groups in turn: one barrier per group)
  for (uint32_t first = 0; first < n; first += GROUP * BLOCK * E, half ^= 1) {
    // x[g]: logical positions t .. t + 3 (in scan order) of tile g; the element sits at n-1-t when reversed
    T x[GROUP][E];
    const uint32_t tiles = (n - first + BLOCK * E - 1) / (BLOCK * E);
#pragma unroll
    for (uint32_t g = 0; g < GROUP; g++) {
      if (g >= tiles) break;
      const uint32_t t = first + (g * BLOCK + threadIdx.x) * E;
      if (t + E <= n) {
        load_vec_loose<T, E>(in + (p.reverse ? n - E - t : t), x[g]);
      } else {
#pragma unroll
        for (uint32_t e = 0; e < E; e++) x[g][p.reverse ? E - 1 - e : e] = t + e < n ? in[p.reverse ? n - 1 - t - e : t + e] : (T)scan_identity<OP, C>();
      }
    }
    C before[GROUP];   // everything in the wave's lanes below this one
#pragma unroll
    for (uint32_t g = 0; g < GROUP; g++) {
      if (g >= tiles) break;
      if (p.reverse) {
        const T x0 = x[g][0], x1 = x[g][1];
        x[g][0] = x[g][3], x[g][1] = x[g][2], x[g][2] = x1, x[g][3] = x0;
      }
      C incl = scan_identity<OP, C>();
#pragma unroll
      for (uint32_t e = 0; e < E; e++) incl = scan_combine<OP, C>(incl, to_arith(x[g][e]));
      incl = wave_scan<OP, C>(incl);
      before[g] = wave_before<OP, C>(incl);
      if (lane == 63) totals[half][g][wave] = incl;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t g = 0; g < GROUP; g++) {
      if (g >= tiles) break;
      const uint32_t t = first + (g * BLOCK + threadIdx.x) * E;
      // (the waves' totals in a row of 16 lanes, scanned)
      static_assert(WAVES == 16 || WAVES == 4, "a power of two of at most 16");
      C total = totals[half][g][lane % WAVES];
      total = scan_combine<OP, C>(lane_move<0x111, 0xf>(total, scan_identity<OP, C>()), total);
      total = scan_combine<OP, C>(lane_move<0x112, 0xf>(total, scan_identity<OP, C>()), total);
      if constexpr (WAVES > 4) {
        total = scan_combine<OP, C>(lane_move<0x114, 0xf>(total, scan_identity<OP, C>()), total);
        total = scan_combine<OP, C>(lane_move<0x118, 0xf>(total, scan_identity<OP, C>()), total);
      }
      const C all = lane_value(total, WAVES - 1), lower = wave == 0 ? scan_identity<OP, C>() : lane_value(total, wave - 1);
      C acc = scan_combine<OP, C>(carry, scan_combine<OP, C>(lower, before[g]));
      carry = scan_combine<OP, C>(carry, all);
      if (t >= n) continue;
      T o[E];
#pragma unroll
      for (uint32_t e = 0; e < E; e++) {
        const C next = scan_combine<OP, C>(acc, to_arith(x[g][e]));
        o[e] = from_arith<T>(p.exclusive ? acc : next);
        acc = next;
      }
      if (t + E <= n) {
        if (p.reverse) {
          const T o0 = o[0], o1 = o[1];
          o[0] = o[3], o[1] = o[2], o[2] = o1, o[3] = o0;
        }
        store_vec_loose<T, E>(out + (p.reverse ? n - E - t : t), o);
      } else {
#pragma unroll
        for (uint32_t e = 0; e + 1 < E; e++)
          if (t + e < n) out[p.reverse ? n - 1 - t - e : t + e] = o[e];
      }
    }
  }
}

// VEC adjacent columns per lane (VEC > 1: inner is a multiple of VEC and the buffers are
// 16-byte aligned, so every access is one 16-byte piece).
template <typename T, int OP, int PHASE, int VEC>
__device__ __forceinline__ void cumulative_cols_impl(const hck_scan_args& p) {
  typedef typename Arith<T>::type C;
  const uint32_t segs = p.segs > 1 ? p.segs : 1;
  const uint32_t innerv = p.inner / VEC;
  const uint64_t t = (uint64_t)blockIdx.x * HCK_BLOCK + threadIdx.x;  // (i, segment, vector column)
  if (t >= (uint64_t)p.outer * segs * innerv) return;
  const uint32_t j = (uint32_t)(t % innerv) * VEC;
  const uint32_t is = (uint32_t)(t / innerv), i = is / segs, seg = is - i * segs;
  const uint32_t lo = segs > 1 ? seg * p.seg_len : 0;
  const uint32_t hi = segs > 1 ? (lo + p.seg_len < p.reduce ? lo + p.seg_len : p.reduce) : p.reduce;
  const size_t base = (size_t)i * p.reduce * p.inner + j;
  const T* in = (const T*)p.in + base;
  T* out = (T*)p.out + base;
  C* carry = (C*)p.carry + (size_t)is * p.inner + j;
  C run[VEC];
#pragma unroll
  for (int v = 0; v < VEC; v++) run[v] = (PHASE == 0 && segs > 1) ? carry[v] : scan_identity<OP, C>();
#pragma unroll 4
  for (uint32_t s = lo; s < hi; s++) {
    const size_t k = (size_t)(p.reverse ? p.reduce - 1 - s : s) * p.inner;
    T x[VEC], o[VEC];
    load_vec<T, VEC>(in + k, 0, 1, x);
#pragma unroll
    for (int v = 0; v < VEC; v++) {
      const C next = scan_combine<OP, C>(run[v], to_arith(x[v]));
      o[v] = from_arith<T>(p.exclusive ? run[v] : next);
      run[v] = next;
    }
    if (PHASE == 0) store_vec<T, VEC>(out, k, o);
  }
  if (PHASE == 1) {
#pragma unroll
    for (int v = 0; v < VEC; v++) carry[v] = run[v];
  }
}

// Segment totals -> what precedes each segment: one wave per line (i, j) scans its `segs` totals
// 64 at a time with shuffles (a lane walking them one by one would take longer than the scan
// of the data itself once a line has thousands of segments).
template <typename C, int OP> __device__ __forceinline__ void cumulative_carry_impl(const hck_scan_args& p) {
  const uint64_t line = (uint64_t)blockIdx.x * (HCK_BLOCK / 64) + (threadIdx.x >> 6);
  if (line >= (uint64_t)p.outer * p.inner) return;  // (whole waves)
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t i = (uint32_t)(line / p.inner), j = (uint32_t)(line - (uint64_t)i * p.inner);
  C* c = (C*)p.carry + (size_t)i * p.segs * p.inner + j;
  C run = scan_identity<OP, C>();
  for (uint32_t s0 = 0; s0 < p.segs; s0 += 64) {
    const uint32_t s = s0 + lane;
    const bool ok = s < p.segs;
    const C incl = wave_scan<OP, C>(ok ? c[(size_t)s * p.inner] : scan_identity<OP, C>());
    if (ok) c[(size_t)s * p.inner] = scan_combine<OP, C>(run, wave_before<OP, C>(incl));
    run = scan_combine<OP, C>(run, __shfl(incl, 63, 64));
  }
}

#define DEF_CUMULATIVE(TN, T)                                                                                   \
  HC_KERNEL void hc_cumulative_sum_rows_##TN(hck_scan_args p) { cumulative_rows_impl<T, SCAN_SUM, 0>(p); }      \
  HC_KERNEL void hc_cumulative_prod_rows_##TN(hck_scan_args p) { cumulative_rows_impl<T, SCAN_PROD, 0>(p); }    \
  HC_KERNEL void hc_cumulative_sum_cols_##TN(hck_scan_args p) { cumulative_cols_impl<T, SCAN_SUM, 0, 1>(p); }   \
  HC_KERNEL void hc_cumulative_prod_cols_##TN(hck_scan_args p) { cumulative_cols_impl<T, SCAN_PROD, 0, 1>(p); } \
  HC_KERNEL void hc_cumulative_sum_colsv_##TN(hck_scan_args p) {                                                \
    cumulative_cols_impl<T, SCAN_SUM, 0, VecWidth<T>::value>(p);                                                \
  }                                                                                                             \
  HC_KERNEL void hc_cumulative_prod_colsv_##TN(hck_scan_args p) {                                               \
    cumulative_cols_impl<T, SCAN_PROD, 0, VecWidth<T>::value>(p);                                               \
  }                                                                                                             \
  HC_KERNEL void hc_cumulative_sum_colsv_totals_##TN(hck_scan_args p) {                                         \
    cumulative_cols_impl<T, SCAN_SUM, 1, VecWidth<T>::value>(p);                                                \
  }                                                                                                             \
  HC_KERNEL void hc_cumulative_prod_colsv_totals_##TN(hck_scan_args p) {                                        \
    cumulative_cols_impl<T, SCAN_PROD, 1, VecWidth<T>::value>(p);                                               \
  }                                                                                                             \
  HC_KERNEL void hc_cumulative_sum_rows_totals_##TN(hck_scan_args p) { cumulative_rows_impl<T, SCAN_SUM, 1>(p); }   \
  HC_KERNEL void hc_cumulative_prod_rows_totals_##TN(hck_scan_args p) { cumulative_rows_impl<T, SCAN_PROD, 1>(p); } \
  HC_KERNEL void hc_cumulative_sum_cols_totals_##TN(hck_scan_args p) { cumulative_cols_impl<T, SCAN_SUM, 1, 1>(p); }   \
  HC_KERNEL void hc_cumulative_prod_cols_totals_##TN(hck_scan_args p) { cumulative_cols_impl<T, SCAN_PROD, 1, 1>(p); }
#define DEF_CUMULATIVE_ROWBLOCK(TN, T, NAME, OP)                                                                                   \
  HC_KERNEL void hc_cumulative_##NAME##_rowblock_##TN(hck_scan_args p) { cumulative_rowblock_impl<T, OP, HCK_BLOCK>(p); }           \
  extern "C" __global__ __launch_bounds__(1024) void hc_cumulative_##NAME##_rowblock_wide_##TN(hck_scan_args p) {                   \
    cumulative_rowblock_impl<T, OP, 1024>(p);                                                                                      \
  }
DEF_CUMULATIVE_ROWBLOCK(f32, float, sum, SCAN_SUM)
DEF_CUMULATIVE_ROWBLOCK(f32, float, prod, SCAN_PROD)
DEF_CUMULATIVE_ROWBLOCK(f16, half_t, sum, SCAN_SUM)
DEF_CUMULATIVE_ROWBLOCK(f16, half_t, prod, SCAN_PROD)
DEF_CUMULATIVE_ROWBLOCK(i64, int64_t, sum, SCAN_SUM)
DEF_CUMULATIVE_ROWBLOCK(i64, int64_t, prod, SCAN_PROD)
DEF_CUMULATIVE(f32, float)
DEF_CUMULATIVE(f16, half_t)
DEF_CUMULATIVE(i64, int64_t)
HC_KERNEL void hc_cumulative_sum_carry_f32(hck_scan_args p) { cumulative_carry_impl<float, SCAN_SUM>(p); }
HC_KERNEL void hc_cumulative_prod_carry_f32(hck_scan_args p) { cumulative_carry_impl<float, SCAN_PROD>(p); }
HC_KERNEL void hc_cumulative_sum_carry_i64(hck_scan_args p) { cumulative_carry_impl<int64_t, SCAN_SUM>(p); }
HC_KERNEL void hc_cumulative_prod_carry_i64(hck_scan_args p) { cumulative_carry_impl<int64_t, SCAN_PROD>(p); }

// ---------------------------------------------------------------- argsort

__device__ __forceinline__ uint64_t sort_key(float x) {
  x = x + 0.0f;  // -0 -> +0: the CPU's comparison treats them as equal
  uint32_t u = __float_as_uint(x);
  u ^= (u >> 31) ? 0xffffffffu : 0x80000000u;
  return (uint64_t)u;
}
__device__ __forceinline__ uint64_t sort_key(int64_t x) { return (uint64_t)x ^ 0x8000000000000000ull; }

constexpr int ARGSORT_MAX = 4096;
// Lanes of a sorting block while there are no more blocks than compute units. What bounds a block alone that merges (int64; 32-bit keys have the
// radix sort there) is the chain of dependent LDS reads: 26 per level and 8 levels with 16 entries per lane, 13 per level and 10 levels with 4. us,
// 256 lanes / 1024: 8 lines of 4096 int64 34.9 / 25.7, and of fp32, merged, 256 lines of 4096 26.6 / 21.6, but 512 33.0 / 33.4 and 1024
// 45.2 / 58.7, where blocks share a unit; 512 entries and fewer 7.6 / 8.2.
constexpr uint32_t SORT_WIDE_BLOCK = 1024;

// What the block sort orders. Keys of 32 significant bits (floats, halfs) travel with their
// index in one 64-bit word (key in the high half), so one integer comparison orders by
// (key, index); 64-bit keys keep the index in a second array. Entry i lives at slot
// i + i / 16: a lane that walks entries 16, 32, ... apart then still spreads over the banks.
constexpr uint32_t SORT_SLOTS = ARGSORT_MAX + ARGSORT_MAX / 16;
__device__ __forceinline__ uint32_t sort_slot(uint32_t i) { return i + (i >> 4); }

template <bool WIDE> struct SortBuf {
  uint64_t* keys;
  uint32_t* idxs;
  __device__ __forceinline__ void put(uint32_t i, uint64_t key, uint32_t idx) const {
    if (WIDE) {
      keys[sort_slot(i)] = key;
      idxs[sort_slot(i)] = idx;
    } else {
      keys[sort_slot(i)] = (key << 32) | idx;
    }
  }
  __device__ __forceinline__ void pad(uint32_t i) const {  // sorts behind every real entry
    keys[sort_slot(i)] = ~0ull;
    if (WIDE) idxs[sort_slot(i)] = 0xffffffffu;
  }
  __device__ __forceinline__ uint64_t key(uint32_t i) const {
    return WIDE ? keys[sort_slot(i)] : keys[sort_slot(i)] >> 32;
  }
  __device__ __forceinline__ uint32_t idx(uint32_t i) const {
    return WIDE ? idxs[sort_slot(i)] : (uint32_t)keys[sort_slot(i)];
  }
};

template <bool WIDE> __device__ __forceinline__ bool entry_before(uint64_t ka, uint32_t ia, uint64_t kb, uint32_t ib) {
  return ka < kb || (WIDE && ka == kb && ia < ib);
}

// before[e]: how many of the n entries from `base` on go before the one at place own + e, `entry[e]`. (Entries of the same
// 64-bit key lie in index order.)
template <bool WIDE, int E>
__device__ __forceinline__ void count_before(const SortBuf<WIDE>& buf, uint32_t base, uint32_t n, const uint64_t (&entry)[E], uint32_t own,
                                             uint32_t (&before)[E]) {
#pragma unroll
  for (int e = 0; e < E; e++) before[e] = 0;
#pragma unroll 8
  for (uint32_t t = 0; t < n; t++) {
    const uint64_t k = buf.keys[sort_slot(base + t)];
#pragma unroll
    for (int e = 0; e < E; e++) before[e] += k < entry[e] || (WIDE && k == entry[e] && base + t < own + e) ? 1 : 0;
  }
}

// Merge sort of E entries per lane, E * BLOCK in all (E up to 16 with 256 lanes, up to 4 with 1024), of which the first `count`
// are wanted, then runs merged pairwise through
// LDS: a lane finds by bisection where the merge path crosses its first output and merges E entries from there, one LDS
// read per entry. A level costs at most 13 + E dependent LDS reads (12 steps of the bisection at runs of 2048, the first entries
// of the two runs) and two barriers, whatever the run length; a bitonic network needs log2(run) stages for the same merge
// (lines of 1000 fp32: 13.5 -> 10.6 us, of 4096: 32 -> 25; int64 55 -> 34). Bound by the latency of those reads.
// The runs to start from: with one entry per lane (two of 32-bit keys), runs of 64, in which an entry's place is counted: all lanes of
// a wave read the same entry, and the reads do not depend on each other; with more, the E that a lane sorts in its
// registers (bitonic network on constant indices). [256, n] fp32 in us, merged from single entries / a bitonic network in LDS / now: n = 64 5.3 / 5.2 /
// 3.0 (argsort_impl alone), 128 6.0 / 5.9 / 4.5, 256 6.5 / 7.6 / 5.5, 512 8.1 / 7.6 / 7.4. (Two int64 entries per lane: counting costs two
// comparisons more, 9.8 us at 512 against 9.5.)
template <bool WIDE, int E, uint32_t BLOCK> __device__ __forceinline__ void merge_sort_lds(const SortBuf<WIDE>& buf, uint32_t count) {
  constexpr bool COUNTED = E == 1 || (E == 2 && !WIDE);
  uint64_t kx[E];
  uint32_t ix[E], to[E];   // an entry, and its place
  const uint32_t first = threadIdx.x * E;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t slot = sort_slot(first + e);
    kx[e] = buf.keys[slot];
    if (WIDE) ix[e] = buf.idxs[slot];
    to[e] = first + e;
  }
  if constexpr (COUNTED) {
    const uint32_t base = first & ~63u, in_run = base >= count ? 0 : count - base < 64 ? count - base : 64;
    uint32_t before[E];
    count_before<WIDE, E>(buf, base, in_run, kx, first, before);
#pragma unroll
    for (int e = 0; e < E; e++)
      if (first + e < count) to[e] = base + before[e];   // (what fills up the last run stays behind it)
    __syncthreads();
  } else {
#pragma unroll
    for (int k = 2; k <= E; k <<= 1)
#pragma unroll
      for (int s = k >> 1; s > 0; s >>= 1)
#pragma unroll
        for (int e = 0; e < E; e++) {
          const int f = e ^ s;
          if (f < e) continue;
          const bool e_after_f = entry_before<WIDE>(kx[f], WIDE ? ix[f] : 0, kx[e], WIDE ? ix[e] : 0);
          const bool swap = e_after_f == ((e & k) == 0);
          const uint64_t klo = swap ? kx[f] : kx[e], khi = swap ? kx[e] : kx[f];
          kx[e] = klo;
          kx[f] = khi;
          if (WIDE) {
            const uint32_t ilo = swap ? ix[f] : ix[e], ihi = swap ? ix[e] : ix[f];
            ix[e] = ilo;
            ix[f] = ihi;
          }
        }
  }
  for (uint32_t run = COUNTED ? 64 : E;; run <<= 1) {
#pragma unroll
    for (int e = 0; e < E; e++) {   // (every lane has read its inputs of the level before)
      const uint32_t slot = sort_slot(to[e]);
      buf.keys[slot] = kx[e];
      if (WIDE) buf.idxs[slot] = ix[e];
      to[e] = first + e;
    }
    __syncthreads();
    if (run >= count) return;
    const uint32_t a0 = first & ~(2 * run - 1), b0 = a0 + run, d = first - a0;
    uint32_t lo = d > run ? d - run : 0, hi = d < run ? d : run;
    while (lo < hi) {
      const uint32_t x = (lo + hi) >> 1, sa = sort_slot(a0 + x), sb = sort_slot(b0 + d - x - 1);
      if (entry_before<WIDE>(buf.keys[sa], WIDE ? buf.idxs[sa] : 0, buf.keys[sb], WIDE ? buf.idxs[sb] : 0)) lo = x + 1;
      else hi = x;
    }
    uint32_t x = a0 + lo, y = b0 + d - lo;         // next entry of either run
    const uint32_t x_end = b0, y_end = b0 + run;   // (an entry past its run's end is never taken; its slot is clamped)
    const uint32_t last = E * BLOCK - 1;
    uint32_t sa = sort_slot(x), sb = sort_slot(y < last ? y : last);
    uint64_t ka = buf.keys[sa], kb = buf.keys[sb];
    uint32_t ia = WIDE ? buf.idxs[sa] : 0, ib = WIDE ? buf.idxs[sb] : 0;
#pragma unroll
    for (int e = 0; e < E; e++) {
      const bool take_a = y >= y_end || (x < x_end && entry_before<WIDE>(ka, ia, kb, ib));
      kx[e] = take_a ? ka : kb;
      if (WIDE) ix[e] = take_a ? ia : ib;
      x += take_a ? 1 : 0;
      y += take_a ? 0 : 1;
      const uint32_t next = take_a ? x : y, slot = sort_slot(next < last ? next : last);
      const uint64_t k = buf.keys[slot];
      ka = take_a ? k : ka;
      kb = take_a ? kb : k;
      if (WIDE) {
        const uint32_t i = buf.idxs[slot];
        ia = take_a ? i : ia;
        ib = take_a ? ib : i;
      }
    }
    __syncthreads();
  }
}

// entries per lane that a sort of `count` <= ARGSORT_MAX entries runs with: a power of two up to ARGSORT_MAX / BLOCK
template <uint32_t BLOCK> __device__ __forceinline__ uint32_t sort_entries(uint32_t count) {
  uint32_t e = 1;
  while (e * BLOCK < count) e <<= 1;
  return e;
}

template <bool WIDE, uint32_t BLOCK> __device__ __forceinline__ void sort_lds(const SortBuf<WIDE>& buf, uint32_t count) {
  static_assert(ARGSORT_MAX == 16 * HCK_BLOCK && (BLOCK == HCK_BLOCK || BLOCK == SORT_WIDE_BLOCK), "entries per lane below assume 4096 entries and 256 or 1024 lanes");
  const uint32_t e = sort_entries<BLOCK>(count);
  if constexpr (BLOCK == HCK_BLOCK) {
    if (e == 16) return merge_sort_lds<WIDE, 16, BLOCK>(buf, count);
    if (e == 8) return merge_sort_lds<WIDE, 8, BLOCK>(buf, count);
  }
  if (e == 4) merge_sort_lds<WIDE, 4, BLOCK>(buf, count);
  else if (e == 2) merge_sort_lds<WIDE, 2, BLOCK>(buf, count);
  else merge_sort_lds<WIDE, 1, BLOCK>(buf, count);
}

// ---- Lines and chunks of 32-bit keys, blocks alone on their compute unit: radix sort of up to four entries per lane.
// A pass of 8 bits: a wave finds, entry by entry, the lanes with the same digit (a ballot per bit), which gives an entry its place among
// its wave's; the block sums up the counts of digits and waves; the entries move through LDS. Four passes for fp32, three for fp16 whatever the
// length, where merging takes ten levels of 13 dependent LDS reads. With four entries bound by the vector ALU (45 operations per entry and pass),
// with one by the latencies of four barriers. us, merged / now: 256 lines of 4096 fp32 21.6 / 17.4, fp16 21.9 / 13.4, of 1500 15.0 / 10.7, 8 of
// 1000 10.4 / 7.7, of 50257 (with the merging of 13 runs) 42.7 / 39.0, 256 of 300 (256 lanes) 7.5 / 6.6, of 128 4.9 / 5.2. Blocks that share
// a unit keep merging (1024 lines of 4096 44.8 / 60.4, of 512 11.9 / 12.7).

template <uint32_t BLOCK> struct RadixLds {
  static constexpr uint32_t WAVES = BLOCK / 64, PITCH = 257;   // (counters of a digit in different banks)
  static constexpr uint32_t ENTRIES = BLOCK == SORT_WIDE_BLOCK ? ARGSORT_MAX : 2 * BLOCK;
  uint32_t keys[ENTRIES], counts[WAVES * PITCH], sums[WAVES];
  uint16_t idxs[ENTRIES];
};

// key[e], idx[e]: entry (E wave + e) 64 + lane; afterwards the entry at that place in ascending order, equal keys in the order they had.
// FIRST: the lowest bit that differs between keys.
template <uint32_t BLOCK, int E, int FIRST> __device__ __forceinline__ void radix_sort(RadixLds<BLOCK>& lds, uint32_t (&key)[E], uint32_t (&idx)[E]) {
  constexpr uint32_t WAVES = RadixLds<BLOCK>::WAVES, PITCH = RadixLds<BLOCK>::PITCH, OWN = WAVES * 256 / BLOCK;
  const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  volatile uint32_t* mine = lds.counts + wave * PITCH;   // (volatile: a wave's LDS accesses are in order, and stay in the program's)
#pragma unroll
  for (int shift = FIRST; shift < 32; shift += 8) {
#pragma unroll
    for (int x = 0; x < 4; x++) mine[lane + 64 * x] = 0;
    uint32_t place[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t d = (key[e] >> shift) & 255;
      uint32_t low = ~0u, high = ~0u;   // the lanes whose entry has the same digit
#pragma unroll
      for (int bit = shift; bit < shift + 8 && bit < 32; bit++) {
        const uint32_t one = (uint32_t)__builtin_amdgcn_sbfe((int)key[e], bit, 1);   // 0 or all ones
        const uint64_t ones = __ballot(one != 0);
        low &= ~((uint32_t)ones ^ one);
        high &= ~((uint32_t)(ones >> 32) ^ one);
      }
      const uint32_t before = __builtin_amdgcn_mbcnt_hi(high, __builtin_amdgcn_mbcnt_lo(low, 0)), seen = mine[d];
      place[e] = seen + before;
      if (before == 0) mine[d] = seen + __popc(low) + __popc(high);
    }
    __syncthreads();
    // exclusive sums in the order of digits, a digit's waves one after the other
    const uint32_t d = tid * OWN / WAVES, w0 = tid * OWN % WAVES;
    uint32_t c[OWN], sum = 0;
#pragma unroll
    for (uint32_t x = 0; x < OWN; x++) c[x] = lds.counts[(w0 + x) * PITCH + d], sum += c[x];
    const uint32_t up = wave_scan<SCAN_SUM, uint32_t>(sum);
    if (lane == 63) lds.sums[wave] = up;
    __syncthreads();
    uint32_t base = up - sum;
#pragma unroll
    for (uint32_t w = 0; w < WAVES; w++) base += w < wave ? lds.sums[w] : 0;
#pragma unroll
    for (uint32_t x = 0; x < OWN; x++) {
      lds.counts[(w0 + x) * PITCH + d] = base;
      base += c[x];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t to = place[e] + mine[(key[e] >> shift) & 255];
      lds.keys[to] = key[e];
      lds.idxs[to] = (uint16_t)idx[e];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) {
      const uint32_t at = (E * wave + e) * 64 + lane;
      key[e] = lds.keys[at];
      idx[e] = lds.idxs[at];
    }
  }
}

// The `count` elements in[t * stride], sorted: f(place, key, t).
template <typename T, uint32_t BLOCK, int E, typename F>
__device__ __forceinline__ void radix_sort_line(RadixLds<BLOCK>& lds, const T* in, size_t stride, uint32_t count, uint32_t flip, F&& f) {
  uint32_t key[E], idx[E];
  const uint32_t first = threadIdx.x / 64 * (64 * E) + threadIdx.x % 64;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const uint32_t t = first + 64 * e;
    idx[e] = t;
    key[e] = t < count ? (uint32_t)sort_key(to_arith(in[(size_t)t * stride])) ^ flip : 0xffffffffu;   // (sorts behind every real entry)
  }
  radix_sort<BLOCK, E, sizeof(T) == 2 ? 13 : 0>(lds, key, idx);   // (a half as a float: 13 bits of the mantissa are clear)
#pragma unroll
  for (int e = 0; e < E; e++)
    if (first + 64 * e < count) f(first + 64 * e, key[e], idx[e]);
}
template <typename T, uint32_t BLOCK, typename F>
__device__ __forceinline__ void radix_sort_line(RadixLds<BLOCK>& lds, const T* in, size_t stride, uint32_t count, uint32_t flip, F&& f) {
  const uint32_t e = sort_entries<BLOCK>(count);
  if constexpr (BLOCK == SORT_WIDE_BLOCK) {
    if (e == 4) return radix_sort_line<T, BLOCK, 4>(lds, in, stride, count, flip, f);
  }
  if (e == 2) radix_sort_line<T, BLOCK, 2>(lds, in, stride, count, flip, f);
  else radix_sort_line<T, BLOCK, 1>(lds, in, stride, count, flip, f);
}

// descending order = ascending order of the inverted key
template <typename C> __device__ __forceinline__ uint64_t key_flip(uint32_t descending) {
  return descending ? ((sizeof(C) == 8) ? ~0ull : 0xffffffffull) : 0ull;
}

template <typename T, uint32_t BLOCK> __device__ __forceinline__ void argsort_impl(const hck_scan_args& p) {
  typedef typename Arith<T>::type C;
  constexpr bool WIDE = sizeof(C) == 8;
  __shared__ uint64_t keys[SORT_SLOTS];
  __shared__ uint32_t idxs[WIDE ? SORT_SLOTS : 1];
  const SortBuf<WIDE> buf{keys, idxs};
  const uint32_t i = blockIdx.x / p.inner, j = blockIdx.x - i * p.inner;
  const size_t base = (size_t)i * p.reduce * p.inner + j;
  const T* in = (const T*)p.in + base;
  int64_t* out = (int64_t*)p.out + base;
  const uint64_t flip = key_flip<C>(p.reverse);
  // One wave's work: the place that a lane counts for its entry is where its index goes. (The other waves end here; a barrier
  // waits for those that are left.)
  if (p.reduce <= 64) {
    const uint32_t t = threadIdx.x;
    if (t >= p.reduce) return;
    buf.put(t, sort_key((C)to_arith(in[(size_t)t * p.inner])) ^ flip, t);
    __syncthreads();
    const uint64_t entry[1] = {keys[sort_slot(t)]};
    uint32_t place[1];
    count_before<WIDE, 1>(buf, 0, p.reduce, entry, t, place);
    out[(size_t)place[0] * p.inner] = (int64_t)t;
    return;
  }
  const uint32_t N = sort_entries<BLOCK>(p.reduce) * BLOCK;
  for (uint32_t t = threadIdx.x; t < N; t += BLOCK) {
    if (t < p.reduce) buf.put(t, sort_key((C)to_arith(in[(size_t)t * p.inner])) ^ flip, t);
    else buf.pad(t);
  }
  __syncthreads();
  sort_lds<WIDE, BLOCK>(buf, p.reduce);
  for (uint32_t t = threadIdx.x; t < p.reduce; t += BLOCK) out[(size_t)t * p.inner] = (int64_t)buf.idx(t);
}

// Which line, and which of its `parts` pieces, block `l` takes. Blocks go to the eight XCDs round robin in launch order, each
// with an L2 of its own: the blocks of a line are given to blocks 8 apart, so that one L2 serves them all.
// (Lines beyond the last whole group of 8: launch order.)
__device__ __forceinline__ void line_on_xcd(uint32_t l, uint32_t parts, uint32_t lines, uint32_t& line, uint32_t& part) {
  const uint32_t grouped = lines / 8 * 8 * parts;
  if (l < grouped) {
    const uint32_t g = l / (8 * parts), r = l - g * 8 * parts;
    line = 8 * g + (r & 7);
    part = r >> 3;
  } else {
    line = l / parts;
    part = l - line * parts;
  }
}

// Long axes, pass 1: block (line, chunk) sorts elements [chunk * ARGSORT_MAX, ...) of its line
// and stores the sorted run: keys (32 bits, or 64 for int64 tensors) and indices.
template <typename T, typename K, uint32_t BLOCK> __device__ __forceinline__ void argsort_chunks_impl(const hck_sort_args& p) {
  typedef typename Arith<T>::type C;
  constexpr bool WIDE = sizeof(C) == 8;
  static_assert(sizeof(K) == sizeof(C), "keys have the size of the arithmetic type");
  __shared__ uint64_t keys[SORT_SLOTS];
  __shared__ uint32_t idxs[WIDE ? SORT_SLOTS : 1];
  const SortBuf<WIDE> buf{keys, idxs};
  const uint32_t chunks = (p.reduce + ARGSORT_MAX - 1) / ARGSORT_MAX;
  uint32_t line, chunk;
  line_on_xcd(blockIdx.x, chunks, p.outer * p.inner, line, chunk);
  const uint32_t i = line / p.inner, j = line - i * p.inner;
  const T* in = (const T*)p.in + (size_t)i * p.reduce * p.inner + j;
  const uint32_t first = chunk * ARGSORT_MAX;
  const uint32_t count = p.reduce - first < ARGSORT_MAX ? p.reduce - first : ARGSORT_MAX;
  const uint64_t flip = key_flip<C>(p.descending);
  for (uint32_t t = threadIdx.x; t < ARGSORT_MAX; t += BLOCK) {
    if (t < count) buf.put(t, sort_key((C)to_arith(in[(size_t)(first + t) * p.inner])) ^ flip, first + t);
    else buf.pad(t);
  }
  __syncthreads();
  sort_lds<WIDE, BLOCK>(buf, count);
  const size_t dst = (size_t)line * p.reduce + first;
  for (uint32_t t = threadIdx.x; t < count; t += BLOCK) {
    ((K*)p.keys_out)[dst + t] = (K)buf.key(t);
    p.idx_out[dst + t] = buf.idx(t);
  }
}

// (all N loads are out before the first is waited for: the compiler would make N branches of them, each with a load
// and a wait)
template <typename K> __device__ __forceinline__ void loaded_together(K (&)[1]) {}
template <typename K> __device__ __forceinline__ void loaded_together(K (&k)[3]) {
  asm volatile("" : "+v"(k[0]), "+v"(k[1]), "+v"(k[2]));
}
template <typename K> __device__ __forceinline__ void loaded_together(K (&k)[7]) {
  asm volatile("" : "+v"(k[0]), "+v"(k[1]), "+v"(k[2]), "+v"(k[3]), "+v"(k[4]), "+v"(k[5]), "+v"(k[6]));
}

// Long axes, pass 2..: WAYS neighbouring runs of length `run` (a power of two times 256) become one. The
// place of an entry is its place in its own run plus, for every other run of the group, the number of
// entries that go before it, found by bisection. The runs lie in index order, so ties go by the run: equal
// keys of an earlier run go before. A lane owns an entry and bisects in up to 8 runs at a time, independent loads
// in every step; neighbouring lanes own neighbouring keys and mostly read the same lines. The pass that
// completes the line writes the index straight to its place in the result.
// Bound by the address path where the tensor fills the device (the lanes of a load go to different lines, four lanes a cycle),
// so the loads are what counts: two passes of 4 ways make 2 * 3 * 13 per entry for 16 runs where one pass of 16 made
// 16 * 13 (argsort fp32, rows: [8, 50257] 56.7 -> 42.8 us, [256, 50257] 820 -> 478, [64, 131072] 842 -> 402; int64 [256, 50257] 1368 -> 753).
// Pairwise merging by coalesced passes, which these took the place of: 88.6, 818, 660 and 962.
// One tile of HCK_BLOCK entries: block `l` of the blocks of all lines.
template <typename K, int WAYS> __device__ __forceinline__ void argsort_rank_tile(const hck_sort_args& p, uint32_t l, uint32_t tiles) {
  constexpr int OTHERS = WAYS - 1;
  uint32_t line, tile;
  line_on_xcd(l, tiles, p.outer * p.inner, line, tile);
  const K* keys = (const K*)p.keys_in + (size_t)line * p.reduce;
  const uint32_t pos = tile * HCK_BLOCK + threadIdx.x;
  const uint32_t own = tile * HCK_BLOCK / p.run;  // a tile lies inside one run
  const uint32_t group = own / WAYS * WAYS;       // (runs are counted from the start of the line)
  const bool valid = pos < p.reduce;
  const K key = valid ? keys[pos] : (K)0;
  uint32_t rank = pos - own * p.run;
  uint32_t start[OTHERS], len[OTHERS], before[OTHERS];
  bool ties[OTHERS];
#pragma unroll
  for (int w = 0; w < OTHERS; w++) {
    const uint32_t r = group + w + (group + w >= own ? 1 : 0);  // the other runs of the group in turn
    const uint64_t s = (uint64_t)r * p.run;
    start[w] = s < p.reduce ? (uint32_t)s : 0;
    len[w] = s >= p.reduce ? 0 : p.reduce - (uint32_t)s < p.run ? p.reduce - (uint32_t)s : p.run;
    ties[w] = r < own;
    before[w] = 0;
  }
  for (uint32_t step = p.run; step > 0; step >>= 1) {
    K k[OTHERS];
#pragma unroll
    for (int w = 0; w < OTHERS; w++) {
      const uint32_t next = before[w] + step;
      k[w] = keys[start[w] + (next <= len[w] ? next - 1 : 0)];
    }
    loaded_together(k);
#pragma unroll
    for (int w = 0; w < OTHERS; w++) {
      const uint32_t next = before[w] + step;
      const bool goes_before = (k[w] < key) | (ties[w] & (k[w] == key));
      before[w] = (next <= len[w]) & goes_before ? next : before[w];
    }
  }
#pragma unroll
  for (int w = 0; w < OTHERS; w++) rank += before[w];
  if (!valid) return;
  const uint32_t place = group * p.run + rank, idx = p.idx_in[(size_t)line * p.reduce + pos];
  if (p.out != nullptr) {
    const uint32_t i = line / p.inner, j = line - i * p.inner;
    ((int64_t*)p.out)[((size_t)i * p.reduce + place) * p.inner + j] = (int64_t)idx;
  } else {
    ((K*)p.keys_out)[(size_t)line * p.reduce + place] = key;
    p.idx_out[(size_t)line * p.reduce + place] = idx;
  }
}

// (Every line rounds its tiles up, so they can be more than a launch's 2^32 - 1 lanes hold: the grid is cut off by the
// host, and a block goes on with the tile a whole grid further.)
template <typename K, int WAYS> __device__ __forceinline__ void argsort_rank_impl(const hck_sort_args& p) {
  const uint32_t tiles = (p.reduce + HCK_BLOCK - 1) / HCK_BLOCK, all = tiles * p.outer * p.inner;
  for (uint32_t l = blockIdx.x; l < all; l += gridDim.x) argsort_rank_tile<K, WAYS>(p, l, tiles);
}

#define DEF_RANK(WAYS)                                                                                     \
  HC_KERNEL void hc_argsort_rank##WAYS##_k32(hck_sort_args p) { argsort_rank_impl<uint32_t, WAYS>(p); }   \
  HC_KERNEL void hc_argsort_rank##WAYS##_k64(hck_sort_args p) { argsort_rank_impl<uint64_t, WAYS>(p); }
DEF_RANK(2)
DEF_RANK(4)
DEF_RANK(8)

template <typename T, uint32_t BLOCK> __device__ __forceinline__ void argsort_radix_impl(const hck_scan_args& p) {
  __shared__ RadixLds<BLOCK> lds;
  const uint32_t i = blockIdx.x / p.inner, j = blockIdx.x - i * p.inner;
  const size_t base = (size_t)i * p.reduce * p.inner + j;
  int64_t* out = (int64_t*)p.out + base;
  radix_sort_line<T, BLOCK>(lds, (const T*)p.in + base, p.inner, p.reduce, (uint32_t)key_flip<float>(p.reverse),
                            [&](uint32_t place, uint32_t, uint32_t t) { out[(size_t)place * p.inner] = (int64_t)t; });
}
template <typename T, uint32_t BLOCK> __device__ __forceinline__ void argsort_chunks_radix_impl(const hck_sort_args& p) {
  __shared__ RadixLds<BLOCK> lds;
  const uint32_t chunks = (p.reduce + ARGSORT_MAX - 1) / ARGSORT_MAX;
  uint32_t line, chunk;
  line_on_xcd(blockIdx.x, chunks, p.outer * p.inner, line, chunk);
  const uint32_t i = line / p.inner, j = line - i * p.inner, first = chunk * ARGSORT_MAX;
  const uint32_t count = p.reduce - first < ARGSORT_MAX ? p.reduce - first : ARGSORT_MAX;
  const size_t run = (size_t)line * p.reduce + first;
  radix_sort_line<T, BLOCK>(lds, (const T*)p.in + ((size_t)i * p.reduce + first) * p.inner + j, p.inner, count, (uint32_t)key_flip<float>(p.descending),
                            [&](uint32_t place, uint32_t key, uint32_t t) {
                              ((uint32_t*)p.keys_out)[run + place] = key;
                              p.idx_out[run + place] = first + t;
                            });
}

#define DEF_ARGSORT(T, TN, K, WIDE_CHUNKS, WIDE_LINE)                                                                             \
  HC_KERNEL void hc_argsort_chunks_##TN(hck_sort_args p) { argsort_chunks_impl<T, K, HCK_BLOCK>(p); }                           \
  HC_KERNEL void hc_argsort_##TN(hck_scan_args p) { argsort_impl<T, HCK_BLOCK>(p); }                                            \
  extern "C" __global__ __launch_bounds__(SORT_WIDE_BLOCK) void hc_argsort_chunks_wide_##TN(hck_sort_args p) { WIDE_CHUNKS(p); } \
  extern "C" __global__ __launch_bounds__(SORT_WIDE_BLOCK) void hc_argsort_wide_##TN(hck_scan_args p) { WIDE_LINE(p); }
#define DEF_ARGSORT_RADIX(T, TN)                                                                                                  \
  DEF_ARGSORT(T, TN, uint32_t, (argsort_chunks_radix_impl<T, SORT_WIDE_BLOCK>), (argsort_radix_impl<T, SORT_WIDE_BLOCK>))         \
  HC_KERNEL void hc_argsort_radix_##TN(hck_scan_args p) { argsort_radix_impl<T, HCK_BLOCK>(p); }
DEF_ARGSORT_RADIX(float, f32)
DEF_ARGSORT_RADIX(half_t, f16)
DEF_ARGSORT(int64_t, i64, uint64_t, (argsort_chunks_impl<int64_t, uint64_t, SORT_WIDE_BLOCK>), (argsort_impl<int64_t, SORT_WIDE_BLOCK>))
