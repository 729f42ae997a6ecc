// fp16 and fp32 GEMM for gfx950 with direct global->LDS loads (buffer_load_dwordx4 ... lds) and,
// for fp16 operands that are contiguous along M/N, transposing LDS reads
// (ds_read_b64_tr_b16). Block tile BM x BN, 4 waves 2 x 2, fp32 accumulate with
// v_mfma_f32_32x32x16_f16 / v_mfma_f32_32x32x2_f32. No operand passes through VGPRs on its
// way to LDS.
//
// LDS: two stages, each one K-slice of 128 bytes (64 halfs, 32 floats):
// [A region: BM*128 bytes][B region: BN*128 bytes]. 128 bytes because that is a cache line: a
// K-contiguous operand is then fetched as whole lines (8 lanes per row), which costs markedly
// less power and fewer texture-address cycles than two 64-byte halves fetched separately.
//   K-contiguous operand (A of NN/NT, B of NT/TT): rows of 128 bytes = eight 16-byte slots,
//     chunk c of row r in slot c ^ (r & 7); MFMA operand = one ds_read_b128, rows r .. r+7 of
//     one read hit eight different slots. For fp32 the four floats of a chunk feed four
//     consecutive MFMAs; lanes 0..31 take chunk 2s and lanes 32..63 chunk 2s+1 in sub-step s,
//     a permutation of k that both operands share.
//   M/N-contiguous fp16 operand (A of TN/TT, B of NN/TN): natural [k][m] layout, 64 k-rows of
//     ROWS halfs, 16-byte slot x of k-row k stored at slot x ^ g(k),
//     g(k) = ((k&7) ^ ((k>>3&1)<<2)) << 1. MFMA operand = two ds_read_b64_tr_b16: in a group
//     of 16 lanes, lane r points at k-row k0 + r/4, columns 4*(r%4)..+3 (8 bytes); the
//     instruction returns to lane i the four k-values of column i. Two reads (k0, k0+4) give
//     a lane its 8 consecutive k for one m, in the same order as the K-contiguous operand.
//   M/N-contiguous fp32 operand: [32 k][ROWS floats], MFMA operands are single ds_read_b32
//     (32 consecutive floats of k-row k for lanes 0..31, of k-row k+4 for lanes 32..63).
// A wave-level DMA instruction fills 1 KiB of LDS in lane order (lane l -> byte 16*l), so
// any permutation of 16-byte pieces inside a 1 KiB block is free: the lane simply fetches
// the global piece that belongs in its slot. Both swizzles stay inside such blocks.
//
// Pipeline. A K-step (one stage) is four sub-steps of one MFMA per accumulator tile, operands
// of the next sub-step being read under the MFMAs of the current one:
//   sub-step 0: second half of the DMA of K-step j+1 into the other stage
//   sub-steps 1, 2: no DMA: the loads in flight get at least these 2 x SLOTS MFMAs to land
//     (measured need: about 600 cycles)
//   wait for this wave's DMA (vmcnt 0), one LDS barrier: the other stage is complete and
//     nobody reads this stage any more
//   sub-step 3: first operands of K-step j+1 are read; first half of the DMA of K-step j+2
//     into this stage.
// DMA instructions are spread over the MFMAs of their sub-step (a burst would stall the
// issuing wave behind the texture-address queue). The two stages are distinct __shared__
// arrays and the loop is unrolled by two so that every LDS access names its stage statically.
#include "common.hip.h"
#include <type_traits>

// length of the DMA window in half sub-steps (see the K loop)
#ifndef HC_DMA_WINDOW_X2
#define HC_DMA_WINDOW_X2 4
#endif

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t Chunk __attribute__((ext_vector_type(4)));  // 16 bytes = 8 halfs

enum { DMA_K = 0, DMA_MN = 1 };

#define LDS_AS __attribute__((address_space(3)))

__device__ __forceinline__ uint32_t swz_k(uint32_t row) { return row & 7u; }
__device__ __forceinline__ uint32_t swz_mn(uint32_t k) { return (((k & 7u) ^ (((k >> 3) & 1u) << 2)) << 1); }

// Workgroup barrier for LDS traffic only: this wave's LDS reads have returned (lgkmcnt), its
// DMA is waited for separately (wait_dma), and nothing is said about global memory. A fence
// builtin would do the same but also waits for every DMA instruction in flight, including
// those that fill stages nobody is about to read. The "memory" clobber keeps the compiler
// from moving LDS accesses across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// s_waitcnt vmcnt(N) with the other counters untouched (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4, lgkmcnt 11:8): at most N of this wave's DMA instructions still in flight.
template <int N> __device__ __forceinline__ void wait_dma() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// One operand of the block tile: where its DMA lanes fetch from and where a wave's MFMA
// operand reads land.
template <typename T, int ROWS, int MODE> struct DmaOperand {
  static constexpr int ES = sizeof(T);
  static constexpr bool F32 = ES == 4;
  static constexpr int NI = ROWS / 32;                        // DMA instructions per wave and K-step
  static constexpr int TILES = ROWS / 64;                     // MFMA tiles per wave along this operand
  // LDS reads per sub-step
  static constexpr int READS = MODE == DMA_K ? TILES : (F32 ? 4 * TILES : 2 * TILES);
  static constexpr int NADDR = MODE == DMA_K ? TILES * 4 : TILES * 2;
  static constexpr int ROWB = ROWS * ES;                      // bytes per k-row (DMA_MN layout)
  static constexpr int BYTES = ROWS * 128;                    // per stage
  // fp16 DMA_MN: the swizzle permutes the ROWS / 8 slots of a k-row inside aligned groups of
  // MN_SWZ_MASK + 1 (a divisor of ROWS / 8 also when that is not a power of two)
  static constexpr uint32_t MN_SWZ_MASK = ((ROWS / 8) & (ROWS / 8 - 1)) == 0 ? ROWS / 8 - 1 : 7;
  static_assert(ROWS % 64 == 0 && (ROWS / 8) % (MN_SWZ_MASK + 1) == 0, "unsupported tile extent");

  uint32_t goff[NI];     // byte offset of this lane's 16-byte piece for DMA instruction i (k = 0)
  uint32_t kstride;      // bytes per unit of k
  uint32_t raddr[NADDR]; // byte offsets (inside the operand's LDS region) of the MFMA operand reads

  // `limit` (edge kernels): extent of this operand along M / N. Rows or 16-byte pieces past it
  // are fetched from the last valid row / piece instead: they only feed outputs that are
  // never stored. 0 = no clamping.
  __device__ __forceinline__ void init(uint32_t rs, uint32_t cs, uint32_t r0, uint32_t woff, uint32_t limit) {
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (MODE == DMA_K) {
      kstride = ES;
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const uint32_t row = (wave * NI + i) * 8 + lane / 8;
        const uint32_t c = (lane % 8) ^ swz_k(row);
        uint32_t grow = r0 + row;
        if (limit && grow >= limit) grow = limit - 1;
        goff[i] = grow * rs * ES + c * 16;
      }
      const uint32_t lrow = lane & 31, lgrp = lane >> 5;
#pragma unroll
      for (int q = 0; q < TILES; q++) {
        const uint32_t r = woff + q * 32 + lrow;
#pragma unroll
        for (int s = 0; s < 4; s++) raddr[q * 4 + s] = r * 128 + (((2 * s + lgrp) ^ swz_k(r)) * 16);
      }
    } else if (F32) {
      // [32 k][ROWS floats]; the 128-byte halves of every 256 bytes swap places in k-rows
      // with bit 2 set: an MFMA operand read touches rows k and k + 4, 32 floats of each
      // (the instructions of a K-slice cover its pieces in order, 64 each: a k-row need not be a
      // whole number of instructions)
      constexpr uint32_t PIECES = ROWB / 16;  // 16-byte pieces per k-row
      static_assert(!F32 || PIECES % 16 == 0, "the swap permutes pieces inside aligned groups of 16");
      kstride = cs * ES;
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const uint32_t flat = (wave * NI + i) * 64 + lane;
        const uint32_t krow = flat / PIECES;
        const uint32_t piece = (flat % PIECES) ^ (((krow >> 2) & 1u) << 3);
        uint32_t col = r0 + piece * 4;
        if (limit && col + 4 > limit) col = limit - 4;
        goff[i] = (krow * cs + col) * ES;
      }
      const uint32_t lrow = lane & 31, lgrp = lane >> 5;
#pragma unroll
      for (int q = 0; q < TILES; q++) {
        const uint32_t n = woff + q * 32 + lrow;  // k = 4 * lgrp + e + 8 * s, e and s as immediates
        raddr[q] = 4 * lgrp * ROWB + ((n ^ (lgrp << 5)) * 4);
      }
    } else {
      constexpr uint32_t SLOTS_PER_ROW = ROWS / 8;
      kstride = cs * 2;
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const uint32_t flat = (wave * NI + i) * 64 + lane;
        const uint32_t krow = flat / SLOTS_PER_ROW;
        const uint32_t slot = (flat % SLOTS_PER_ROW) ^ (swz_mn(krow) & MN_SWZ_MASK);
        uint32_t col = r0 + slot * 8;
        if (limit && col + 8 > limit) col = limit - 8;
        goff[i] = (krow * cs + col) * 2;
      }
      const uint32_t j = lane >> 4, r16 = lane & 15;
#pragma unroll
      for (int q = 0; q < TILES; q++) {
        const uint32_t m = woff + q * 32 + 16 * (j & 1) + 4 * (r16 & 3);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint32_t k = 8 * (j >> 1) + 4 * h + (r16 >> 2);  // + 16 * s as an immediate offset
          raddr[q * 2 + h] = k * ROWB + (((m >> 3) ^ (swz_mn(k) & MN_SWZ_MASK)) * 16) + (m & 7) * 2;
        }
      }
    }
  }

  // k offset, inside a K-slice, of the piece this lane fetches with DMA instruction i
  __device__ __forceinline__ uint32_t klocal(int i) const {
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (MODE == DMA_K) {
      const uint32_t row = (wave * NI + i) * 8 + lane / 8;
      return ((lane % 8) ^ swz_k(row)) * (16 / ES);
    }
    constexpr uint32_t PER_ROW = ROWB / 16;
    return ((wave * NI + i) * 64 + lane) / PER_ROW;
  }

  // DMA instruction i of this wave for the K-slice starting at k0: 1 KiB into `region`.
  // A buffer load: the descriptor (base of the operand, no stride, range 2^32 - 16 bytes) lives
  // in scalar registers, the lane offset goes in as it is and the K offset as the scalar
  // offset, so no vector or scalar address arithmetic stands in front of the load. The host
  // keeps operands of this kernel below 4 GiB.
  // Edge kernels (kend != 0): lanes whose piece lies at k >= kend pass an offset beyond the
  // descriptor's range, which reads as zero, so the ragged last slice contributes nothing.
  __device__ __forceinline__ void dma(int i, const T* base, uint32_t k0, char* region, uint32_t kend = 0) const {
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xfffffff0u, 0x00020000);
    uint32_t off = goff[i];
    if (kend != 0 && k0 + 128 / ES > kend) {  // wave-uniform
      if (k0 + klocal(i) >= kend) off = 0xfffffff0u;
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (LDS_AS void*)(region + (wave * NI + i) * 1024), 16, off,
                                             k0 * kstride, 0, 0);
  }

  // Edge kernels: clears what the piece straddling `kend` holds beyond it (gemm_zero_piece_tail),
  // after this wave's DMA of the K-slice starting at k0 has landed in `region`.
  __device__ __forceinline__ void zero_k_tail(char* region, uint32_t k0, uint32_t kend) const {
    if (MODE != DMA_K) return;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < NI; i++)
      gemm_zero_piece_tail<T>(region + (wave * NI + i) * 1024 + lane * 16, k0 + klocal(i), kend);
  }

  // Read number u of sub-step s into the operand registers of tile u (DMA_K), half u%2 of
  // tile u/2 (DMA_MN, fp16) or element u%4 of tile u/4 (DMA_MN, fp32).
  __device__ __forceinline__ void read(int u, int s, const char* region, Chunk* frag) const {
    if (MODE == DMA_K) {
      frag[u] = *reinterpret_cast<const Chunk*>(region + raddr[u * 4 + s]);
    } else if (F32) {
      const int q = u / 4, e = u % 4;
      frag[q][e] = *reinterpret_cast<const uint32_t*>(region + raddr[q] + (8 * s + e) * ROWB);
    } else {
      const int q = u / 2, h = u % 2;
      typedef short short4v __attribute__((ext_vector_type(4)));
      const short4v v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (LDS_AS short4v*)(region + raddr[q * 2 + h] + s * 16 * ROWB));
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 w = __builtin_bit_cast(u32x2, v);
      frag[q][2 * h] = w[0];
      frag[q][2 * h + 1] = w[1];
    }
  }
};

// ONE: the whole K is a single 128-byte slice (attention scores over 64-wide heads). Nothing to
// prefetch and nothing to overlap inside the workgroup, so the variant fetches its one slice,
// multiplies and stores, with one stage of LDS (`lds1` unused): twice as many workgroups fit a CU,
// which is what hides the latencies of such a launch. (The general loop would fetch the clamped
// "next" slices into the second stage and wait for them twice before the write-out.)
// RING4: four stages instead of two (`lds2`, `lds3`), three K-slices ahead. For the small tiles
// whose workgroup has a compute unit to itself: what a K-step of such a tile costs is mostly fixed
// (waits, barrier, scalar bookkeeping: the four-stage pipeline of 64-byte slices spends about 275
// cycles per slice on a 64 x 64 tile, of which the MFMAs are 128), so the slices should be long,
// and with one workgroup per compute unit only a deep ring keeps enough loads in flight.
// kchunk (the third build, see the kernels at the end): the workgroup multiplies the kchunk values of K from i * kchunk on, i = blockIdx.y or, of a
// group, blockIdx.y % parts, and stores TO = float; 0: all of K. CHAIN: the workgroup takes one part after the other and adds them up like the launch
// that follows the parts, in the same order: the same bits.
template <typename T, int BM, int BN, int MODE_A, int MODE_B, bool EDGE, bool ONE = false, bool RING4 = false, typename TO = T, bool GROUP = false, bool CHAIN = false>
__device__ __forceinline__ void gemm_dma2_impl(const hck_gemm_args& p, char* lds0, char* lds1, char* lds2 = nullptr,
                                               char* lds3 = nullptr, const uint32_t kchunk = 0, const uint32_t parts = 1) {
  static_assert(!(ONE && RING4), "one slice needs no ring");
  constexpr int MT = BM / 64, NT = BN / 64;
  constexpr int SLOTS = MT * NT;
  typedef DmaOperand<T, BM, MODE_A> OpA;
  typedef DmaOperand<T, BN, MODE_B> OpB;
  constexpr bool F32 = sizeof(T) == 4, F32_OUT = sizeof(TO) == 4;
  constexpr uint32_t BK = 128 / sizeof(T);  // K-slice of one stage
  constexpr int READS = OpA::READS + OpB::READS;
  constexpr int NDMA = OpA::NI + OpB::NI;  // per wave and K-step
  constexpr int HALF = NDMA / 2;
  constexpr int A_BYTES = OpA::BYTES;

  uint32_t tm, tn;
  uint32_t block_in_product, batch_of_block;
  gemm_block_and_batch(block_in_product, batch_of_block);
  gemm_tile_of_block(p, block_in_product, tm, tn);
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  const uint32_t batch = batch_of_block;
#ifdef HC_GEMM_MERGED
  // (the second build of this file, kernels *_m: what a recording's rewrite needs)
  uint32_t batch_hi = batch, batch_lo = 0;
  if (p.bdiv != 0) {
    batch_hi = batch / p.bdiv;
    batch_lo = batch - batch_hi * p.bdiv;
  }
  const T* A = (const T*)p.a + batch_hi * p.a_bs + batch_lo * p.a_bs2;
  const T* B = (const T*)p.b + batch_hi * p.b_bs + batch_lo * p.b_bs2;
  T* C = (T*)p.c + batch_hi * p.c_bs + batch_lo * p.c_bs2;
  if (p.group != 0) {  // a member of a group of products over the same A
    A = (const T*)p.a;
    B = (const T*)gemm_table_entry(p.g_b, batch);
    C = (T*)gemm_table_entry(p.g_c, batch);
  }
  const void* const ep_p0 = gemm_epilogue_operand(p, 0, batch);
  const void* const ep_p1 = gemm_epilogue_operand(p, 1, batch);
  const void* const ep_p2 = gemm_epilogue_operand(p, 2, batch);
  const uint32_t K = p.K;
#elif defined(HC_GEMM_PARTS)
  const uint32_t member = GROUP ? batch / parts : 0, part = batch - member * parts;
  const T* A = (const T*)p.a + part * p.a_bs;
  const T* B = (const T*)(GROUP ? gemm_table_entry(p.g_b, member) : p.b) + part * p.b_bs;
  TO* C = (TO*)(GROUP ? gemm_table_entry(p.g_c, member) : p.c) + part * p.c_bs;
  const uint32_t K = min(p.K - part * kchunk, kchunk);
#else
  const T* A = (const T*)p.a + batch * p.a_bs;
  const T* B = (const T*)p.b + batch * p.b_bs;
  TO* C = (TO*)p.c + batch * p.c_bs;
  const uint32_t K = p.K;
#endif

  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  const uint32_t lrow = lane & 31, lgrp = lane >> 5;

  floatx16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;

  OpA oa;
  OpB ob;
  oa.init(p.a_rs, p.a_cs, m0, wm, EDGE ? p.a_lim : 0);
  ob.init(p.b_cs, p.b_rs, n0, wn, EDGE ? p.b_lim : 0);
  const uint32_t kend = EDGE ? K : 0;

  struct Frags {
    Chunk a[MT];
    Chunk b[NT];
  };
  // unit u of the operand reads of a sub-step: B's reads first, then A's
  auto read_unit = [&](Frags& f, const char* stage, int s, int u) {
    if (u < OpB::READS) ob.read(u, s, stage + A_BYTES, f.b);
    else if (u < READS) oa.read(u - OpB::READS, s, stage, f.a);
  };
  // unit u of the DMA of the K-slice starting at k0
  // `tail`: a compile-time flag. Only the last K-slice can be ragged, so only the DMA that may
  // fetch it carries the range check of the edge kernels (a scalar compare and a branch in
  // front of every DMA instruction otherwise, in the middle of the MFMA stream).
  auto dma_unit = [&](auto tail, int u, uint32_t k0, char* stage) {
    const uint32_t ke = decltype(tail)::value ? kend : 0;
    if (u < OpA::NI) oa.dma(u, A, k0, stage, ke);
    else if (u < NDMA) ob.dma(u - OpA::NI, B, k0, stage + A_BYTES, ke);
  };
  typedef std::integral_constant<bool, EDGE> Tail;     // checks where the kernel has them at all
  typedef std::integral_constant<bool, false> NoTail;
  // MFMA t of a sub-step; operands swapped (B first) so that a lane holds four consecutive
  // n for one m (see the epilogue).
  auto mma_one = [&](const Frags& f, int t) {
    const int i = t / NT, j = t % NT;
    if constexpr (F32) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        // (copies first: a bit_cast applied directly to a vector element reads element 0)
        const uint32_t wb = f.b[j][e], wa = f.a[i][e];
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(__builtin_bit_cast(float, wb),
                                                         __builtin_bit_cast(float, wa), acc[i][j], 0, 0, 0);
      }
    } else {
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, f.b[j]),
                                                         __builtin_bit_cast(half8, f.a[i]), acc[i][j], 0, 0, 0);
    }
  };
  // reads per MFMA slot of a sub-step
  constexpr int RPS = (READS + SLOTS - 1) / SLOTS;
  // The DMA of a K-slice is spread evenly over a window of W MFMA slots that starts right
  // after the barrier that frees its stage (sub-step 3 of the step before the previous one,
  // then sub-steps 0 and 1): unit u goes out in window slot u * W / NDMA. The rest of the
  // 3 * SLOTS .. 4 * SLOTS slots before the next barrier is the time the last loads get to land.
  constexpr int W = SLOTS * HC_DMA_WINDOW_X2 / 2 > 0 ? SLOTS * HC_DMA_WINDOW_X2 / 2 : 1;
  static_assert(W <= 3 * SLOTS, "the DMA window ends with sub-step 1");
  auto window_slot = [](int u) { return u * W / NDMA; };
  // units of the first window part (sub-step 3): [0, U0)
  constexpr int U0 = (SLOTS * NDMA + W - 1) / W < NDMA ? (SLOTS * NDMA + W - 1) / W : NDMA;

  const uint32_t nk = (K + BK - 1) / BK;
  auto kclamp = [&](uint32_t j) { return (j < nk ? j : nk - 1) * BK; };  // steps past the end repeat the last one
  // (edge kernels) K is not a whole number of 16-byte pieces: the last slice of a K-contiguous
  // operand is cleaned up after it has landed
  const bool ktail = EDGE && K % (16 / sizeof(T)) != 0;
  auto zero_tail = [&](char* stage, uint32_t k0) {
    oa.zero_k_tail(stage, k0, kend);
    ob.zero_k_tail(stage + A_BYTES, k0, kend);
  };
  Frags f0, f1;

  // sub-step: MFMAs on `use`, operands of the following sub-step (number s_next of `from`)
  // into `fill`, and the DMA units of window part `part` (0, 1, 2; -1: none) of the K-slice
  // at k0 into `to`
  auto substep = [&](auto tail, const Frags& use, Frags& fill, const char* from, int s_next, int part, char* to,
                     uint32_t k0) {
#pragma unroll
    for (int t = 0; t < SLOTS; t++) {
      if (part >= 0) {
#pragma unroll
        for (int u = 0; u < NDMA; u++)
          if (window_slot(u) == part * SLOTS + t) dma_unit(tail, u, k0, to);
      }
#pragma unroll
      for (int e = 0; e < RPS; e++) read_unit(fill, from, s_next, t * RPS + e);
      mma_one(use, t);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  floatx16 sum[MT][NT];   // (CHAIN) the parts so far
  uint32_t steps_left = kchunk / BK;
  bool first_part = true;
  auto end_part = [&] {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int jj = 0; jj < NT; jj++)
#pragma unroll
        for (int v = 0; v < 16; v++) {
          sum[i][jj][v] = first_part ? acc[i][jj][v] : sum[i][jj][v] + acc[i][jj][v];
          acc[i][jj][v] = 0.0f;
        }
    first_part = false;
    steps_left = kchunk / BK;
  };

  // K-step j out of `cur`; `nxt` receives the rest of K-step j+1, then `cur` the start of j+2
  auto step = [&](auto tail, char* cur, char* nxt, uint32_t j) {
    __builtin_amdgcn_sched_barrier(0);
    substep(tail, f0, f1, cur, 1, 1, nxt, kclamp(j + 1));
    substep(tail, f1, f0, cur, 2, 2, nxt, kclamp(j + 1));
    substep(tail, f0, f1, cur, 3, -1, nullptr, 0);
    wait_dma<0>();  // K-step j+1 of this wave has landed ...
    if constexpr (decltype(tail)::value) {
      if (ktail && j + 2 == nk) zero_tail(nxt, (j + 1) * BK);
    }
    lds_barrier();  // ... and everybody's; nobody reads cur any more
    __builtin_amdgcn_sched_barrier(0);
    substep(tail, f1, f0, nxt, 0, 0, cur, kclamp(j + 2));
    if constexpr (CHAIN) {
      if (--steps_left == 0 || j + 1 == nk) end_part();
    }
  };

  // Ring of four: K-step j out of `cur`; `nxt` holds K-step j+1 once the wait passes; the stage
  // of K-step j-1 (`prev`, free since the barrier of the step before) receives K-step j+3.
  auto step4 = [&](auto tail, char* cur, char* nxt, char* prev, uint32_t j) {
    const uint32_t k3 = kclamp(j + 3);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(tail, u, k3, prev);
    substep(tail, f0, f1, cur, 1, -1, nullptr, 0);
    substep(tail, f1, f0, cur, 2, -1, nullptr, 0);
    substep(tail, f0, f1, cur, 3, -1, nullptr, 0);
    static_assert(2 * NDMA < 64, "more loads in flight than the counter holds");
    wait_dma<2 * NDMA>();  // K-step j+1 of this wave has landed (in flight: j+2 and j+3) ...
    if constexpr (decltype(tail)::value) {
      if (ktail && j + 2 == nk) zero_tail(nxt, (j + 1) * BK);
    }
    lds_barrier();  // ... and everybody's; nobody reads cur any more
    __builtin_amdgcn_sched_barrier(0);
    substep(tail, f1, f0, nxt, 0, -1, nullptr, 0);
    if constexpr (CHAIN) {
      if (--steps_left == 0 || j + 1 == nk) end_part();
    }
  };

  if constexpr (RING4) {
    // prologue: K-steps 0, 1 and 2
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(Tail{}, u, 0, lds0);
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(Tail{}, u, kclamp(1), lds1);
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(Tail{}, u, kclamp(2), lds2);
    wait_dma<2 * NDMA>();
    if constexpr (EDGE) {
      if (ktail && nk == 1) zero_tail(lds0, 0);
    }
    lds_barrier();
#pragma unroll
    for (int u = 0; u < READS; u++) read_unit(f0, lds0, 0, u);
    uint32_t j = 0;
    if constexpr (EDGE) {  // K-step j fetches slice j+3: a group of four steps from j <= nk - 8 never fetches the last slice
      for (; j + 8 <= nk; j += 4) {
        step4(NoTail{}, lds0, lds1, lds3, j);
        step4(NoTail{}, lds1, lds2, lds0, j + 1);
        step4(NoTail{}, lds2, lds3, lds1, j + 2);
        step4(NoTail{}, lds3, lds0, lds2, j + 3);
      }
    }
    for (; j + 3 < nk; j += 4) {
      step4(Tail{}, lds0, lds1, lds3, j);
      step4(Tail{}, lds1, lds2, lds0, j + 1);
      step4(Tail{}, lds2, lds3, lds1, j + 2);
      step4(Tail{}, lds3, lds0, lds2, j + 3);
    }
    if (j < nk) step4(Tail{}, lds0, lds1, lds3, j);
    if (j + 1 < nk) step4(Tail{}, lds1, lds2, lds0, j + 1);
    if (j + 2 < nk) step4(Tail{}, lds2, lds3, lds1, j + 2);
  } else if constexpr (ONE) {
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(Tail{}, u, 0, lds0);
    wait_dma<0>();
    if constexpr (EDGE) {
      if (ktail) zero_tail(lds0, 0);
    }
    lds_barrier();
#pragma unroll
    for (int u = 0; u < READS; u++) read_unit(f0, lds0, 0, u);
    substep(NoTail{}, f0, f1, lds0, 1, -1, nullptr, 0);
    substep(NoTail{}, f1, f0, lds0, 2, -1, nullptr, 0);
    substep(NoTail{}, f0, f1, lds0, 3, -1, nullptr, 0);
    substep(NoTail{}, f1, f0, lds0, 0, -1, nullptr, 0);  // (its reads repeat sub-step 0's: nobody uses them)
  } else {
    // prologue: K-step 0 and the first window part of K-step 1
#pragma unroll
    for (int u = 0; u < NDMA; u++) dma_unit(Tail{}, u, 0, lds0);
#pragma unroll
    for (int u = 0; u < U0; u++) dma_unit(Tail{}, u, kclamp(1), lds1);
    wait_dma<U0>();
    if constexpr (EDGE) {
      if (ktail && nk == 1) zero_tail(lds0, 0);
    }
    lds_barrier();
#pragma unroll
    for (int u = 0; u < READS; u++) read_unit(f0, lds0, 0, u);

    uint32_t j = 0;
    if constexpr (EDGE) {  // K-step j fetches slices j+1 and j+2: up to j = nk-4 the last slice is not among them
      for (; j + 5 <= nk; j += 2) {
        step(NoTail{}, lds0, lds1, j);
        step(NoTail{}, lds1, lds0, j + 1);
      }
    }
    for (; j + 1 < nk; j += 2) {
      step(Tail{}, lds0, lds1, j);
      step(Tail{}, lds1, lds0, j + 1);
    }
    if (j < nk) step(Tail{}, lds0, lds1, j);
  }
  if constexpr (CHAIN) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int jj = 0; jj < NT; jj++) acc[i][jj] = sum[i][jj];
  }
  wait_dma<0>();  // no LDS write of this workgroup may be in flight when it ends

  // Epilogue. With the operands swapped, the MFMA tile is C^T: lane l holds m = l % 32 and,
  // in registers 4g..4g+3, the four consecutive columns n = 8g + 4*(l/32) + (0..3). Stored
  // directly that would be short pieces of 32 different rows per instruction, so the wave's
  // part of C goes through LDS in slabs of 32 rows (both stages are free now; wave w uses
  // half of a stage) and leaves as 16-byte pieces, whole rows of the slab contiguous. 16-byte unit u
  // of row r sits at unit u ^ s(r) to spread the column-wise writes over the banks. A wave's
  // LDS instructions execute in order, so a slab may be overwritten right after its reads.
  lds_barrier();
  constexpr uint32_t MINE = ONE ? (BM + BN) * 32 : (BM + BN) * 64;  // bytes of LDS per wave for the write-out
  char* mine = ONE ? lds0 + wave * MINE : (wave < 2 ? lds0 : lds1) + (wave & 1) * MINE;
  constexpr uint32_t ES = sizeof(TO), WN = BN / 2, RB = WN * ES, UNITS = RB / 16;
  constexpr uint32_t SLAB = 32 * RB, NSLAB = MINE / SLAB;
  static_assert(NSLAB >= 1 && (32 * UNITS) % 64 == 0, "a slab must fit half a stage");
  // (the swizzle stays inside aligned groups of USWZ + 1 units, a divisor of UNITS)
  constexpr uint32_t USWZ = (UNITS & (UNITS - 1)) == 0 ? UNITS - 1 : (UNITS % 8 == 0 ? 7 : 3);
  static_assert(UNITS % (USWZ + 1) == 0, "unsupported tile width");
  auto unit_swz = [&](uint32_t r) { return (RB >= 256 ? r : r * RB / 256) & USWZ; };
#ifdef HC_GEMM_MERGED
  // (operations merged into this product: if 64 lanes are whole rows of units, a lane's columns
  // are the same for all its pieces and the row operands are fetched once)
  constexpr bool EP_COL_FIXED = 64 % UNITS == 0;
  const uint32_t ep_col = n0 + wn + (lane % UNITS) * (16 / ES);
  Chunk ep_r0 = Chunk{}, ep_r1 = Chunk{}, ep_r2 = Chunk{};
  if (EP_COL_FIXED && p.ep_kind[0] != HCK_EP_NONE) {
    const bool ok = !EDGE || ep_col < p.N;
    ep_r0 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[0], ep_p0, ep_col, ok);
    ep_r1 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[1], ep_p1, ep_col, ok);
    ep_r2 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[2], ep_p2, ep_col, ok);
  }
#endif
  // One copy of the write-out per kind of epilogue (MODE 0: plain stores; 1: merged additions; 2:
  // with a matrix operand; 3: additions and GELU). The plain one is all that the kernels of the
  // ordinary build contain; the kernels a recording's rewrite uses are a second build of this file
  // (HC_GEMM_MERGED, names ending in _m) that picks the mode per launch and also knows two-level
  // batches and groups of products. Kept apart on purpose: with the merged code in the same kernel
  // the plain fp16 4096^3 product ran 7 % slower (1216 against 1313 TFLOP/s on the same device, same
  // main loop instruction for instruction), and where the plain path shared blocks with code that
  // loads, the compiler guarded those loads' registers with waits that, at run time, wait for the
  // plain path's own stores (one in-order counter for loads and stores).
#ifdef HC_GEMM_MERGED
  auto write_out = [&](auto mode_c) {
    constexpr int MODE = decltype(mode_c)::value;
#else
  {
    constexpr int MODE = 0;
#endif
#pragma unroll
    for (int i = 0; i < MT; i++) {
      char* slab = mine + (i % NSLAB) * SLAB;
#pragma unroll
      for (int j = 0; j < NT; j++) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          if constexpr (F32_OUT) {
            floatx4 h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = acc[i][j][4 * g + e];
            *reinterpret_cast<floatx4*>(slab + lrow * RB + (((j * 8 + 2 * g + lgrp) ^ unit_swz(lrow)) * 16)) = h;
          } else {
            half4v h;
#pragma unroll
            for (int e = 0; e < 4; e++) h[e] = narrow<half_t>(acc[i][j][4 * g + e]);
            *reinterpret_cast<half4v*>(slab + lrow * RB + (((j * 4 + g) ^ unit_swz(lrow)) * 16) + lgrp * 8) = h;
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private region: no barrier needed
      if constexpr (MODE == 0) {
#pragma unroll
        for (uint32_t it = 0; it < 32 * UNITS / 64; it++) {
          const uint32_t piece = it * 64 + lane, r = piece / UNITS, u = piece % UNITS;
          const Chunk v = *reinterpret_cast<const Chunk*>(slab + r * RB + ((u ^ unit_swz(r)) * 16));
          const uint32_t row = m0 + wm + i * 32 + r, col = n0 + wn + u * (16 / ES);
          gemm_store_piece<TO, Chunk, EDGE, gemm_loose_stores<EDGE, BM, BN>()>(C + (size_t)row * p.c_rs + col, row, col, p.M, p.N, v, slab + r * RB + ((u ^ unit_swz(r)) * 16));
        }
      }
#ifdef HC_GEMM_MERGED
      if constexpr (MODE != 0) {
        gemm_store_slab_merged_as<T, Chunk, EDGE, 32 * UNITS / 64, EP_COL_FIXED, (MODE == 3 ? 1 : 4), MODE == 2, MODE == 3>(
            p, ep_p0, ep_p1, ep_p2, ep_r0, ep_r1, ep_r2, C,
            [=](uint32_t it) {
              const uint32_t piece = it * 64 + lane, r = piece / UNITS, u = piece % UNITS;
              return *reinterpret_cast<const Chunk*>(slab + r * RB + ((u ^ unit_swz(r)) * 16));
            },
            [=](uint32_t it) { return m0 + wm + i * 32 + (it * 64 + lane) / UNITS; },
            [=](uint32_t it) { return n0 + wn + ((it * 64 + lane) % UNITS) * (16 / ES); });
      }
#endif
      asm volatile("" ::: "memory");
    }
#ifdef HC_GEMM_MERGED
  };
  const bool ep_matrix = p.ep_kind[0] == HCK_EP_ADD_MATRIX || p.ep_kind[1] == HCK_EP_ADD_MATRIX || p.ep_kind[2] == HCK_EP_ADD_MATRIX;
  const bool ep_gelu = p.ep_kind[0] == HCK_EP_GELU || p.ep_kind[1] == HCK_EP_GELU || p.ep_kind[2] == HCK_EP_GELU;
  if (p.ep_kind[0] == HCK_EP_NONE) write_out(std::integral_constant<int, 0>{});
  else if (ep_gelu) write_out(std::integral_constant<int, 3>{});
  else if (ep_matrix) write_out(std::integral_constant<int, 2>{});
  else write_out(std::integral_constant<int, 1>{});
#else
  }
#endif
}

// Two variants per kernel: whole tiles only, and "_e" (edge) for M, N that are not multiples of
// the tile and K that is not a multiple of the K-slice (64 halfs, 32 floats).
#ifdef HC_GEMM_MERGED
#define HC_GEMM_NAME(base) base##_m
#else
#define HC_GEMM_NAME(base) base
#endif
#define DEF_DMA(T, TN, BM, BN, AN, AM, BNAME, BMODE)                                                  \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds1[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, false>(p, lds0, lds1);                                       \
  }                                                                                                   \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME##_e)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds1[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, true>(p, lds0, lds1);                                        \
  }
#define DEF_DMA_ONE(T, TN, BM, BN, AN, AM, BNAME, BMODE)                                              \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME##_1)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, false, true>(p, lds0, nullptr);                              \
  }                                                                                                   \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME##_1_e)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, true, true>(p, lds0, nullptr);                               \
  }
// (every stage a __shared__ array of its own: the compiler then knows that a DMA into one stage does
// not touch the stage a read comes from)
#define DEF_DMA_RING4(T, TN, BM, BN, AN, AM, BNAME, BMODE)                                            \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME##_r4)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds1[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds2[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds3[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, false, false, true>(p, lds0, lds1, lds2, lds3);              \
  }                                                                                                   \
  extern "C" __global__ __launch_bounds__(256) void HC_GEMM_NAME(hc_gemm_##TN##_dma2_##BM##x##BN##_##AN##BNAME##_r4_e)( \
      hck_gemm_args p) {                                                                              \
    __shared__ __attribute__((aligned(1024))) char lds0[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds1[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds2[(BM + BN) * 128];                             \
    __shared__ __attribute__((aligned(1024))) char lds3[(BM + BN) * 128];                             \
    gemm_dma2_impl<T, BM, BN, AM, BMODE, true, false, true>(p, lds0, lds1, lds2, lds3);               \
  }
#ifdef HC_GEMM_PARTS
// Products of few tiles over a long K: as many workgroups as compute units, each a tile over a part of K (blockIdx.y) into fp32 partial
// sums, which a second launch adds up, parts in order. 64 x 64 tiles fetch whole cache lines, so that a part of K takes little
// longer than its bytes need.
// Groups (_g) in kernels of their own: what tells a member from its part costs 0.35 us where it is not wanted, and two stages leave room for
// the workgroups of all members side by side.
#define DEF_PART(T, TN, AN, AM, BNAME, BMODE, E, SUFFIX)                                              \
  extern "C" __global__ __launch_bounds__(256) void hc_gemm_##TN##_part_64x64_##AN##BNAME##SUFFIX(hck_gemm_part_args p) { \
    __shared__ __attribute__((aligned(1024))) char lds0[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds1[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds2[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds3[128 * 128];                                   \
    gemm_dma2_impl<T, 64, 64, AM, BMODE, E, false, true, float>(p.g, lds0, lds1, lds2, lds3, p.kchunk, p.parts); \
  }                                                                                                   \
  extern "C" __global__ __launch_bounds__(256) void hc_gemm_##TN##_part_64x64_##AN##BNAME##SUFFIX##_g(hck_gemm_part_args p) { \
    __shared__ __attribute__((aligned(1024))) char lds0[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds1[128 * 128];                                   \
    gemm_dma2_impl<T, 64, 64, AM, BMODE, E, false, false, float, true>(p.g, lds0, lds1, nullptr, nullptr, p.kchunk, p.parts); \
  }
#define DEF_PART_LAYOUT(T, TN, AN, AM, BNAME, BMODE) \
  DEF_PART(T, TN, AN, AM, BNAME, BMODE, false, )     \
  DEF_PART(T, TN, AN, AM, BNAME, BMODE, true, _e)
#define DEF_PARTS(T, TN)                          \
  DEF_PART_LAYOUT(T, TN, k, DMA_K, k, DMA_K)      \
  DEF_PART_LAYOUT(T, TN, k, DMA_K, n, DMA_MN)     \
  DEF_PART_LAYOUT(T, TN, m, DMA_MN, k, DMA_K)     \
  DEF_PART_LAYOUT(T, TN, m, DMA_MN, n, DMA_MN)
DEF_PARTS(half_t, f16)
DEF_PARTS(float, f32)

// A lane adds up four neighbouring outputs (a row of partial sums is a whole number of those), loads of four parts at a time on their way.
template <typename T> __device__ __forceinline__ void gemm_part_sum(const hck_gemm_part_sum_args& p, const void* sums, uint32_t q, T (&y)[4]) {
  const size_t part = (size_t)p.g.M * (p.ld / 4);
  const floatx4* src = (const floatx4*)sums + q;
  floatx4 s = src[0];
  uint32_t i = 1;
  for (; i + 4 <= p.parts; i += 4) {
    floatx4 v[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) v[u] = src[(i + u) * part];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) s += v[u];
  }
  for (; i < p.parts; i++) s += src[i * part];
#pragma unroll
  for (int x = 0; x < 4; x++) y[x] = narrow<T>(s[x]);
}
template <typename T> __device__ __forceinline__ void gemm_part_sum_impl(const hck_gemm_part_sum_args& p) {
  const uint32_t per_row = p.ld / 4, q = blockIdx.x * HCK_BLOCK + threadIdx.x;
  if (q >= p.g.M * per_row) return;
  const uint32_t row = q / per_row, col = (q - row * per_row) * 4;
  T y[4];
  gemm_part_sum<T>(p, p.sums, q, y);
  T* dst = (T*)p.g.c + (size_t)row * p.g.c_rs + col;
  if (col + 4 <= p.g.N) {
    store_vec_loose<T, 4>(dst, y);
  } else {
#pragma unroll
    for (uint32_t x = 0; x < 3; x++)
      if (col + x < p.g.N) dst[x] = y[x];
  }
}
extern "C" __global__ __launch_bounds__(HCK_BLOCK) void hc_gemm_part_sum_f16(hck_gemm_part_sum_args p) { gemm_part_sum_impl<half_t>(p); }
extern "C" __global__ __launch_bounds__(HCK_BLOCK) void hc_gemm_part_sum_f32(hck_gemm_part_sum_args p) { gemm_part_sum_impl<float>(p); }

// The same with what a recording merged into the product, and for a group of products (only with rows of C of whole 16-byte pieces): one of three bodies per
// launch like the tiled kernels' write-out, the operands' loads in front of those of the partial sums. Product, bias and residual, fp16, us,
// one launch without parts / parts with the operations launched apart / this: 16 x 3072 x 768 11.5 / 12.7 / 8.9, 512 x 4096 x 1024
// 18.6 / 22.1 / 17.6.
template <typename T, bool MATRIX, bool GELU> __device__ __forceinline__ void gemm_part_sum_merged_as(const hck_gemm_part_sum_args& p) {
  typedef uint32_t Piece __attribute__((ext_vector_type(sizeof(T))));   // four outputs
  const uint32_t per_row = p.ld / 4, q = blockIdx.x * HCK_BLOCK + threadIdx.x;
  if (q >= p.g.M * per_row) return;
  const uint32_t row = q / per_row, col = (q - row * per_row) * 4;
  const uint32_t member = blockIdx.y;
  const bool grouped = p.g.group != 0;
  const void *p0 = gemm_epilogue_operand(p.g, 0, member), *p1 = gemm_epilogue_operand(p.g, 1, member), *p2 = gemm_epilogue_operand(p.g, 2, member);
  T* c = (T*)(grouped ? gemm_table_entry(p.g.g_c, member) : p.g.c);
  const Piece r0 = gemm_epilogue_row_piece<T, Piece>(p.g.ep_kind[0], p0, col, true), r1 = gemm_epilogue_row_piece<T, Piece>(p.g.ep_kind[1], p1, col, true),
              r2 = gemm_epilogue_row_piece<T, Piece>(p.g.ep_kind[2], p2, col, true);
  Piece m = Piece{};
  if (MATRIX) m = gemm_epilogue_matrix_piece<T, Piece>(p.g, p0, p1, p2, row, col);
  T y[4];
  gemm_part_sum<T>(p, grouped ? gemm_table_entry(p.g_sums, member) : p.sums, q, y);
  Piece v;
  __builtin_memcpy(&v, y, sizeof(v));
  *reinterpret_cast<Piece*>(c + (size_t)row * p.g.c_rs + col) = gemm_epilogue_apply<T, Piece, MATRIX, GELU>(p.g, v, r0, r1, r2, m);
}
template <typename T> __device__ __forceinline__ void gemm_part_sum_merged(const hck_gemm_part_sum_args& p) {
  const uint32_t k0 = p.g.ep_kind[0], k1 = p.g.ep_kind[1], k2 = p.g.ep_kind[2];
  if (k0 == HCK_EP_GELU || k1 == HCK_EP_GELU || k2 == HCK_EP_GELU) gemm_part_sum_merged_as<T, false, true>(p);
  else if (k0 == HCK_EP_ADD_MATRIX || k1 == HCK_EP_ADD_MATRIX || k2 == HCK_EP_ADD_MATRIX) gemm_part_sum_merged_as<T, true, false>(p);
  else gemm_part_sum_merged_as<T, false, false>(p);
}
extern "C" __global__ __launch_bounds__(HCK_BLOCK) void hc_gemm_part_sum_f16_m(hck_gemm_part_sum_args p) { gemm_part_sum_merged<half_t>(p); }
extern "C" __global__ __launch_bounds__(HCK_BLOCK) void hc_gemm_part_sum_f32_m(hck_gemm_part_sum_args p) { gemm_part_sum_merged<float>(p); }
#elif defined(HC_GEMM_CHAINS)
// Groups of fp16 products in parts of K whose tiles keep most of the device busy by themselves (the host's rule and figures: fuse_product_groups). Built with
// what the second build has: the write-out takes what a recording merged.
#define DEF_CHAIN(AN, AM, BNAME, BMODE, E, SUFFIX)                                                    \
  extern "C" __global__ __launch_bounds__(256) void hc_gemm_f16_chain_64x64_##AN##BNAME##SUFFIX##_m(hck_gemm_part_args p) { \
    __shared__ __attribute__((aligned(1024))) char lds0[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds1[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds2[128 * 128];                                   \
    __shared__ __attribute__((aligned(1024))) char lds3[128 * 128];                                   \
    gemm_dma2_impl<half_t, 64, 64, AM, BMODE, E, false, true, half_t, false, true>(p.g, lds0, lds1, lds2, lds3, p.kchunk); \
  }
#define DEF_CHAIN_LAYOUT(AN, AM, BNAME, BMODE) \
  DEF_CHAIN(AN, AM, BNAME, BMODE, false, )     \
  DEF_CHAIN(AN, AM, BNAME, BMODE, true, _e)
DEF_CHAIN_LAYOUT(k, DMA_K, k, DMA_K)
DEF_CHAIN_LAYOUT(k, DMA_K, n, DMA_MN)
DEF_CHAIN_LAYOUT(m, DMA_MN, k, DMA_K)
DEF_CHAIN_LAYOUT(m, DMA_MN, n, DMA_MN)
#else
#define DEF_DMA_RING4_TILE(T, TN, BM, BN)                                                             \
  DEF_DMA_RING4(T, TN, BM, BN, k, DMA_K, k, DMA_K)                                                    \
  DEF_DMA_RING4(T, TN, BM, BN, k, DMA_K, n, DMA_MN)                                                   \
  DEF_DMA_RING4(T, TN, BM, BN, m, DMA_MN, k, DMA_K)                                                   \
  DEF_DMA_RING4(T, TN, BM, BN, m, DMA_MN, n, DMA_MN)
// (single-slice variants: layouts with an operand that is contiguous along K, the only ones the host
// sends here)
#define DEF_DMA_ONE_TILE(T, TN, BM, BN)                                                               \
  DEF_DMA_ONE(T, TN, BM, BN, k, DMA_K, k, DMA_K)                                                      \
  DEF_DMA_ONE(T, TN, BM, BN, k, DMA_K, n, DMA_MN)                                                     \
  DEF_DMA_ONE(T, TN, BM, BN, m, DMA_MN, k, DMA_K)
#define DEF_DMA_TILE(T, TN, BM, BN)                                                                   \
  DEF_DMA(T, TN, BM, BN, k, DMA_K, k, DMA_K)                                                          \
  DEF_DMA(T, TN, BM, BN, k, DMA_K, n, DMA_MN)                                                         \
  DEF_DMA(T, TN, BM, BN, m, DMA_MN, k, DMA_K)                                                         \
  DEF_DMA(T, TN, BM, BN, m, DMA_MN, n, DMA_MN)
#define DEF_DMA_TYPE(T, TN)                                                                           \
  DEF_DMA_TILE(T, TN, 256, 256)                                                                       \
  DEF_DMA_TILE(T, TN, 256, 128)                                                                       \
  DEF_DMA_TILE(T, TN, 128, 128)                                                                       \
  DEF_DMA_TILE(T, TN, 256, 64)                                                                        \
  DEF_DMA_TILE(T, TN, 128, 64)                                                                        \
  DEF_DMA_TILE(T, TN, 64, 64)
// HC_GEMM_ONLY=16 / 32: the fp16 / fp32 kernels only (the second build of this file is compiled as two
// code objects side by side; as one it was the longest step of the whole build)
#if !defined(HC_GEMM_ONLY) || HC_GEMM_ONLY == 16
DEF_DMA_TYPE(half_t, f16)
// (fp16, the two smallest tiles: 2048 x 2048 x 512 on 64 x 64 tiles 11.9 -> 9.7 us, 512 x 4096 x 512
// 19.1 -> 15.0; 128 x 128 tiles and fp32 gain nothing from it)
DEF_DMA_RING4_TILE(half_t, f16, 128, 64)
DEF_DMA_RING4_TILE(half_t, f16, 64, 64)
DEF_DMA_ONE_TILE(half_t, f16, 256, 128)
DEF_DMA_ONE_TILE(half_t, f16, 128, 128)
DEF_DMA_ONE_TILE(half_t, f16, 128, 64)
DEF_DMA_ONE_TILE(half_t, f16, 64, 64)
#endif
#if !defined(HC_GEMM_ONLY) || HC_GEMM_ONLY == 32
DEF_DMA_TYPE(float, f32)
DEF_DMA_ONE_TILE(float, f32, 256, 128)
DEF_DMA_ONE_TILE(float, f32, 128, 128)
DEF_DMA_ONE_TILE(float, f32, 128, 64)
DEF_DMA_ONE_TILE(float, f32, 64, 64)
// (extents that are not powers of two: fp32 only, fp16 has them on the 16x16x32 pipeline)
DEF_DMA_TILE(float, f32, 256, 192)
DEF_DMA_TILE(float, f32, 192, 256)
DEF_DMA_TILE(float, f32, 192, 192)
#endif
#endif   // HC_GEMM_PARTS, HC_GEMM_CHAINS
