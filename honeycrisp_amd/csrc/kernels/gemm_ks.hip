// fp16 and fp32 GEMM for gfx950 whose workgroups split K over their waves: every wave of a workgroup multiplies the
// whole MT x NT tile over its own share of K, and the W partial tiles are added up through LDS at the end, in wave order.
//
// For products with few tiles: a row or a batch of rows against a weight, small models. The tiled kernels (gemm_dma*)
// give such a product one workgroup per 64 x 64 outputs whose four waves walk all of K together: 16 x 4096 x 4096 is 64
// workgroups on 256 compute units, and the time is K steps times the latency of one (fp32: times the 64 cycles per pair
// of k of the matrix instruction). Here tiles are as small as 16 x 32 and K is cut in 4 or 8 without a second launch or
// memory traffic for partial sums. Nobody waits for anybody inside the K loop: no barriers, a wave's operands are its own.
// (Cutting K over workgroups instead, the last of a tile adding up fp32 tiles left in memory, was built and measured:
// storing, counting and fetching cost 4 us per product, more than it gave on all but a few shapes.)
// What bounds them: the 1 KiB loads (18 to 21 cycles of a compute unit's address path each) and the latency of the
// first ones; one narrower than 16 bytes per lane costs nearly as much, which is why operands that are contiguous along
// M / N go through LDS. Measured in us, launch included, before -> after: fp32 603 x 512 x 512 11.1 -> 7.6, 603 x 2048 x 512
// 32.4 -> 19.4, 256 x 256 x 256 6.0 -> 3.8, 128 x 1024 x 1024 17.1 -> 8.9, 16 x 4096 x 4096 60.1 -> 17.2 (64 MB: 3.9 TB/s);
// fp16 16 x 4096 x 4096 14.9 -> 13.3, 16 x 1024 x 512 5.8 -> 3.8, 32 x 512 x 512 4.4 -> 3.1.
#include "common.hip.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t Chunk __attribute__((ext_vector_type(4)));  // 16 bytes

enum { KS_K = 0, KS_MN = 1 };

#define LDS_AS __attribute__((address_space(3)))
#define KS_OUT_OF_RANGE 0xfffffff0u

// One operand of a wave's tile: ROWS of M (or N), a K block of 64 bytes (32 halfs, 16 floats): ROWS / 16 loads of 1 KiB.
//   KS_K:  contiguous along K. A lane's 16-byte piece is k = PER * g .. of row 16 q + i (lane = 16 g + i), straight into registers.
//   KS_MN: contiguous along M / N, through LDS (DMA), or, where a lane's V = ROWS / 16 elements are 16 bytes (fp32, 64 rows), straight into registers.
template <typename T, int ROWS, int MODE> struct KsOperand {
  static constexpr int ES = sizeof(T);
  static constexpr bool F32 = ES == 4;
  static constexpr int V = ROWS / 16;
  static constexpr int PER = 16 / ES;            // k per lane and block
  static constexpr int KB = 4 * PER;             // k per block
  static constexpr bool LDS = MODE == KS_MN && V * ES != 16;
  static constexpr int BYTES = LDS ? KB * ROWS * ES : 0;   // LDS of a block
  static constexpr uint32_t ROWB = ROWS * ES;              // bytes of a k-row in LDS
  struct Regs {
    uint32_t w[LDS ? 1 : V][4];
  };
  uint32_t off[MODE == KS_K || LDS ? V : 4];
  uint32_t raddr[LDS && !F32 ? V : 1];
  uint32_t kstride;                               // bytes per k
  const T* ptr;
  uint32_t bytes;

  // LDS: k-row number r of a block (in LDS order) holds this k
  static __device__ __forceinline__ uint32_t k_of(uint32_t r) {
    if (F32) return 4 * (r & 3) + (r >> 2);                            // r = 4 j + g: the rows of an MFMA's k = 4 g + j side by side
    return 8 * ((r >> 2) & 3) + 4 * (r >> 4) + (r & 3);                // r = 16 h + 4 g + x: likewise for a transposing read, k = 8 g + 4 h + x
  }
  // fp16: the 32-byte column group c of k-row r sits at group c ^ swz(r): the 16 rows that a transposing read touches then cover all banks evenly
  static __device__ __forceinline__ uint32_t swz(uint32_t r) { return F32 ? 0 : (r / (8 / V)) & (V - 1); }

  // rs, cs: strides along M / N and along K, in elements; `limit`: extent along M / N; rows past it are fetched
  // from the last valid ones (they only feed outputs that are never stored). loose: rows are no whole number of 16-byte
  // pieces; the last piece of the last one may reach up to 16 bytes past the operand (the host has looked).
  __device__ __forceinline__ void init(const T* base, uint32_t rs, uint32_t cs, uint32_t r0, uint32_t limit, uint32_t K, bool loose) {
    const uint32_t lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
    ptr = base;
    bytes = ((limit - 1) * rs + (K - 1) * cs + 1) * ES + (loose ? 16 : 0);
    kstride = cs * ES;
    if constexpr (MODE == KS_K) {
#pragma unroll
      for (int q = 0; q < V; q++) {
        uint32_t row = r0 + 16 * q + i16;
        if (row >= limit) row = limit - 1;
        off[q] = row * rs * ES + g * 16;
      }
    } else if constexpr (LDS) {
      constexpr uint32_t PIECES = ROWB / 16, RPI = 64 / PIECES;   // 16-byte pieces per k-row, k-rows per load
#pragma unroll
      for (int q = 0; q < V; q++) {
        const uint32_t r = q * RPI + lane / PIECES;
        uint32_t piece = lane % PIECES;
        if (!F32) piece ^= swz(r) << 1;
        uint32_t row = r0 + piece * PER;
        if (row + PER > limit) row = limit - PER;
        off[q] = row * ES + k_of(r) * kstride;
      }
      if constexpr (F32) {
        raddr[0] = g * ROWB + i16 * (V * 4);
      } else {
#pragma unroll
        for (int q = 0; q < V; q++) {
          const uint32_t r = 4 * g + (i16 >> 2);
          raddr[q] = r * ROWB + ((q ^ swz(r)) * 32) + (i16 & 3) * 8;
        }
      }
    } else {
      uint32_t row = r0 + i16 * V;
      if (row + V > limit) row = limit - V;
#pragma unroll
      for (int e = 0; e < 4; e++) off[e] = row * ES + (g * PER + e) * kstride;
    }
  }

  // The block of K that starts at k0. EK: K may not be a whole number of blocks; pieces at k >= K read as zero.
  template <bool EK> __device__ __forceinline__ void load(Regs& f, char* region, uint32_t k0, uint32_t K) const {
    const uint32_t lane = threadIdx.x & 63, g = lane >> 4;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)ptr, 0, bytes, 0x00020000);
    if constexpr (LDS) {
      constexpr uint32_t PIECES = ROWB / 16, RPI = 64 / PIECES;
#pragma unroll
      for (int q = 0; q < V; q++) {
        const bool in = !EK || k0 + k_of(q * RPI + lane / PIECES) < K;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (LDS_AS void*)(region + q * 1024), 16, in ? off[q] : KS_OUT_OF_RANGE,
                                                 k0 * kstride, 0, 0);
      }
    } else {
#pragma unroll
      for (int q = 0; q < V; q++) {
        const bool in = !EK || k0 + g * PER + (MODE == KS_K ? 0 : q) < K;
        const Chunk v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, in ? off[q] : KS_OUT_OF_RANGE, k0 * kstride, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) f.w[q][e] = v[e];
      }
    }
  }

  // Clears what the pieces of a KS_K operand that straddle K hold beyond it (the next row's first elements).
  __device__ __forceinline__ void clear_tail(Regs& f, uint32_t k0, uint32_t K) const {
    if constexpr (MODE == KS_K) {
      const uint32_t first = k0 + ((threadIdx.x & 63) >> 4) * PER;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        uint32_t keep = 0xffffffffu;
        if (F32) keep = first + e < K ? keep : 0;
        else keep = first + 2 * e + 1 < K ? keep : first + 2 * e < K ? 0xffffu : 0;
#pragma unroll
        for (int q = 0; q < V; q++) f.w[q][e] &= keep;
      }
    }
  }

  // fp32: what the tiles feed to the MFMA of k = 4 g + j
  __device__ __forceinline__ void values(const Regs& f, const char* region, int j, float (&v)[V]) const {
    if constexpr (LDS) {
      Vec<float, V> t = *reinterpret_cast<const Vec<float, V>*>(region + raddr[0] + 4 * j * ROWB);
#pragma unroll
      for (int q = 0; q < V; q++) v[q] = t.v[q];
    } else {
#pragma unroll
      for (int q = 0; q < V; q++) {
        const uint32_t w = MODE == KS_K ? f.w[q][j] : f.w[j][q];
        v[q] = __builtin_bit_cast(float, w);
      }
    }
  }
  // fp16: the eight k of tile q
  __device__ __forceinline__ half8 value8(const Regs& f, const char* region, int q) const {
    Chunk v;
    if constexpr (LDS) {
      typedef short short4v __attribute__((ext_vector_type(4)));
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const short4v t = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LDS_AS short4v*)(region + raddr[q] + h * 16 * ROWB));
        const u32x2 w = __builtin_bit_cast(u32x2, t);
        v[2 * h] = w[0], v[2 * h + 1] = w[1];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = f.w[q][e];
    }
    return __builtin_bit_cast(half8, v);
  }
  // row of the tile that index i (0 .. 15) of MFMA tile q stands for
  static constexpr bool INTERLEAVED = MODE == KS_MN && F32;
  static __device__ __forceinline__ uint32_t row_of(uint32_t q, uint32_t i) { return INTERLEAVED ? V * i + q : 16 * q + i; }
};

// Workgroup -> tile: workgroups with equal number mod 8 run on one XCD; each XCD gets a contiguous band of tiles.
__device__ __forceinline__ void ks_tile(const hck_gemm_args& p, uint32_t block, uint32_t& tm, uint32_t& tn) {
  const uint32_t tile = hck_band_tile(block, p.tiles_m * p.tiles_n);
  tm = tile / p.tiles_n;
  tn = tile - tm * p.tiles_n;
}

template <typename T, int MT, int NT, int MODE_A, int MODE_B, int W, int D, bool EK>
__device__ __forceinline__ void gemm_ks_impl(const hck_gemm_args& p, char* const (&stage)[5], float* part) {
  typedef KsOperand<T, MT, MODE_A> OpA;
  typedef KsOperand<T, NT, MODE_B> OpB;
  constexpr bool F32 = sizeof(T) == 4;
  constexpr int VA = OpA::V, VB = OpB::V;
  constexpr uint32_t KB = OpA::KB;
  constexpr uint32_t LD = NT + 4;   // floats per row of a partial tile in LDS

  uint32_t tm, tn;
  ks_tile(p, blockIdx.x, tm, tn);
  const uint32_t m0 = tm * MT, n0 = tn * NT;
  const uint32_t batch = blockIdx.y;
#ifdef HC_GEMM_MERGED
  const T* A = (const T*)p.a;
  const T* B = (const T*)p.b;
  T* C = (T*)p.c;
  if (p.group != 0) {
    B = (const T*)gemm_table_entry(p.g_b, batch);
    C = (T*)gemm_table_entry(p.g_c, batch);
  }
  const void* const ep_p0 = gemm_epilogue_operand(p, 0, batch);
  const void* const ep_p1 = gemm_epilogue_operand(p, 1, batch);
  const void* const ep_p2 = gemm_epilogue_operand(p, 2, batch);
#else
  const T* A = (const T*)p.a + batch * p.a_bs;
  const T* B = (const T*)p.b + batch * p.b_bs;
  T* C = (T*)p.c + batch * p.c_bs;
#endif
  const uint32_t lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  OpA oa;
  OpB ob;
  const bool straddles = EK && p.K % OpA::PER != 0;   // K is no whole number of pieces
  oa.init(A, p.a_rs, p.a_cs, m0, p.a_lim, p.K, EK && !HC_GEMM_IS_MERGED);
  ob.init(B, p.b_cs, p.b_rs, n0, p.b_lim, p.K, EK && !HC_GEMM_IS_MERGED);

  floatx4 acc[VA][VB];
#pragma unroll
  for (int i = 0; i < VA; i++)
#pragma unroll
    for (int j = 0; j < VB; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

  const uint32_t nk = (p.K + KB - 1) / KB;
  const uint32_t begin = wave * nk / W, end = (wave + 1) * nk / W;
  struct Frag {
    typename OpA::Regs a;
    typename OpB::Regs b;
  };
  Frag f[D];
  constexpr uint32_t SLOT = OpA::BYTES + OpB::BYTES;   // a wave's part of a stage
  auto load = [&](int d, uint32_t block) {
    char* mine = stage[d] + wave * SLOT;
    oa.template load<EK>(f[d].a, mine, block * KB, p.K);
    ob.template load<EK>(f[d].b, mine + OpA::BYTES, block * KB, p.K);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto mma = [&](int d, uint32_t block) {
    Frag& x = f[d];
    if (straddles && block + 1 == nk) oa.clear_tail(x.a, block * KB, p.K), ob.clear_tail(x.b, block * KB, p.K);
    const char* mine = stage[d] + wave * SLOT;
    if constexpr (F32) {
      float a[4][VA], b[4][VB];
#pragma unroll
      for (int e = 0; e < 4; e++) oa.values(x.a, mine, e, a[e]), ob.values(x.b, mine + OpA::BYTES, e, b[e]);
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < VA; i++)
#pragma unroll
          for (int j = 0; j < VB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e][i], b[e][j], acc[i][j], 0, 0, 0);
    } else {
      half8 a[VA], b[VB];
#pragma unroll
      for (int i = 0; i < VA; i++) a[i] = oa.value8(x.a, mine, i);
#pragma unroll
      for (int j = 0; j < VB; j++) b[j] = ob.value8(x.b, mine + OpA::BYTES, j);
#pragma unroll
      for (int i = 0; i < VA; i++)
#pragma unroll
        for (int j = 0; j < VB; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Waits until at most N of the wave's loads are in flight (only operands that go through LDS need it said; the
  // compiler counts the others itself).
  constexpr int LPB = VA + VB;
  static_assert((D - 1) * LPB < 64, "vmcnt is a 6-bit counter");
  auto landed = [&](auto n_c) {
    constexpr int N = decltype(n_c)::value;
    if constexpr (SLOT != 0) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
      asm volatile("" ::: "memory");
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  typedef std::integral_constant<int, (D - 1) * LPB> InFlight;
  typedef std::integral_constant<int, 0> None;

  // (Loads behind a condition make the compiler wait for all loads wherever it waits next, since it no longer knows
  // how many are in flight: the pipelined loop and the loads in front of it have none.)
  uint32_t j = begin;
  if (begin + 2 * D <= end) {
#pragma unroll
    for (int d = 0; d < D; d++) load(d, begin + d);
    do {
#pragma unroll
      for (int d = 0; d < D; d++) {
        landed(InFlight{});
        mma(d, j + d);
        load(d, j + d + D);
      }
      j += D;
    } while (j + 2 * D <= end);
  } else {
#pragma unroll
    for (int d = 0; d < D; d++)
      if (begin + d < end) load(d, begin + d);
  }
  // (the last one or two rounds: loads only where blocks are left, and waits for all of them)
#pragma unroll
  for (int d = 0; d < D; d++)
    if (j + d < end) {
      landed(None{});
      mma(d, j + d);
      if (j + d + D < end) load(d, j + d + D);
    }
#pragma unroll
  for (int d = 0; d < D; d++)
    if (j + D + d < end) {
      landed(None{});
      mma(d, j + D + d);
    }

  // The wave's partial tile into LDS: of tile (i, j) a lane holds rows 4 g + r (r = 0 .. 3) of column i16.
  float* mine = part + wave * (MT * LD);
#pragma unroll
  for (int i = 0; i < VA; i++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float* row = mine + OpA::row_of(i, 4 * g + r) * LD;
      if constexpr (OpB::INTERLEAVED) {
        float v[VB];
#pragma unroll
        for (int j2 = 0; j2 < VB; j2++) v[j2] = acc[i][j2][r];
        store_vec<float, VB>(row, VB * i16, v);
      } else {
#pragma unroll
        for (int j2 = 0; j2 < VB; j2++) row[OpB::row_of(j2, i16)] = acc[i][j2][r];
      }
    }
  __syncthreads();

  constexpr uint32_t PER = 16 / sizeof(T), PIECES = MT * NT / PER, ROW_PIECES = NT / PER;
#pragma unroll
  for (uint32_t it = 0; it < (PIECES + W * 64 - 1) / (W * 64); it++) {
    const uint32_t piece = it * (W * 64) + threadIdx.x;
    if (PIECES % (W * 64) != 0 && piece >= PIECES) break;
    const uint32_t r = piece / ROW_PIECES, c = piece % ROW_PIECES * PER;
    const uint32_t row = m0 + r, col = n0 + c;
    if (row >= p.M || col >= p.N) continue;
    const float* src = part + r * LD + c;
    floatx4 s[PER / 4];
#pragma unroll
    for (uint32_t x = 0; x < PER / 4; x++) s[x] = *reinterpret_cast<const floatx4*>(src + 4 * x);
#pragma unroll
    for (int w = 1; w < W; w++)
#pragma unroll
      for (uint32_t x = 0; x < PER / 4; x++) s[x] += *reinterpret_cast<const floatx4*>(src + w * (MT * LD) + 4 * x);
    T y[PER];
#pragma unroll
    for (uint32_t x = 0; x < PER; x++) y[x] = narrow<T>(s[x / 4][x % 4]);
    Chunk v;
    __builtin_memcpy(&v, y, 16);
#ifdef HC_GEMM_MERGED
    if (p.ep_kind[0] != HCK_EP_NONE) {
      const bool matrix = p.ep_kind[0] == HCK_EP_ADD_MATRIX || p.ep_kind[1] == HCK_EP_ADD_MATRIX || p.ep_kind[2] == HCK_EP_ADD_MATRIX;
      const bool gelu = p.ep_kind[0] == HCK_EP_GELU || p.ep_kind[1] == HCK_EP_GELU || p.ep_kind[2] == HCK_EP_GELU;
      const Chunk r0 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[0], ep_p0, col, true);
      const Chunk r1 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[1], ep_p1, col, true);
      const Chunk r2 = gemm_epilogue_row_piece<T, Chunk>(p.ep_kind[2], ep_p2, col, true);
      const Chunk none = Chunk{};
      if (gelu) v = gemm_epilogue_apply<T, Chunk, false, true>(p, v, r0, r1, r2, none);
      else if (matrix)
        v = gemm_epilogue_apply<T, Chunk, true, false>(p, v, r0, r1, r2,
                                                       gemm_epilogue_matrix_piece<T, Chunk>(p, ep_p0, ep_p1, ep_p2, row, col));
      else v = gemm_epilogue_apply<T, Chunk, false, false>(p, v, r0, r1, r2, none);
    }
#endif
    T* dst = C + (size_t)row * p.c_rs + col;
    if (!EK || HC_GEMM_IS_MERGED) {
      *reinterpret_cast<Chunk*>(dst) = v;
    } else if (col + PER <= p.N) {
      struct __attribute__((packed, aligned(sizeof(T)))) Loose {
        Chunk v;
      };
      reinterpret_cast<Loose*>(dst)->v = v;
    } else {
#pragma unroll
      for (uint32_t x = 0; x + 1 < PER; x++)
        if (col + x < p.N) dst[x] = y[x];
    }
  }
}

#ifdef HC_GEMM_MERGED
#define HC_GEMM_NAME(base) base##_m
#else
#define HC_GEMM_NAME(base) base
#endif
// (both operands through LDS: a stage less, so that they fit)
#define KS_DEPTH(D, AM, BM) (AM == KS_MN && BM == KS_MN ? D - 1 : D)
// (Every stage is a __shared__ array of its own: the compiler then knows that a DMA into one does not touch the one a read comes from.)
#define KS_SLOT(T, MT, NT, AM, BM) (KsOperand<T, MT, AM>::BYTES + KsOperand<T, NT, BM>::BYTES)
#define KS_STAGE(T, MT, NT, W, D, AM, BM, i) \
  __shared__ __attribute__((aligned(1024))) char st##i[i < D && KS_SLOT(T, MT, NT, AM, BM) ? W * KS_SLOT(T, MT, NT, AM, BM) : 16];
#define KS_BODY(T, MT, NT, W, D, AM, BM, EK)                                                                     \
  KS_STAGE(T, MT, NT, W, D, AM, BM, 0) KS_STAGE(T, MT, NT, W, D, AM, BM, 1) KS_STAGE(T, MT, NT, W, D, AM, BM, 2)  \
  KS_STAGE(T, MT, NT, W, D, AM, BM, 3) KS_STAGE(T, MT, NT, W, D, AM, BM, 4) \
  __shared__ __attribute__((aligned(16))) float part[W * MT * (NT + 4)];                                          \
  char* const stages[5] = {st0, st1, st2, st3, st4};                                                         \
  gemm_ks_impl<T, MT, NT, AM, BM, W, D, EK>(p, stages, part);
#define DEF_KS(T, TN, MT, NT, W, D, OCC, AN, AM, BNAME, BMODE)                                                   \
  extern "C" __global__ __launch_bounds__(W * 64, OCC) void HC_GEMM_NAME(                                         \
      hc_gemm_##TN##_ks_##MT##x##NT##_##AN##BNAME)(hck_gemm_args p) {                                      \
    KS_BODY(T, MT, NT, W, KS_DEPTH(D, AM, BMODE), AM, BMODE, false)                                                                    \
  }                                                                                                               \
  extern "C" __global__ __launch_bounds__(W * 64, OCC) void HC_GEMM_NAME(                                         \
      hc_gemm_##TN##_ks_##MT##x##NT##_##AN##BNAME##_e)(hck_gemm_args p) {                                  \
    KS_BODY(T, MT, NT, W, KS_DEPTH(D, AM, BMODE), AM, BMODE, true)                                                                     \
  }
// (OCC: wavefronts per SIMD that the registers have to leave room for)
#define DEF_KS_LAYOUTS(T, TN, MT, NT, W, D, OCC, AN, AM)     \
  DEF_KS(T, TN, MT, NT, W, D, OCC, AN, AM, k, KS_K)          \
  DEF_KS(T, TN, MT, NT, W, D, OCC, AN, AM, n, KS_MN)
#define DEF_KS_TILE(T, TN, MT, NT, W, D, OCC)                \
  DEF_KS_LAYOUTS(T, TN, MT, NT, W, D, OCC, k, KS_K)          \
  DEF_KS_LAYOUTS(T, TN, MT, NT, W, D, OCC, m, KS_MN)
// In the second build DM stages and room for OCCM wavefronts, where A is contiguous along K: a group of such products has up to four
// times the workgroups of one product, so that a compute unit has several to run, and with two stages two of them run
// side by side and hide each other's start and write-out (four stages: one, the registers). Groups of two to four 32 x 64 products
// 0.77 to 1.0 of the time on four stages, 0.87 in the mean of 20 with A along K, single ones with a row added 0.92 to 1.0; 32 x 32 0.88 to
// 1.01, 0.96 of 40: 3 x 925 x 328 x 280 16.0 -> 13.1 us, 2 x 119 x 1176 x 4024 39.2 -> 31.5, 4 x 47 x 552 x 3728 21.1 -> 19.9.
// With A along M (1.0, up to 1.07) its LDS leaves room for one workgroup anyway.
#ifdef HC_GEMM_MERGED
#define DEF_KS_TILE_M(T, TN, MT, NT, W, D, OCC, DM, OCCM)    \
  DEF_KS_LAYOUTS(T, TN, MT, NT, W, DM, OCCM, k, KS_K)        \
  DEF_KS_LAYOUTS(T, TN, MT, NT, W, D, OCC, m, KS_MN)
#else
#define DEF_KS_TILE_M(T, TN, MT, NT, W, D, OCC, DM, OCCM) DEF_KS_TILE(T, TN, MT, NT, W, D, OCC)
#endif
DEF_KS_TILE(half_t, f16, 16, 32, 8, 5, 2)
DEF_KS_TILE(float, f32, 16, 32, 8, 5, 2)
DEF_KS_TILE_M(float, f32, 32, 32, 4, 4, 2, 2, 4)
DEF_KS_TILE_M(float, f32, 32, 64, 8, 4, 2, 2, 4)
// Only for groups of products, which the second build runs: on 16 x 32 tiles a group of three has three times as many workgroups, of
// which a compute unit holds one (five stages), and runs them in rounds. This tile gives the same sums, twice the outputs per fetched
// column of B, and its two stages leave room for two workgroups. 3 products of 35 x 512 x 2176 with a bias 14.7 -> 9.7 us (four stages:
// 11.8), of 16 x 3008 x 3904 25.0 -> 22.3.
#ifdef HC_GEMM_MERGED
#define DEF_KS_GROUP_TILE DEF_KS_TILE
#define DEF_KS_GROUP_KK(T, TN, MT, NT, W, D, OCC) DEF_KS(T, TN, MT, NT, W, D, OCC, k, KS_K, k, KS_K)
#else
#define DEF_KS_GROUP_TILE(...)
#define DEF_KS_GROUP_KK(...)
#endif
DEF_KS_GROUP_TILE(half_t, f16, 32, 32, 8, 2, 4)
// Likewise for fp32 groups with both operands along K, whose loads of 16 rows' 64 bytes each bound the 32 x 64 tile: a third fewer per output.
// A workgroup fills a compute unit's LDS, so only where the group is one round of them (use_group_tile_kernel). Against 32 x 64:
// 2 x 238 x 3656 x 1968 102.5 -> 75.4 us, 3 x 43 x 2144 x 4264 51.9 -> 39.6; other layouts and more tiles gain nothing (0.97 to 1.18 in the mean).
DEF_KS_GROUP_KK(float, f32, 64, 64, 8, 2, 2)
