// The MFMA kernel of libiris_hip (fused_mfma_kernel) with the types it shares with the generic
// kernel (FusedParams, the flag helpers), its tile shapes and its launch code.  The kernel is
// instantiated for 3 input types x 5 tile shapes x 2 operand layouts (plus the one-round builds);
// each input type is compiled in a translation unit of its own (iris_hip_mfma_<type>.hip), which
// instantiates dispatch_mfma_in<IN> below, so that the build can compile them side by side.
#pragma once

#include "any_epilogue.h"

// Stages of the slot-sum pipeline of the eight-wave tile (see reduce_chunks).
#ifndef IRIS_HIP_EPILOGUE_DEPTH
#define IRIS_HIP_EPILOGUE_DEPTH 2
#endif

// ------------------------------------------------------------------------------------------------
// MFMA kernel configuration
// ------------------------------------------------------------------------------------------------
enum { IN_BF16 = 0, IN_F16 = 1, IN_FP8 = 2 };

template <int IN_, int BM_, int BN_, int BK_, int WM_, int WN_, int STAGES_, bool B_KCONTIG_>
struct MfmaCfg {
  static constexpr int IN = IN_;
  static constexpr int ES = (IN_ == IN_FP8) ? 1 : 2;
  static constexpr int CE = kChunkBytes / ES;           // elements per 16-byte chunk
  // MFMA block: 16x16x32 for 16-bit data on the eight-wave tile, else 32x32 (why: mfma_block16 below).
  static constexpr int BLK = (IN_ != IN_FP8 && WM_ * WN_ == 8) ? 16 : 32;
  static constexpr int KM = (IN_ == IN_FP8) ? 64 : BLK == 16 ? 32 : 16;  // k per MFMA
  static constexpr int QUADS = BLK * BLK / 256;         // runs of four consecutive n that a lane owns of a block
  static constexpr int BM = BM_, BN = BN_, BK = BK_, STAGES = STAGES_;
  static constexpr bool B_KCONTIG = B_KCONTIG_;
  static constexpr int WM = WM_, WN = WN_, NW = WM_ * WN_, NT = 64 * NW;
  static constexpr int TM = BM / WM, TN = BN / WN;  // per-wave block
  static constexpr int MB = TM / BLK, NB = TN / BLK;  // MFMA blocks per wave
  static constexpr int KSLICES = BK / KM;
  static constexpr int NFRAG = (IN_ == IN_FP8) ? 2 : 1;   // 16-byte pieces per operand fragment
  static constexpr int RBA = BK * ES;                        // bytes per A tile row
  static constexpr int RBB = B_KCONTIG ? BK * ES : BN * ES;  // bytes per B tile row
  static constexpr int A_BYTES = BM * RBA;
  static constexpr int B_BYTES = B_KCONTIG ? BN * RBB : BK * RBB;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int LA = A_BYTES / kDmaBytes / NW;  // direct-to-LDS loads per thread per K step
  static constexpr int LB = B_BYTES / kDmaBytes / NW;
  static constexpr int RING_BYTES = STAGES * STAGE_BYTES;
  // Epilogue staging: the whole output tile in 16-bit elements.  The accumulator-layout writes put one
  // row per lane, so rows must not start on the same LDS banks.  The four-wave tiles pad every row by 16
  // bytes and stage over the (dead) operand ring from its start.  The eight-wave tile has no LDS to
  // spare for padding: it XORs the 16-byte chunk index with the row instead, and stages above the first
  // ring slot, which leaves that slot free to take the first K step of the workgroup's NEXT tile while
  // this tile's epilogue is still streaming (160 KiB = one ring slot + the staged tile).
  static constexpr bool STAGE_SWIZZLED = (NW == 8);
  static constexpr int STAGE_OFF = STAGE_SWIZZLED ? STAGE_BYTES : 0;
  static constexpr int TROW = STAGE_SWIZZLED ? BN * 2 : BN * 2 + 16;
  static constexpr int TILE_BYTES = BM * TROW;
  static constexpr int SMEM_BYTES = RING_BYTES > STAGE_OFF + TILE_BYTES ? RING_BYTES : STAGE_OFF + TILE_BYTES;
  static_assert(SMEM_BYTES <= 160 * 1024, "LDS budget of a gfx950 CU");
  static_assert(!STAGE_SWIZZLED || ((BN / 8) & (BN / 8 - 1)) == 0, "chunk swizzle needs a power-of-two row");
  // LDS byte offset of byte `b` of row `row` of the staged tile.
  __host__ __device__ static constexpr int stage_offset(int row, int b) {
    if (STAGE_SWIZZLED) return STAGE_OFF + row * TROW + ((((b >> 4) ^ row) & (BN / 8 - 1)) << 4) + (b & 15);
    return row * TROW + b;
  }
  // The same for a place `rows` further down and `bytes` further right, from the offset of a lane's first one.  Swizzled rows:
  // the lane's row and chunk have none of the bits that rows (modulo a period of the swizzle) and bytes set, so the chunk's
  // place changes by an XOR with a constant.  (The swizzle of each of a thread's 32 places anew: 4096x4096x64 fp16 as a
  // plain product 12.3 us instead of 11.8, 16384x8192x128 102.4 instead of 96.7.)
  __host__ __device__ static constexpr int stage_step(int first, int rows, int bytes) {
    if (STAGE_SWIZZLED) return (first ^ (bytes ^ ((rows & (BN / 8 - 1)) << 4))) + rows * TROW;
    return first + rows * TROW + bytes;
  }
  static_assert(!STAGE_SWIZZLED || (TM % (BN / 8) == 0 && STAGE_OFF % TROW == 0), "places of a lane an XOR apart");
  // Four-wave tiles whose ring fits twice into a CU's LDS run two workgroups per CU, so that the
  // memory round trips of one workgroup's epilogue hide behind the other's K loop.
  static constexpr int WG_PER_CU = (NW == 4 && SMEM_BYTES <= 80 * 1024) ? 2 : 1;
  static constexpr int WAVES_PER_SIMD = WG_PER_CU * NW / 4;
  static_assert(NT % (BN / 8) == 0 && BM % (NT / (BN / 8)) == 0, "epilogue pass shape");
  static_assert(A_BYTES % (kDmaBytes * NW) == 0 && B_BYTES % (kDmaBytes * NW) == 0, "tile/loader mismatch");
  static_assert(BK % KM == 0 && TM % BLK == 0 && TN % BLK == 0, "tile/MFMA mismatch");
  static_assert(STAGES >= (NW == 8 ? 5 : 3), "ring too short for the K loop");
  static_assert((STAGES - 2) * (LA + LB) <= 63, "vmcnt field too small for this prefetch depth");
};

template <int IN>
struct OutOf { using type = OutBF16; };
template <>
struct OutOf<IN_F16> { using type = OutF16; };

// wait_vmcnt with lgkmcnt(0): every LDS read of this wave has returned as well.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4));
}

constexpr unsigned kInvalidOffset = 0x80000000u;

// Buffer resource words for a raw buffer (stride 0) over [base, base + 2^31).  Bounds are enforced
// per lane by the callers: an invalid lane presents offset 0x80000000, which is past num_records
// and therefore loads zero.
__device__ __forceinline__ i32x4_t make_rsrc_words(unsigned long long b) {
  i32x4_t r;
  r.x = __builtin_amdgcn_readfirstlane((int)(unsigned)b);
  r.y = __builtin_amdgcn_readfirstlane((int)(unsigned)(b >> 32));
  r.z = 0x7FFFFFFF;
  r.w = 0x00020000;
  return r;
}

// One wave-wide 16-byte direct-to-LDS load: lane l deposits global bytes [voff + soff, +16) of the
// buffer at LDS address lds_base + 16*l.  Written as inline assembly so that the compiler's
// wait-count pass does not serialise LDS reads behind loads that target other ring slots; the
// kernel orders them itself with wait_vmcnt() and workgroup barriers.
__device__ __forceinline__ void dma16(i32x4_t rsrc, unsigned lds_base, unsigned voff, unsigned soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_base), "v"(voff), "s"(rsrc), "s"(soff)
               : "memory");
}

// Read one accumulator register.  The "a" constraint keeps the MFMA results in the accumulation
// registers until the epilogue consumes them, instead of copying all of them to VGPRs at once.
__device__ __forceinline__ float acc_read(float a) {
  float v;
  asm("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
  return v;
}

__device__ __forceinline__ unsigned lds_address(const void* p) {
  return (unsigned)(unsigned long long)(LDS_AS const char*)p;
}

template <class CFG>
struct MfmaAcc {
  typename std::conditional<CFG::BLK == 16, f32x4_t, f32x16_t>::type v[CFG::MB][CFG::NB];
};

// Operand fragments of one k-slice for a wave's block.
template <class CFG>
struct Frags {
  i32x4_t a[CFG::MB][CFG::NFRAG];
  i32x4_t b[CFG::NB][CFG::NFRAG];
};

// One 32x32 MFMA with the operands in the order (B fragment, A fragment): the accumulator then
// holds D[n][m], i.e. each lane owns 4 consecutive n for one m.
template <int IN, int NF>
__device__ __forceinline__ f32x16_t mfma_block(const i32x4_t (&a)[NF], const i32x4_t (&b)[NF], f32x16_t c) {
  if constexpr (IN == IN_BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, b[0]),
                                                   __builtin_bit_cast(bf16x8_t, a[0]), c, 0, 0, 0);
  } else if constexpr (IN == IN_F16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, b[0]),
                                                  __builtin_bit_cast(f16x8_t, a[0]), c, 0, 0, 0);
  } else {
    i32x8_t av, bv;
    av.lo = a[0]; av.hi = a[1];
    bv.lo = b[0]; bv.hi = b[1];
    // cbsz = blgp = 0 selects e4m3 for both operands; zero scale operands select the unscaled
    // instruction (v_mfma_f32_32x32x64_f8f6f4).
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(bv, av, c, 0, 0, 0, 0, 0, 0);
  }
}

// One 16x16 MFMA of 16-bit data, operands in the same order.  The eight-wave tile multiplies with this shape: busy with
// random data, the chip runs against its power limit, and a 16x16x32 product, which reads and writes its accumulators half
// as often per flop as a 32x32x16 one, takes less of it (products from registers alone, eight waves of 128x64 per CU,
// normal bf16 operands: 1750 against 2010 TFLOP/s, 2060 with the order of quad_block; both 2400 on zeros).  The
// results are those of two 32x32x16 products, bit for bit (the same rows on both tiles, random data: tests/test_gpu_k_steps.py).
template <int IN>
__device__ __forceinline__ f32x4_t mfma_block16(const i32x4_t (&a)[1], const i32x4_t (&b)[1], f32x4_t c) {
  if constexpr (IN == IN_BF16)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b[0]), __builtin_bit_cast(bf16x8_t, a[0]), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, b[0]), __builtin_bit_cast(f16x8_t, a[0]), c, 0, 0, 0);
}

// The product a tile configuration is built on.
template <class CFG, class ACC>
__device__ __forceinline__ ACC mfma_of(const i32x4_t (&a)[CFG::NFRAG], const i32x4_t (&b)[CFG::NFRAG], ACC c) {
  if constexpr (CFG::BLK == 16) return mfma_block16<CFG::IN>(a, b, c);
  else return mfma_block<CFG::IN, CFG::NFRAG>(a, b, c);
}

// A copy of the kernel's argument block with every field materialised in registers at this point: the
// empty asm statements use the values, so their loads are issued together, up front.  Left to itself the
// compiler loads each field next to its first use and waits for it there, which put some twenty
// dependent scalar round trips in front of the first operand load of a launch.
__device__ __forceinline__ FusedParams pin_kernel_arguments(const FusedParams& a) {
  FusedParams q = a;
  asm volatile("" : "+s"(q.A), "+s"(q.B), "+s"(q.C), "+s"(q.aux), "+s"(q.locks), "+s"(q.bias), "+s"(q.heap_bases),
               "+s"(q.status), "+s"(q.spin_limit));
  asm volatile("" : "+s"(q.s_am), "+s"(q.s_ak), "+s"(q.s_bk), "+s"(q.s_bn), "+s"(q.s_cm), "+s"(q.s_cn), "+s"(q.s_bias));
  asm volatile("" : "+s"(q.M), "+s"(q.N), "+s"(q.K), "+s"(q.K_local), "+s"(q.M_local), "+s"(q.gather), "+s"(q.rank),
               "+s"(q.world), "+s"(q.flag_bm), "+s"(q.flag_bn), "+s"(q.epi), "+s"(q.acc_mode), "+s"(q.clear_c), "+s"(q.all_owners),
               "+s"(q.sum_peers), "+s"(q.bias_dtype), "+s"(q.scale));
  asm volatile("" : "+s"(q.tiles_m), "+s"(q.tiles_n), "+s"(q.group_m), "+s"(q.num_xcd), "+s"(q.row_offset),
               "+s"(q.hb_in_args));
  asm volatile("" : "+s"(q.hb_arg[0]), "+s"(q.hb_arg[1]), "+s"(q.hb_arg[2]), "+s"(q.hb_arg[3]), "+s"(q.hb_arg[4]),
               "+s"(q.hb_arg[5]), "+s"(q.hb_arg[6]), "+s"(q.hb_arg[7]));
#ifdef IRIS_HIP_PHASE_STAMPS
  asm volatile("" : "+s"(q.stamps), "+s"(q.stamp_rows));
#endif
  return q;
}

// The same for the tiled kernel, limited to what it needs before its first operand load (it has no
// registers to spare for holding the epilogue's arguments across the K loop).
__device__ __forceinline__ FusedParams pin_loader_arguments(const FusedParams& a) {
  FusedParams q = a;
  asm volatile("" : "+s"(q.A), "+s"(q.B), "+s"(q.s_am), "+s"(q.s_bk), "+s"(q.s_bn), "+s"(q.M), "+s"(q.N), "+s"(q.K),
               "+s"(q.K_local), "+s"(q.M_local), "+s"(q.gather), "+s"(q.rank), "+s"(q.world), "+s"(q.tiles_m),
               "+s"(q.tiles_n), "+s"(q.group_m), "+s"(q.num_xcd));
  return q;
}

// The staged tile of a configuration, for finish_any.  Swizzled rows keep the 16-byte chunks whole: a piece that starts inside one
// (the last of a row that is not a whole number of pieces) is put together from two of them.
template <class CFG>
struct StagedTile {
  char* base;
  __device__ __forceinline__ char* at(int row, int byte) const { return base + CFG::stage_offset(row, byte); }
  __device__ __forceinline__ u32x4_t piece(int row, int byte) const {
    if constexpr (!CFG::STAGE_SWIZZLED) {
      return *(const LDS_AS u32x4_any_t*)(LDS_AS char*)at(row, byte);
    } else {
      const u32x4_t v = *(const LDS_AS u32x4_t*)(LDS_AS char*)at(row, byte & ~15);
      if ((byte & 15) == 0) return v;
      const u32x4_t w = *(const LDS_AS u32x4_t*)(LDS_AS char*)at(row, (byte & ~15) + 16);
      const int shift = byte & 15;
      const unsigned long long lo = v[0] | (unsigned long long)v[1] << 32, hi = v[2] | (unsigned long long)v[3] << 32;
      const unsigned long long lo2 = w[0] | (unsigned long long)w[1] << 32, hi2 = w[2] | (unsigned long long)w[3] << 32;
      const unsigned long long x0 = shift < 8 ? lo : hi, x1 = shift < 8 ? hi : lo2, x2 = shift < 8 ? lo2 : hi2;
      const int bits = (shift & 7) * 8;
      const unsigned long long y0 = bits ? x0 >> bits | x1 << (64 - bits) : x0, y1 = bits ? x1 >> bits | x2 << (64 - bits) : x1;
      return (u32x4_t){(unsigned)y0, (unsigned)(y0 >> 32), (unsigned)y1, (unsigned)(y1 >> 32)};
    }
  }
};

// ------------------------------------------------------------------------------------------------
// MFMA kernel
// ------------------------------------------------------------------------------------------------
// ONE_ROUND: the launch has a workgroup for every tile, so a workgroup handles at most one.  The
// tile loop is then known to run once, which lets the compiler drop everything it otherwise carries
// from tile to tile (measured: 1.2 us of a 9 us launch on decode-sized problems).
//
// STREAMK (eight-wave tile only): the tail policy for tile counts that do not fill the last round of
// workgroups (iris_layout::split_plan has the scheme).  Inside every XCD's span of tiles, the tiles of
// the full rounds are handed out whole, as in the other builds.  In the last round the workgroups that
// would find no tile help the others: a helper multiplies a piece of a tile's K steps, stores its fp32
// accumulators to the piece's slot of p.sk_partials (write-through) and sets the slot's flag to
// p.sk_epoch; the tile's main workgroup multiplies the first K steps, waits for its helpers' flags, adds
// their partial sums in ascending piece order and runs the ordinary epilogue.  Helpers are the XCD's
// first workgroups and never wait, mains wait only for helpers - workgroups with lower indices, which
// the hardware dispatches first - so the waits end whatever part of the grid is resident.
//
// ANY_ROWS: the rows of C and aux start and end anywhere (any_epilogue.h), N is not a whole number of 16-byte pieces; A and
// B are whole pieces all the same, because they lie so or because pack_kernel has laid them out (pack_kernel.h).
template <class CFG, bool ONE_ROUND, bool STREAMK = false, bool ANY_ROWS = false>
__global__ void __launch_bounds__(CFG::NT, CFG::WAVES_PER_SIMD) fused_mfma_kernel(const FusedParams p_in) {
  static_assert(!ANY_ROWS || (ONE_ROUND && !STREAMK), "any rows: one workgroup per tile");
  static_assert(!STREAMK || (CFG::NW == 8 && !ONE_ROUND), "split tiles: eight-wave tile, looping build");
  using Out = typename OutOf<CFG::IN>::type;
  // LDS layouts of A (and of B given K-contiguous, whose rows are as long), and of row-major B
  using ATile = typename std::conditional<CFG::BLK == 16, RowTile16<CFG::RBA>, RowTile<CFG::RBA>>::type;
  using BColTile = typename std::conditional<CFG::BLK == 16, ColTile16<CFG::RBB>, ColTile<CFG::RBB, CFG::ES>>::type;
  constexpr int ES = CFG::ES, CE = CFG::CE, BM = CFG::BM, BN = CFG::BN, BK = CFG::BK, BLK = CFG::BLK;
  constexpr int MB = CFG::MB, NB = CFG::NB, TM = CFG::TM, TN = CFG::TN, NW = CFG::NW, NT = CFG::NT;
  constexpr bool PINGPONG = CFG::NW == 8;
  constexpr int STAGES = CFG::STAGES, LA = CFG::LA, LB = CFG::LB, NFRAG = CFG::NFRAG, KS = CFG::KSLICES;

  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const FusedParams q_args = pin_loader_arguments(p_in);  // the loaders' kernel arguments, fetched in one batch
  const FusedParams& p = q_args;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / CFG::WN, wn = wave % CFG::WN;

  // Heap bases of the first slots, read once (scalar loads) before the kernel stores anything.
  unsigned long long hb[kMaxCachedSlots];
  if (p.hb_in_args) {  // kernel arguments when the host knew them
#pragma unroll
    for (int r = 0; r < kMaxCachedSlots; ++r) hb[r] = (unsigned long long)p.hb_arg[r];
  } else if (p.heap_bases) {  // else independent loads behind one branch (indices clamped to the world size)
#pragma unroll
    for (int r = 0; r < kMaxCachedSlots; ++r) hb[r] = (unsigned long long)p.heap_bases[min(r, p.world - 1)];
  } else {
#pragma unroll
    for (int r = 0; r < kMaxCachedSlots; ++r) hb[r] = 0ull;
  }
#pragma unroll
  for (int r = 0; r < kMaxCachedSlots; ++r) hb[r] = uniform64(hb[r]);  // scalar registers, whichever branch ran
  unsigned long long hb_own = 0ull;
  if (p.rank < kMaxCachedSlots) {
#pragma unroll
    for (int r = 0; r < kMaxCachedSlots; ++r) hb_own = (r == p.rank) ? hb[r] : hb_own;
  } else {
    hb_own = uniform64((unsigned long long)p.heap_bases[p.rank]);
  }
  auto heap_base = [&](int r) -> unsigned long long {
    unsigned long long v = 0;
    if (r < kMaxCachedSlots) {
#pragma unroll
      for (int q = 0; q < kMaxCachedSlots; ++q) v = (r == q) ? hb[q] : v;
    } else {
      v = (unsigned long long)p.heap_bases[r];
    }
    return v;
  };
  // Address in slot r of own-slot address `own`.
  auto in_slot = [&](unsigned long long own, int r) -> unsigned long long { return heap_base(r) + (own - hb_own); };

  // ---- loader descriptors (tile independent) ---------------------------------------------------
  // A: row tile [BM][RBA].
  int la_row[LA], la_k[LA];
  unsigned la_off[LA];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    int row, c;
    ATile::from_lds((wave + i * NW) * kDmaBytes + lane * kChunkBytes, row, c);
    la_row[i] = row;
    la_k[i] = c * CE;
    la_off[i] = (unsigned)(row * p.s_am * ES + c * kChunkBytes);
  }
  // B: col tile [BK][BN*ES] (row-major B) or row tile [BN][RBA] (B given K-contiguous).
  int lb_row[LB], lb_col[LB];  // col tile: (k row, n element); row tile: (n row, k element)
  unsigned lb_off[LB];
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    int row, c;
    const int off = (wave + i * NW) * kDmaBytes + lane * kChunkBytes;
    if constexpr (CFG::B_KCONTIG) {
      ATile::from_lds(off, row, c);
      lb_off[i] = (unsigned)(row * p.s_bn * ES + c * kChunkBytes);
    } else {
      BColTile::from_lds(off, row, c);
      lb_off[i] = (unsigned)(row * p.s_bk * ES + c * kChunkBytes);
    }
    lb_row[i] = row;
    lb_col[i] = c * CE;
  }

  // ---- fragment read offsets (relative to the slot's A / B region) -------------------------------
  auto frag_row = [&]() { return BLK == 16 ? mma16_row(lane) : frag16_row(lane); };
  auto frag_chunk = [&](int kk, int h) {
    return CFG::IN == IN_FP8 ? frag8_chunk(lane, kk, h) : BLK == 16 ? mma16_chunk(lane, kk) : frag16_chunk(lane, kk);
  };
  int fa_off[KS][NFRAG];
#pragma unroll
  for (int kk = 0; kk < KS; ++kk)
#pragma unroll
    for (int h = 0; h < NFRAG; ++h) fa_off[kk][h] = ATile::lds_offset(wm * TM + frag_row(), frag_chunk(kk, h));
  // B operand: K-contiguous B reads exactly like A; row-major B uses transpose reads.
  constexpr int NTR = (CFG::IN == IN_FP8 || BLK == 16) ? 1 : 2;  // distinct swizzles among the transpose reads
  int fb_off[CFG::B_KCONTIG ? KS : NB][CFG::B_KCONTIG ? NFRAG : NTR];
  if constexpr (CFG::B_KCONTIG) {
#pragma unroll
    for (int kk = 0; kk < KS; ++kk)
#pragma unroll
      for (int h = 0; h < NFRAG; ++h) fb_off[kk][h] = ATile::lds_offset(wn * TN + frag_row(), frag_chunk(kk, h));
  } else {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int j = 0; j < NTR; ++j) {
        const int krow = CFG::IN == IN_FP8 ? tr8_krow(lane, 0, 0) : BLK == 16 ? mma16_tr_krow(lane, 0, 0) : tr16_krow(lane, 0, j);
        const int n = wn * TN + nb * BLK + (CFG::IN == IN_FP8 ? tr8_ncol(lane) : BLK == 16 ? mma16_tr_ncol(lane) : tr16_ncol(lane));
        fb_off[nb][j] = BColTile::lds_offset(krow, n / CE) + (n % CE) * ES;
      }
  }

  // Read the fragments of k-slice kk of ring slot `slot`.
  auto load_frag_b = [&](i32x4_t (&dst)[NFRAG], int slot_off, int kk, int nb) {  // slot_off: byte offset of the ring slot
    const char* sb = smem + slot_off + CFG::A_BYTES;
    if constexpr (CFG::B_KCONTIG) {
#pragma unroll
      for (int h = 0; h < NFRAG; ++h)
        dst[h] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sb + fb_off[kk][h] + nb * BLK * CFG::RBB);
    } else if constexpr (CFG::IN == IN_FP8) {
      i32x2_t t[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        t[r] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (LDS_AS i32x2_t*)(LDS_AS char*)(sb + fb_off[nb][0] + (kk * 64 + 8 * r) * CFG::RBB));
      dst[0] = (i32x4_t){t[0].x, t[0].y, t[1].x, t[1].y};
      dst[NFRAG - 1] = (i32x4_t){t[2].x, t[2].y, t[3].x, t[3].y};
    } else {
      i32x2_t t[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        t[j] = __builtin_bit_cast(i32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (LDS_AS i16x4_t*)(LDS_AS char*)(sb + fb_off[nb][NTR == 2 ? j : 0] + (kk * CFG::KM + (NTR == 2 ? 0 : 4 * j)) * CFG::RBB)));
      dst[0] = (i32x4_t){t[0].x, t[0].y, t[1].x, t[1].y};
    }
  };
  auto load_frag_a = [&](Frags<CFG>& f, int slot_off, int kk, int mb) {
    const char* sa = smem + slot_off;
#pragma unroll
    for (int h = 0; h < NFRAG; ++h)
      f.a[mb][h] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sa + fa_off[kk][h] + mb * BLK * CFG::RBA);
  };
  auto load_frags = [&](Frags<CFG>& f, int slot_off, int kk) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) load_frag_b(f.b[nb], slot_off, kk, nb);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) load_frag_a(f, slot_off, kk, mb);
  };

  const int total_tiles = p.tiles_m * p.tiles_n;
  const int nsrc = (p.gather == GATHER_K) ? p.world : 1;
  const int klocal = (p.gather == GATHER_K) ? p.K_local : p.K;
  const int nkb = cdiv(klocal, BK);
  const int nsteps = nsrc * nkb;
  const unsigned smem_base = __builtin_amdgcn_readfirstlane(lds_address(smem));
  const unsigned long long a_own = (unsigned long long)p.A;

  // Split tiles (iris_layout::split_plan): every workgroup first takes its whole tiles, dp_rounds of
  // them at positions dp_first + round * wg_per_xcd of the grouped order; then the last round's tiles,
  // at positions sk_first + j, go to a main and its helpers.  Partial sum slot (and flag) of piece i >= 1
  // of tile j: sk_slot0 + j * per_tile + i - 1.
  enum { ITEM_WHOLE = 0, ITEM_PART = 1, ITEM_OWNER = 2 };  // the kinds of iris_layout::split_item
  int sk_first = 0, sk_left = 0, sk_slot0 = 0, sk_served = 0, dp_first = 0, dp_rounds = 0, dp_it = 0, wg_per_xcd = 1, sk_local = 0;
  SplitPlan plan = {0, 1, nsteps, 0};
  if constexpr (STREAMK) {
    const int xcd = blockIdx.x % p.num_xcd;
    sk_local = blockIdx.x / p.num_xcd;
    wg_per_xcd = gridDim.x / p.num_xcd;
    const int span = cdiv(total_tiles, p.num_xcd);
    const int first = min(xcd * span, total_tiles);
    const int mine = min(span, total_tiles - first);  // tiles of this XCD
    dp_rounds = mine / wg_per_xcd;
    sk_left = mine - dp_rounds * wg_per_xcd;          // tiles of the last, partly filled round
    dp_first = first + sk_local;
    sk_first = first + dp_rounds * wg_per_xcd;
    sk_slot0 = xcd * wg_per_xcd;
    plan = split_plan(sk_left, wg_per_xcd, nsteps, p.sk_gather_cost, p.sk_pass_cost);
  }

  // Looping workgroups of the eight-wave tile fetch the first K step of their next tile into ring slot 0
  // as soon as the K loop of the current tile is over (the staged tile lives above that slot): the loads
  // go out ahead of the epilogue's stores instead of behind them, and their latency - cold operand panels,
  // 2-3 us - passes under the epilogue.
  constexpr bool PREFETCH_NEXT = CFG::STAGE_SWIZZLED && !ONE_ROUND && !STREAMK;
  bool first_step_prefetched = false;
  const int order_xcd = p.interleave ? 1 : p.num_xcd;  // see FusedParams::interleave

  for (int it = 0; ONE_ROUND ? it < 1 : true; ++it) {
    int tidx, k_begin = 0, k_end = nsteps, item = ITEM_WHOLE, partners = 0, slot = 0;
    if constexpr (STREAMK) {
      if (dp_it < dp_rounds) {
        tidx = dp_first + dp_it * wg_per_xcd;
        ++dp_it;
      } else {
        int j;
        if (!split_item(plan, sk_left, wg_per_xcd, nsteps, sk_local, sk_served++, j, k_begin, k_end, item, partners, slot)) break;
        tidx = sk_first + j;
        slot += sk_slot0;
      }
    } else {
      tidx = xcd_tile_index(blockIdx.x, gridDim.x, it, total_tiles, order_xcd);
      if (tidx < 0) break;
      tidx += p.tile_rotate;
      if (tidx >= total_tiles) tidx -= total_tiles;
    }
    PHASE_STAMP(0);
    int tm, tn;
    grouped_tile(tidx, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- per-tile loader state ---------------------------------------------------------------
    // Row validity is folded into the per-lane offsets once per tile.
    unsigned a_voff[LA], b_voff[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) a_voff[i] = (m0 + la_row[i] < p.M) ? la_off[i] : kInvalidOffset;
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      if constexpr (CFG::B_KCONTIG)
        b_voff[i] = (n0 + lb_row[i] < p.N) ? lb_off[i] : kInvalidOffset;
      else
        b_voff[i] = (n0 + lb_col[i] < p.N) ? lb_off[i] : kInvalidOffset;
    }
    // Byte offset of this tile's first A row inside the slot that holds it.
    int a_slot = p.rank;
    long long a_row0 = m0;
    if (p.gather == GATHER_M) {
      a_slot = m0 / p.M_local;
      a_row0 = m0 - (long long)a_slot * p.M_local;
    }
    if (p.gather == GATHER_K) a_slot = k_begin / nkb;  // the source that holds the first K step
    const unsigned long long a_tile_off = (unsigned long long)(a_row0 * p.s_am * ES);
    const i32x4_t rb = make_rsrc_words((unsigned long long)p.B + (unsigned long long)n0 * (CFG::B_KCONTIG ? p.s_bn : 1) * ES);
    i32x4_t ra = make_rsrc_words((p.gather == GATHER_NONE ? a_own : in_slot(a_own, a_slot)) + a_tile_off);

    // Loader position: next K step to issue = (i_src, i_kb), i_step overall.
    int i_step = k_begin, i_src = k_begin / nkb, i_kb = k_begin - (k_begin / nkb) * nkb;

    // The direct-to-LDS loads of one K step, issued one at a time so that the main loop can spread
    // them between its MFMAs (a wave issues in order: a burst of loads right after the barrier would
    // hold back the MFMAs behind it while the memory pipeline absorbs the burst).  Steps past the end
    // load nothing (every lane is out of range and deposits zeros), which keeps the per-thread count
    // of outstanding loads identical on every step that has any.
    struct StepLoads {
      int klim;
      unsigned sa, sb, a_soff, b_soff;
    };
    auto begin_step = [&](int slot_off) {  // slot_off: byte offset of the ring slot to fill
      StepLoads L;
      const bool live = i_step < k_end;
      const int k0 = i_kb * BK;
      L.klim = live ? klocal - k0 : 0;  // k elements of this step that exist
      L.sa = smem_base + slot_off + wave * kDmaBytes;
      L.sb = L.sa + CFG::A_BYTES;
      L.a_soff = (unsigned)(k0 * ES);
      const long long kglob = (long long)i_src * klocal + k0;
      L.b_soff = __builtin_amdgcn_readfirstlane(
          CFG::B_KCONTIG ? (unsigned)(kglob * ES) : (unsigned)(kglob * p.s_bk * ES));
      return L;
    };
    auto load_offset = [&](const StepLoads& L, int j) -> unsigned {  // per-lane offset of load j
      if (j < LA) return (la_k[j] < L.klim) ? a_voff[j] : kInvalidOffset;
      const int i = j - LA;
      const int kpos = CFG::B_KCONTIG ? lb_col[i] : lb_row[i];
      return (kpos < L.klim) ? b_voff[i] : kInvalidOffset;
    };
    auto issue_at = [&](const StepLoads& L, int j, unsigned v) {
      if (j < LA)
        dma16(ra, L.sa + j * NW * kDmaBytes, v, L.a_soff);
      else
        dma16(rb, L.sb + (j - LA) * NW * kDmaBytes, v, L.b_soff);
    };
    auto issue_one = [&](const StepLoads& L, int j) { issue_at(L, j, load_offset(L, j)); };  // j in [0, LA + LB)
    auto end_step = [&]() {
      ++i_step;
      ++i_kb;
      const bool source_done = PINGPONG ? __builtin_expect(i_kb == nkb, 0) : i_kb == nkb;  // (the four-wave loop is slower with the hint)
      if (source_done) {  // next source slot (gather along K only)
        i_kb = 0;
        ++i_src;
        if (p.gather == GATHER_K && i_src < nsrc) ra = make_rsrc_words(in_slot(a_own, i_src) + a_tile_off);
      }
    };
    auto issue = [&](int slot) {
      const StepLoads L = begin_step(slot * CFG::STAGE_BYTES);
#pragma unroll
      for (int j = 0; j < LA + LB; ++j) issue_one(L, j);
      end_step();
    };

    MfmaAcc<CFG> acc;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 4 * CFG::QUADS; ++i) acc.v[mb][nb][i] = 0.f;

    // ---- prologue: the first K steps, wait for the first of them ------------------------------------
    // Four-wave loop: STAGES-1 steps.  Two-group loop: three (a slot, and the next one's first fragments, are read while a third
    // one is refilled).  When the first step is there already, from its prefetch, what the first product waits for is the loads'
    // acceptance, 0.3 us a step: the early waves then stay two steps ahead, and the late ones send their third step out after the barrier.
    const bool late = PINGPONG && wave >= 4;
    const bool there = PREFETCH_NEXT && first_step_prefetched;
    const int ahead = late || !there ? 3 : 2;  // K steps in flight before the loop starts
    if constexpr (PINGPONG) {
      if (there) end_step();  // only the loader position moves on
      else issue(0);
      issue(1);
      if (!there) {
        issue(2);
        wait_vmcnt<2 * (LA + LB)>();
      } else {
        wait_vmcnt<LA + LB>();
      }
    } else {
#pragma unroll
      for (int s = 0; s < STAGES - 1; ++s) issue(s);
      wait_vmcnt<(STAGES - 2) * (LA + LB)>();
    }
    first_step_prefetched = false;
    __builtin_amdgcn_s_barrier();
    PHASE_STAMP(1);
    Frags<CFG> fr[KS < 2 ? 2 : KS];  // one set per k-slice (two for the loops that double-buffer)
    if constexpr (!PINGPONG) load_frags(fr[0], 0, 0);

    // ---- main loop ----------------------------------------------------------------------------
    // Invariant at the top of step s: the operands of step s are in LDS and visible to all waves,
    // and the fragments of its first k-slice are in flight.  The step first makes sure step s+1
    // has landed too, so that its first fragments can be fetched while step s still computes.
    // The four-wave tiles have registers to spare and run the loop unrolled over the ring positions,
    // which turns every LDS address of a step into a constant offset (5-10 % on those tiles); the
    // eight-wave tile would spill and keeps the ring position in a register.
    constexpr int RING_UNROLL = (NW == 4) ? STAGES : 1;
    int s = k_begin, ring_pos = 0;
    if constexpr (PINGPONG) {
      static_assert(KS == 1 && MB % 2 == 0 && NB % 2 == 0, "eight-wave loop: one k-slice per step, blocks in quadrants");
      // Eight waves, two per SIMD: waves 0-3 and waves 4-7 run half a step apart.  A step is a memory phase (the
      // direct-to-LDS loads of a later step) and a compute phase (the products, with the fragment reads
      // in their shadow), each closed by a workgroup barrier, so that on every SIMD one wave feeds the matrix pipe
      // while the other one has the memory port to itself.  A direct-to-LDS load does not issue in the shadow of an
      // MFMA: a wave takes some 80 cycles to get one accepted.
      //
      // A memory phase also reads the left half of B's fragments of its step; a compute phase reads A's lower rows of its
      // own step (quad_block needs them half way through) and of the next step A's upper rows, into the registers that
      // the first half has done with, and the right half of B, into those free in the last quadrant.  The next step's
      // slot has landed for all waves by then - the late group waits for it at the end of its previous memory phase -,
      // which takes a ring of five: this step's slot, the next one's, one that is being waited for, one with loads in
      // flight, and the one being refilled, which the other group may have left only half a step ago.
      //
      // The last steps, which have nothing to load any more, are a loop of their own: to load nothing takes as long as to load.
      // Memory phases are as long as compute phases, so what else stands in them counts: a test of whether there is anything
      // to load cost 4 to 7 % with long K, and without the hints of which way a step usually goes the compiler kept
      // the usual way's scalars in vector registers in the build for split tiles (1 to 3 %).
      //
      // What bounds it is power, with anything but zeros in the operands (bf16 4096x4096x8192 as a plain product, whole
      // launch: 186 us on normal data, 138 on zeros).  Before - 32x32x16 products, half of the fragments read in the
      // memory phase, a ring of four - it took 203 (zeros 130: one wave per SIMD issues a 16x16x32 product every 17
      // cycles, not 16), 8192x1792x4096 98 -> 92; 16x16x32 products in that loop 197 and 98; every fragment of B read in the
      // memory phase 189; the left half of B one step ahead as well, through a copy, 188.
      // The loader position of the common case - a whole K step inside one source - is carried in
      // scalar registers that advance by constants, and its loads need no per-lane k test; partial
      // steps, source changes and the empty steps past the end take the general path.
      const unsigned b_inc = __builtin_amdgcn_readfirstlane(
          CFG::B_KCONTIG ? (unsigned)(BK * ES) : (unsigned)((long long)BK * p.s_bk * ES));
      unsigned a_so = 0, b_so = 0;
      int k_left = 0;
      auto resync = [&]() {
        a_so = (unsigned)(i_kb * BK * ES);
        const long long kglob = (long long)i_src * klocal + (long long)i_kb * BK;
        b_so = __builtin_amdgcn_readfirstlane(
            CFG::B_KCONTIG ? (unsigned)(kglob * ES) : (unsigned)(kglob * p.s_bk * ES));
        k_left = i_step < k_end ? klocal - i_kb * BK : 0;
      };
      unsigned rd = 0;                                    // byte offset of the slot this step reads
      unsigned wr = ahead * CFG::STAGE_BYTES;             // ... and of the slot it refills
      const unsigned wr_wave = smem_base + wave * kDmaBytes;
      constexpr int NMFMA = MB * NB, HA = MB / 2, HB = NB / 2, Q = NMFMA / 4;
      __builtin_amdgcn_sched_barrier(0);  // (no fragment read moves up past the prologue's barrier)
#pragma unroll
      for (int nb = HB; nb < NB; ++nb) load_frag_b(fr[0].b[nb], 0, 0, nb);
#pragma unroll
      for (int mb = 0; mb < HA; ++mb) load_frag_a(fr[0], 0, 0, mb);
      if (late) {
        if (there) issue(2);
        wait_vmcnt<LA + LB>();
        __builtin_amdgcn_s_barrier();
      }
      resync();
      auto product = [&](int i) {
        int mb, nb;
        quad_block<MB, NB>(i, mb, nb);
        acc.v[mb][nb] = mfma_of<CFG>(fr[0].a[mb], fr[0].b[nb], acc.v[mb][nb]);
      };
      auto k_step = [&](auto loads) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < HB; ++nb) load_frag_b(fr[0].b[nb], rd, 0, nb);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(loads)::value) {
          if (__builtin_expect(k_left >= BK, 1)) {
#pragma unroll
            for (int j = 0; j < LA; ++j) dma16(ra, wr_wave + wr + j * NW * kDmaBytes, a_voff[j], a_so);
#pragma unroll
            for (int i = 0; i < LB; ++i)
              dma16(rb, wr_wave + wr + CFG::A_BYTES + i * NW * kDmaBytes, b_voff[i], b_so);
          } else {
            const StepLoads L = begin_step(wr);
#pragma unroll
            for (int j = 0; j < LA + LB; ++j) issue_one(L, j);
          }
          end_step();
          if (__builtin_expect(i_kb == 0, 0)) {
            resync();
          } else {
            a_so += BK * ES;
            b_so += b_inc;
            k_left -= BK;
          }
        }
        const unsigned rd_next = rd + CFG::STAGE_BYTES == CFG::RING_BYTES ? 0 : rd + CFG::STAGE_BYTES;
        // Own fragment reads done, and own loads landed: of step s+2, of waves that are two steps ahead s+1, and at the end all.
        wait_vmcnt_lgkm0<decltype(loads)::value ? LA + LB : 0>();
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NMFMA; ++i) {
          product(i);
#pragma unroll
          for (int pc = 0; pc < HA; ++pc) {
            if (pc * Q / HA == i) load_frag_a(fr[0], rd, 0, HA + pc);             // this step's lower rows
            if (2 * Q + pc * Q / HA == i) load_frag_a(fr[0], rd_next, 0, pc);     // the next step's upper rows
          }
#pragma unroll
          for (int pc = 0; pc < HB; ++pc) {
            if (3 * Q + pc * Q / HB == i) load_frag_b(fr[0].b[HB + pc], rd_next, 0, HB + pc);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        rd = rd_next;
        wr = wr + CFG::STAGE_BYTES == CFG::RING_BYTES ? 0 : wr + CFG::STAGE_BYTES;
      };
      for (const int last = k_end - ahead; s < last; ++s) k_step(std::true_type{});
      for (; s < k_end; ++s) k_step(std::false_type{});
      if (!late) __builtin_amdgcn_s_barrier();
    } else
    while (s < k_end) {
#pragma unroll
    for (int u = 0; u < RING_UNROLL; ++u) {
      if (s >= k_end) break;
      ++s;
      const int slot = (RING_UNROLL == 1) ? ring_pos : u;
      // LDS is one coherent memory per CU, so a bare s_barrier (no fence, hence no forced wait for
      // the fragment reads in flight) orders the operand ring between the waves.
      wait_vmcnt<(STAGES - 3) * (LA + LB)>();  // this thread's loads of step s+1 have landed
      __builtin_amdgcn_s_barrier();             // everyone's have; everyone is past step s-1
      int pslot = slot + STAGES - 1;
      if (pslot >= STAGES) pslot -= STAGES;
      const StepLoads L = begin_step(pslot * CFG::STAGE_BYTES);  // refills the slot the previous step used
      const int nslot = slot + 1 == STAGES ? 0 : slot + 1;
      constexpr int NSLOT = KS * MB;          // MFMA groups of a step; the loads are spread over them
      constexpr int NLOAD = LA + LB;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        if (kk + 1 < KS)
          load_frags(fr[(kk + 1) & 1], slot * CFG::STAGE_BYTES, kk + 1);
        else
          load_frags(fr[(kk + 1) & 1], nslot * CFG::STAGE_BYTES, 0);
        const Frags<CFG>& f = fr[kk & 1];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
          for (int j = 0; j < NLOAD; ++j)
            if (j * NSLOT / NLOAD == kk * MB + mb) issue_one(L, j);
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc.v[mb][nb] = mfma_of<CFG>(f.a[mb], f.b[nb], acc.v[mb][nb]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      end_step();
      static_assert(KS % 2 == 0 || KS == 1, "fragment double buffer assumes an even slice count");
      if constexpr (KS == 1) {
        // With one slice per step the two buffers alternate across steps.
        Frags<CFG> t = fr[0];
        fr[0] = fr[1];
        fr[1] = t;
      }
      ring_pos = nslot;
    }
    }

    // The ring is reused as epilogue staging: drain the (empty) loads still in flight and make
    // sure every wave has finished reading operands.
    wait_vmcnt<0>();
    __syncthreads();
    PHASE_STAMP(2);

    if constexpr (STREAMK) {
      // Partial sums travel in the accumulators' own layout: 16-byte piece j of thread t at byte
      // (j * NT + t) * 16 of the piece's slot, so that every wave instruction moves 1 KiB.
      constexpr int PIECES = MB * NB * CFG::QUADS;  // 16-byte pieces per thread
      constexpr long long SLOT_BYTES = (long long)PIECES * NT * 16;
      if (item == ITEM_PART) {
        // (The base goes through an empty asm so that the compiler computes the pieces' addresses here, one
        // at a time, instead of keeping all of them in registers from the top of the kernel.)
        unsigned long long slot_base = (unsigned long long)p.sk_partials + (unsigned long long)slot * SLOT_BYTES;
        asm volatile("" : "+s"(slot_base));
        char* const dst = (char*)slot_base + tid * 16;
#pragma unroll
        for (int j = 0; j < PIECES; ++j) {
          const int mb = j / (NB * CFG::QUADS), nb = j / CFG::QUADS % NB, q = j % CFG::QUADS;
          u32x4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = __float_as_uint(acc_read(acc.v[mb][nb][4 * q + e]));
          store16_system_of_valu_data(dst + (long long)j * NT * 16, v);
          __builtin_amdgcn_sched_barrier(0);  // one piece at a time: the scheduler would read all 128 registers first
        }
        // Published like an aux tile: stores acknowledged by every wave, then one relaxed flag store.
        wait_vmcnt<0>();
        __syncthreads();
        if (tid == 0) __hip_atomic_store(p.sk_flags + slot, p.sk_epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        PHASE_STAMP(3);
        continue;  // the ring is free (barrier above); no epilogue for a partial sum
      }
      if (item == ITEM_OWNER) {
        if (tid < partners) {
          const int* flag = p.sk_flags + (slot + tid);
          // Relaxed polls and one acquire fence at the end: an acquire load per poll would invalidate the
          // XCD's L2 on every turn while the helpers next door are still storing (measured: their 256 KiB
          // took 25 us that way).
          long long polls = 0;
          while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != p.sk_epoch) {
            if (p.spin_limit > 0 && ++polls >= p.spin_limit) {
              if (p.status) __hip_atomic_store(p.status, IRIS_HIP_STATUS_SPIN_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
              break;
            }
            __builtin_amdgcn_s_sleep(8);
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
        }
        __syncthreads();
      }
    }

    if constexpr (PREFETCH_NEXT) {
      int nidx = xcd_tile_index(blockIdx.x, gridDim.x, it + 1, total_tiles, order_xcd);
      if (nidx >= 0) {
        nidx += p.tile_rotate;
        if (nidx >= total_tiles) nidx -= total_tiles;
        int ntm, ntn;
        grouped_tile(nidx, p.tiles_m, p.tiles_n, p.group_m, ntm, ntn);
        const int nm0 = ntm * BM, nn0 = ntn * BN;
        int n_slot = p.rank;
        long long n_row0 = nm0;
        if (p.gather == GATHER_M) {
          n_slot = nm0 / p.M_local;
          n_row0 = nm0 - (long long)n_slot * p.M_local;
        }
        if (p.gather == GATHER_K) n_slot = 0;
        const i32x4_t nra = make_rsrc_words((p.gather == GATHER_NONE ? a_own : in_slot(a_own, n_slot)) + (unsigned long long)(n_row0 * p.s_am * ES));
        const i32x4_t nrb = make_rsrc_words((unsigned long long)p.B + (unsigned long long)nn0 * (CFG::B_KCONTIG ? p.s_bn : 1) * ES);
        const unsigned sa = smem_base + wave * kDmaBytes, sb = sa + CFG::A_BYTES;  // ring slot 0
#pragma unroll
        for (int j = 0; j < LA; ++j) {
          const bool ok = nm0 + la_row[j] < p.M && la_k[j] < klocal;
          dma16(nra, sa + j * NW * kDmaBytes, ok ? la_off[j] : kInvalidOffset, 0u);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
          const bool ok = CFG::B_KCONTIG ? (nn0 + lb_row[i] < p.N && lb_col[i] < klocal) : (nn0 + lb_col[i] < p.N && lb_row[i] < klocal);
          dma16(nrb, sb + i * NW * kDmaBytes, ok ? lb_off[i] : kInvalidOffset, 0u);
        }
        first_step_prefetched = true;
      }
    }

    // ---- epilogue -------------------------------------------------------------------------------
    // The whole output tile is first written to LDS in the output type (the operand ring is dead
    // by now), which frees the accumulators; both phases then stream rows of the tile, 16 bytes per
    // lane and BN*2 contiguous bytes per row, with many loads in flight per thread.
    {
      // Split tiles: 16-byte pieces of a partial sum, in the layout its workgroup stored them in.
      constexpr int PIECES = MB * NB * CFG::QUADS, NBATCH = 4, BATCH = PIECES / NBATCH;
      constexpr long long SLOT_BYTES = (long long)PIECES * NT * 16;
      float badd[MB] = {};
      if constexpr (MB <= 2) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          if (p.bias) {
            const int gm = m0 + wm * TM + mb * BLK + acc_col(lane);
            if (gm < p.M) badd[mb] = load_scalar_as_float(p.bias, (long long)gm * p.s_bias, p.bias_dtype);
          }
        }
      } else if (p.bias) {
        // Every load is out before the first is used (a block at a time the blocks of sixteen rows made eight round trips of
        // it, 6 of the 113 us of a plain fp16 16384x8192x128 with bias).  Rows past the end, which are never stored, take the last one's.
        // (The four-wave tiles, with one or two rows a lane, are 0.6 % slower in this form, bias or not: fp16 two-shot 896x2880x512.)
        const bool wide = p.bias_dtype == IRIS_HIP_FP32;
        unsigned raw[MB];
        auto row_of = [&](int mb) -> long long {
          const int gm = m0 + wm * TM + mb * BLK + (BLK == 16 ? mma16_acc_col(lane) : acc_col(lane));
          return (long long)min(gm, p.M - 1) * p.s_bias;
        };
        if (wide) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) raw[mb] = ((const unsigned*)p.bias)[row_of(mb)];
        } else {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) raw[mb] = ((const unsigned short*)p.bias)[row_of(mb)];
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          badd[mb] = wide ? __uint_as_float(raw[mb]) : p.bias_dtype == IRIS_HIP_BF16 ? bf16_bits_to_float((unsigned short)raw[mb]) : f16_bits_to_float((unsigned short)raw[mb]);
      }
      // The lane index as the staging addresses see it goes through an empty asm: the compiler would otherwise compute
      // them once, ahead of the tile loop, and carry more registers through the K loop.  A lane has one address, of its
      // first piece; the others are a constant away from it.
      int lane_s = lane;
      asm volatile("" : "+v"(lane_s));
      const int stage_first = CFG::stage_offset(wm * TM + (BLK == 16 ? mma16_acc_col(lane_s) : acc_col(lane_s)),
                                                (wn * TN + (BLK == 16 ? mma16_acc_row(lane_s, 0) : acc_row(lane_s, 0))) * 2);
      // Piece j of the thread: 4 consecutive n of one m, from their fp32 sums to the staged tile.
      auto stage_piece = [&](int j, const float (&sum)[4]) {
        const int mb = j / (NB * CFG::QUADS), nb = j / CFG::QUADS % NB, q = j % CFG::QUADS;
        float h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = sum[e] * p.scale + badd[mb];
        u32x2_t w;
        w.x = Out::pack(h[0], h[1]);
        w.y = Out::pack(h[2], h[3]);
        *(LDS_AS u32x2_t*)(LDS_AS char*)(smem + CFG::stage_step(stage_first, mb * BLK, (nb * BLK + 8 * q) * 2)) = w;
      };
      auto own_piece = [&](int j, float (&sum)[4]) {
        const int mb = j / (NB * CFG::QUADS), nb = j / CFG::QUADS % NB, q = j % CFG::QUADS;
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] = acc_read(acc.v[mb][nb][4 * q + e]);
      };
      bool staged = false;
      if constexpr (STREAMK) {
        if (item == ITEM_OWNER && partners > 0) {
          // own sum + the helper's partial sum, a quarter of the pieces at a time.  (The accumulators are only read: adding into them in place makes the compiler
          // move the whole tile through VGPRs.)
          staged = true;
          unsigned long long base = (unsigned long long)p.sk_partials + (unsigned long long)slot * SLOT_BYTES;
          asm volatile("" : "+s"(base));  // addresses are formed where they are used, not hoisted out of the tile loop
          const char* const src = (const char*)base + tid * 16;
          auto load_batch = [&](u32x4_t (&dst)[BATCH], const char* src, int b) {
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
              dst[i] = __builtin_nontemporal_load((const u32x4_t*)(src + (long long)(b * BATCH + i) * NT * 16));
          };
          {  // the next batch is on its way while this one is staged
            u32x4_t buf[2][BATCH];
            load_batch(buf[0], src, 0);
#pragma unroll
            for (int b = 0; b < NBATCH; ++b) {
              if (b + 1 < NBATCH) load_batch(buf[(b + 1) & 1], src, b + 1);
#pragma unroll
              for (int i = 0; i < BATCH; ++i) {
                float sum[4];
                own_piece(b * BATCH + i, sum);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += __uint_as_float(buf[b & 1][i][e]);
                stage_piece(b * BATCH + i, sum);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
      }
      if (!staged) {
#pragma unroll
        for (int j = 0; j < PIECES; ++j) {
          float sum[4];
          own_piece(j, sum);
          stage_piece(j, sum);
        }
      }
    }
    __syncthreads();
    PHASE_STAMP(3);

    if constexpr (ANY_ROWS) {
      using Elem = typename std::conditional<CFG::IN == IN_F16, ElemF16, ElemBF16>::type;
      finish_any<Elem, BM, BN, NT, CFG::NW == 8 ? 16 : 14, true>(p, StagedTile<CFG>{smem}, m0, n0, tid);
      return;
    } else {

    constexpr int CPR = BN / 8;            // 16-byte chunks per tile row
    constexpr int RPP = NT / CPR;          // tile rows covered by one pass of the workgroup
    constexpr int PASSES = BM / RPP;
    int tid_s = tid;  // as lane_s above: per-thread staging offsets are formed here, not ahead of the tile loop
    asm volatile("" : "+v"(tid_s));
    const int t_row = tid_s / CPR, t_chunk = tid_s % CPR;
    const int gn = n0 + t_chunk * 8;
    const bool col_ok = gn < p.N;
    // LDS offset of this thread's chunk in pass ps: t_pass[ps & 1] + ps * RPP * TROW (the passes are RPP
    // rows apart; with the swizzled layout the chunk's place in the row alternates between two values).
    static_assert(!CFG::STAGE_SWIZZLED || (2 * RPP) % CPR == 0, "the swizzle must repeat every two passes");
    const int t_pass[2] = {CFG::stage_offset(t_row, t_chunk * 16), CFG::stage_offset(t_row + RPP, t_chunk * 16) - RPP * CFG::TROW};

    // Phase 1: C (plain store) or aux (own slot).  When no peer contributes (world of one, or peers
    // switched off) the reduced tile equals the own tile, so C is written in the same pass and
    // phase 2 is skipped.
    const bool flags = epi_has_flags(p.epi);
    const bool solo = flags && (!p.sum_peers || p.world == 1);
    {
      const int ftn1 = cdiv(p.N, p.flag_bn);
      const int ftotal1 = cdiv(p.M, p.flag_bm) * ftn1;
      const unsigned long long c_base = (unsigned long long)p.C;
      if (p.epi == EPI_ATOMIC) {
        // The tile is added into every rank's C (iris/mem/triton/context.py:689-702) with packed 16-bit
        // atomics of one dword each.  Dword d of a pass belongs to thread d mod NT, so that one wave
        // instruction covers 256 contiguous bytes (two whole lines for the L2's atomic units); with
        // each thread adding the four dwords of its own 16-byte chunk an instruction touched eight
        // lines with eight dwords each, and the launch ran at a quarter of the rate.
        constexpr int DPR = BN / 2;                   // dwords per tile row
        constexpr int DPP = RPP * DPR;                // dwords per pass (= 4 * NT)
        for (int ps = 0; ps < PASSES; ++ps) {
#pragma unroll
          for (int j = 0; j < DPP / NT; ++j) {
            const int d = j * NT + tid;
            const int row = ps * RPP + d / DPR, dc = d % DPR;
            const int gm = m0 + row, gc = n0 + 2 * dc;
            if (gm >= p.M || gc >= p.N) continue;
            const unsigned w = *(const LDS_AS unsigned*)(LDS_AS char*)(smem + CFG::stage_offset(row, dc * 4));
            const long long eoff = ((long long)(gm + p.row_offset) * p.s_cm + gc) * 2;
            for (int pr = 0; pr < p.world; ++pr) {
              if (p.clear_c && pr == p.rank) *(unsigned*)(p.C + eoff) = added_to_zero(w);
              else atomic_add_packed<Out>((char*)(in_slot(c_base, pr) + eoff), w);
            }
          }
        }
      } else if (!flags) {
#pragma unroll 4
        for (int ps = 0; ps < PASSES; ++ps) {
          const int gm = m0 + ps * RPP + t_row;
          const u32x4_t v = *(const LDS_AS u32x4_t*)(LDS_AS char*)(smem + t_pass[ps & 1] + ps * RPP * CFG::TROW);
          if (gm < p.M && col_ok) {
            const long long eoff = ((long long)(gm + p.row_offset) * p.s_cm + gn) * 2;
            if (p.epi == EPI_ALL_GATHER) {
              // the tile goes to every rank's gathered output (iris/mem/triton/context.py:841-864)
              for (int pr = 0; pr < p.world; ++pr) __builtin_nontemporal_store(v, (u32x4_t*)(in_slot(c_base, pr) + eoff));
            } else {
              __builtin_nontemporal_store(v, (u32x4_t*)(p.C + eoff));
            }
          }
        }
      } else {
        const bool by_owner = p.epi != EPI_ONE_SHOT && (solo || p.clear_c);
#pragma unroll 4
        for (int ps = 0; ps < PASSES; ++ps) {
          const int gm = m0 + ps * RPP + t_row;
          const u32x4_t v = *(const LDS_AS u32x4_t*)(LDS_AS char*)(smem + t_pass[ps & 1] + ps * RPP * CFG::TROW);
          if (gm < p.M && col_ok) {
            const long long eoff = ((long long)gm * p.s_cm + gn) * 2;
            if (p.whole_lines) store16_system_nt(p.aux + eoff, v);
            else store16_system(p.aux + eoff, v);  // aux: read by the peers as soon as the flag is up
            int owner = p.rank;
            if (by_owner) {
              owner = owner_of(p.epi, (gm / p.flag_bm) * ftn1 + gn / p.flag_bn, ftotal1, p.world, p.rank);
              // Another rank's tile: zeros, behind the aux stores (8192 x 4096 reduce-scatter: a fill of its own took 10 us).
              if (p.clear_c && owner != p.rank) __builtin_nontemporal_store((u32x4_t){0u, 0u, 0u, 0u}, (u32x4_t*)(p.C + eoff));
            }
            if (solo && (p.all_owners || owner == p.rank)) {
              if (p.epi == EPI_TWO_SHOT) {
                for (int pr = 0; pr < p.world; ++pr) __builtin_nontemporal_store(v, (u32x4_t*)(in_slot(c_base, pr) + eoff));
              } else {
                const int dst = p.all_owners ? owner : p.rank;
                __builtin_nontemporal_store(v, (u32x4_t*)(in_slot(c_base, dst) + eoff));
              }
            }
          }
        }
      }
    }

    PHASE_STAMP(4);
    if (flags) {
      // Publish: the aux tile was stored write-through at system scope; every wave waits until its
      // stores are acknowledged, the workgroup meets, and the threads that own flags raise them
      // (no L2 write-back is needed any more).  The peers' flags are polled by one set of threads for
      // the whole workgroup (relaxed loads, one acquire when a flag is up); letting every wave poll
      // and run ahead measured slower.
      // The peers' flags are looked at once while the own stores are still on their way: a thread that
      // found the flags it is responsible for up already - peers that finished first - has their round
      // trip hidden behind that wait and does not poll after the own flags are raised.  Every thread
      // knows only about its own flags; the barrier behind the polling makes it common knowledge.
      const bool up_already = solo ? true : probe_peer_flags<BM, BN, NT>(p, m0, n0, tid);
      wait_vmcnt<0>();
      __syncthreads();
      PHASE_STAMP(5);
      raise_flags<BM, BN, NT, true>(p, m0, n0, tid);
      if (!solo) {
        if (!up_already) wait_peer_flags<BM, BN, NT>(p, m0, n0, tid);
        __syncthreads();
      }
      PHASE_STAMP(6);

      // Phase 2: reduce the flag tiles this rank is responsible for.  The peer loads are issued
      // unconditionally (rows this thread does not reduce read the tile origin instead) and for a
      // compile-time number of peers, so that all loads of a group of passes are in flight
      // together; only the stores are predicated.
      const bool ref_chain = (p.acc_mode == IRIS_HIP_ACC_REFERENCE) && !Out::kFp32SumInReference;
      const unsigned long long aux_own = (unsigned long long)p.aux, c_own = (unsigned long long)p.C;
      const int ftn = cdiv(p.N, p.flag_bn);
      const int ftotal = cdiv(p.M, p.flag_bm) * ftn;
      const int fcol = gn / p.flag_bn;
      const int npeers = p.sum_peers ? p.world - 1 : 0;
      // Peer aux bases in ascending rank order, own rank skipped.
      unsigned long long pb[kMaxCachedSlots - 1];
#pragma unroll
      for (int i = 0; i < kMaxCachedSlots - 1; ++i) pb[i] = (i < p.rank ? hb[i] : hb[i + 1]) + (aux_own - hb_own);
      const long long safe_off = ((long long)m0 * p.s_cm + n0) * 2;  // first element of the tile

      // The peers' tiles are read once and C is written once.  C, and the peers' tiles of launches that move more than
      // the last-level cache takes in, go past the caches' keep policy (non-temporal): they neither displace the operands nor -
      // what costs more - make that cache write back whatever dirty lines it holds (4096 x 4096 x 1376
      // bf16 with seven peers, after a 256 MB buffer had been zeroed: phase 2 68 -> 39 us).  Smaller launches read the peers' tiles
      // through the caches (peers_past_caches in iris_hip.hip has the line and the figures).
      // Chunks are handed to the threads either over the whole kernel tile (RECT false: thread t
      // takes chunk t of every pass, ownership looked up per chunk) or over one rectangle of it,
      // rows [r0, r1) and `ncw` chunks from column c0, all of which `rect_owner` reduces (RECT true).
      auto reduce_chunks = [&](auto np_tag, auto nt_tag, auto rect_tag, int r0, int r1, int c0, int ncw, int rect_owner) {
        constexpr int NP = decltype(np_tag)::value;  // peers with cached bases; -1: any number
        constexpr bool RECT = decltype(rect_tag)::value;
        auto load_peer = [](unsigned long long at) {
          return decltype(nt_tag)::value ? __builtin_nontemporal_load((const u32x4_t*)at) : *(const u32x4_t*)at;
        };
        constexpr int NPV = NP > 0 ? NP : 1;
        const int npasses = RECT ? cdiv((r1 - r0) * ncw, NT) : PASSES;
        // One pass of the workgroup: the addresses of this thread's chunk, the peers' chunks requested, the
        // own chunk read from LDS ...
        struct Pass {
          bool active;
          long long eoff;
          int owner;
          u32x4_t own, pv[NPV];
        };
        auto issue = [&](int ps, Pass& st) {
          int gm, gc, lds_off;
          if constexpr (RECT) {
            const unsigned idx = (unsigned)(ps * NT + tid);
            const unsigned row = idx / (unsigned)ncw;
            gm = r0 + (int)row;
            gc = c0 + (int)(idx - row * (unsigned)ncw) * 8;
            st.owner = rect_owner;
            st.active = gm < r1;
            lds_off = st.active ? CFG::stage_offset(gm - m0, (gc - n0) * 2) : CFG::stage_offset(0, 0);
          } else {
            gm = m0 + ps * RPP + t_row;
            gc = gn;
            st.owner = p.rank;
            if (p.epi != EPI_ONE_SHOT) {  // one-shot reduces every tile: no owner arithmetic
              const int t = (gm / p.flag_bm) * ftn + fcol;
              st.owner = owner_of(p.epi, t, ftotal, p.world, p.rank);
            }
            st.active = gm < p.M && col_ok && (p.all_owners || st.owner == p.rank);
            lds_off = t_pass[ps & 1] + ps * RPP * CFG::TROW;
          }
          st.eoff = st.active ? ((long long)gm * p.s_cm + gc) * 2 : safe_off;
          if constexpr (NP > 0) {
#pragma unroll
            for (int i = 0; i < NP; ++i) st.pv[i] = load_peer(pb[i] + st.eoff);
          }
          st.own = *(const LDS_AS u32x4_t*)(LDS_AS char*)(smem + lds_off);
        };
        // ... and its second half: the fp32 sum in ascending rank order from the own value, one cast, the stores.
        auto finish = [&](const Pass& st) {
          float sum[8];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            sum[2 * e] = Out::to_float((unsigned short)(st.own[e] & 0xFFFF));
            sum[2 * e + 1] = Out::to_float((unsigned short)(st.own[e] >> 16));
          }
          auto add_peer = [&](const u32x4_t& v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              sum[2 * e] += Out::to_float((unsigned short)(v[e] & 0xFFFF));
              sum[2 * e + 1] += Out::to_float((unsigned short)(v[e] >> 16));
            }
            if (ref_chain) {
#pragma unroll
              for (int e = 0; e < 8; ++e) sum[e] = Out::to_float(Out::from_float(sum[e]));
            }
          };
          if constexpr (NP > 0) {
#pragma unroll
            for (int i = 0; i < NP; ++i) add_peer(st.pv[i]);
          } else if constexpr (NP < 0) {
            for (int pr = 0; pr < p.world; ++pr)
              if (pr != p.rank) add_peer(load_peer(in_slot(aux_own, pr) + st.eoff));
          }
          u32x4_t res;
#pragma unroll
          for (int e = 0; e < 4; ++e) res[e] = Out::pack(sum[2 * e], sum[2 * e + 1]);
          if (st.active) {
            if (p.epi == EPI_TWO_SHOT) {
              __builtin_nontemporal_store(res, (u32x4_t*)(c_own + st.eoff));
              for (int pr = 0; pr < p.world; ++pr)
                if (pr != p.rank) __builtin_nontemporal_store(res, (u32x4_t*)(in_slot(c_own, pr) + st.eoff));
            } else {
              const int dst = p.all_owners ? st.owner : p.rank;
              __builtin_nontemporal_store(res, (u32x4_t*)((dst == p.rank ? c_own : in_slot(c_own, dst)) + st.eoff));
            }
          }
        };
        if constexpr (NW == 8 && NP >= 4 && ONE_ROUND) {
          // Eight-wave tile with many peers, one tile per workgroup: the passes run as a pipeline of DEPTH
          // stages - the loads of the next pass are on their way while one pass is summed and stored - so
          // that the bytes a CU has in flight do not fall to zero between groups of passes (4096 x 4096 x 1376
          // with seven peers: 92.9 -> 90.8 us against groups of two passes; three stages spill and gain
          // nothing more).  Looping workgroups keep the groups: their launches run 1-7 % slower with the
          // pipeline (fp8 16384 x 8192 x 1024: 494 -> 501 us with two stages, 527 with three) - a CU takes
          // no more than about 39 GB/s of such loads however many are in flight, and the steadier stream
          // of one workgroup only takes bandwidth from the others that are streaming at the time.  The
          // four-wave tiles gain nothing from a pipeline of four stages either (-2 to +3 % over ten shapes).
          constexpr int DEPTH = IRIS_HIP_EPILOGUE_DEPTH;
          const int last = RECT ? npasses : min(PASSES, cdiv(p.M - m0, RPP));  // passes below the last row of the matrix are skipped
          Pass st[DEPTH];
#pragma unroll
          for (int d = 0; d < DEPTH; ++d)
            if (d < last) issue(d, st[d]);
          for (int ps = 0; ps < last; ps += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
              if (ps + d < last) {
                finish(st[d]);
                if (ps + d + DEPTH < last) issue(ps + d + DEPTH, st[d]);
              }
            }
          }
        } else {
          // Passes whose loads are issued together.  Every group is one memory round trip (2 us on a
          // launch of 10-20 us), so the four-wave tiles, which have the registers, take four passes
          // at a time also with seven peers, and groups below the last row of the matrix are skipped.
          constexpr int G0 = (NP >= 4 && NW == 8) ? 2 : 4;
          constexpr int G = G0 < PASSES ? G0 : PASSES;
          static_assert(PASSES % G == 0, "pass grouping");
          for (int pg = 0; pg < npasses; pg += G) {
            if (!RECT && m0 + pg * RPP >= p.M) break;
            Pass st[G];
#pragma unroll
            for (int g = 0; g < G; ++g) issue(pg + g, st[g]);
#pragma unroll
            for (int g = 0; g < G; ++g) finish(st[g]);
          }
        }
      };
      // Variants with tile owners (two-shot, reduce-scatter): only the flag tiles this rank owns are
      // reduced, and a kernel tile may hold none, one or several of them.  When the flag tiles are
      // large enough to keep the workgroup busy, each owned one is streamed as a rectangle by all
      // threads, and a kernel tile without an owned flag tile issues nothing at all; with small flag
      // tiles the threads keep their places in the kernel tile and the stores are predicated.
      auto reduce_tile = [&](auto np_tag, auto nt_tag) {
        const int m1 = min(m0 + BM, p.M), n1 = min(n0 + BN, p.N);
        const bool by_rect = p.epi != EPI_ONE_SHOT && min(p.flag_bm, BM) * (min(p.flag_bn, BN) / 8) * 2 >= NT;
        if (!by_rect) {
          reduce_chunks(np_tag, nt_tag, std::false_type{}, 0, 0, 0, 0, 0);
          return;
        }
        for (int fr = m0 / p.flag_bm; fr * p.flag_bm < m1; ++fr)
          for (int fc = n0 / p.flag_bn; fc * p.flag_bn < n1; ++fc) {
            const int owner = owner_of(p.epi, fr * ftn + fc, ftotal, p.world, p.rank);
            if (!p.all_owners && owner != p.rank) continue;
            const int r0 = max(m0, fr * p.flag_bm), r1 = min(m1, (fr + 1) * p.flag_bm);
            const int c0 = max(n0, fc * p.flag_bn), c1 = min(n1, (fc + 1) * p.flag_bn);
            reduce_chunks(np_tag, nt_tag, std::true_type{}, r0, r1, c0, (c1 - c0) / 8, owner);
          }
      };
      auto reduce_with = [&](auto np_tag) {
        if (p.stream_peers) reduce_tile(np_tag, std::true_type{});
        else reduce_tile(np_tag, std::false_type{});
      };
      switch (solo ? -2 : (p.world <= kMaxCachedSlots ? npeers : -1)) {
        case -2: break;  // C was written in phase 1
        case 1: reduce_with(std::integral_constant<int, 1>{}); break;
        case 3: reduce_with(std::integral_constant<int, 3>{}); break;
        case 7: reduce_with(std::integral_constant<int, 7>{}); break;
        // (Other numbers of ranks always read past the caches: with both ways for them the kernel of eight, e4m3 16384x8192x1024,
        // goes from 499 to 506 us, and three ranks bf16 8192x4096x640 from 101.2 to 104.1; small launches would gain, six 2048x2880x640
        // 35.4 -> 30.1.)
        default: reduce_tile(std::integral_constant<int, -1>{}, std::true_type{}); break;
      }
    }
    PHASE_STAMP(7);
#ifdef IRIS_HIP_PHASE_STAMPS
    wait_vmcnt<0>();
    PHASE_STAMP(8);
#endif
    }  // !ANY_ROWS
    // Staging shares LDS with the operand ring of the next tile: every wave must be done reading it.
    // A bare barrier - __syncthreads() would also wait for this tile's global stores to be
    // acknowledged (1-4 us), which nothing here depends on; they drain behind the next tile's
    // first loads, or behind the end of the kernel.
    __builtin_amdgcn_s_waitcnt((0xF) | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0), vmcnt and expcnt free
    __builtin_amdgcn_s_barrier();
  }
}

// ------------------------------------------------------------------------------------------------
// Launch of the MFMA kernel
// ------------------------------------------------------------------------------------------------
template <class CFG, bool ONE_ROUND, bool STREAMK = false, bool ANY_ROWS = false>
int launch_mfma_grid(const FusedParams& p, int device, int grid, hipStream_t stream) {
  // The dynamic-LDS limit is a per-device attribute of the kernel: set it once on every device used
  // (atomic flags: two host threads may both set it, which is harmless, but neither skips it).
  static std::atomic<bool> attr_set[64];
  if (device < 0 || device >= 64) return iris_host::fail("device index %d out of range", device);
  if (!attr_set[device].load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute((const void*)fused_mfma_kernel<CFG, ONE_ROUND, STREAMK, ANY_ROWS>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, CFG::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    attr_set[device].store(true, std::memory_order_release);
  }
  hipLaunchKernelGGL((fused_mfma_kernel<CFG, ONE_ROUND, STREAMK, ANY_ROWS>), dim3(grid), dim3(CFG::NT), CFG::SMEM_BYTES, stream, p);
  return (int)hipGetLastError();
}

// Tail policy of the eight-wave tile (the STREAMK builds of the kernel): worth it when the last round of
// workgroups would leave a good part of the chip without a tile for many K steps.  Returns the grid to
// launch (every CU, a multiple of the XCD count) or 0 when tiles are better handed out whole.
//   iris_hip_set_split_tiles(0) / IRIS_HIP_STREAMK=0 never splits, 1 splits whenever the last round is
//   not full and has at least 4 K steps, -1 (default) decides by the rule below.  Results differ from the unsplit launch only in
//   the order of the fp32 sums over K.
template <class CFG>
int split_tile_grid(FusedParams& p, int total, int cu_count) {
  if constexpr (CFG::NW != 8) return 0;
  const int mode = iris_host::split_tile_mode();
  if (mode == 0 || p.no_workspace_alloc || p.num_xcd < 1) return 0;
  const int grid = cu_count - cu_count % p.num_xcd;
  if (grid < p.num_xcd) return 0;
  const int wg_per_xcd = grid / p.num_xcd;
  const int span = cdiv(total, p.num_xcd);     // tiles of an XCD (the last one may have fewer)
  const int left = span % wg_per_xcd;          // tiles of its last, partly filled round
  if (left == 0) return 0;
  const int nsrc = p.gather == GATHER_K ? p.world : 1;
  const int nsteps = nsrc * cdiv(p.gather == GATHER_K ? p.K_local : p.K, CFG::BK);
  // Mode 1 plans without the costs of passing partial sums on: whatever can be split is split.
  p.sk_gather_cost = mode == 1 ? 0 : kSplitGatherCost;
  p.sk_pass_cost = mode == 1 ? 0 : kSplitPassCost;
  const SplitPlan plan = split_plan(left, wg_per_xcd, nsteps, p.sk_gather_cost, p.sk_pass_cost);
  if (plan.per_tile == 0) return 0;
  if (mode == 1 || mode == 2) return grid;  // 2: whatever the plan expects any gain from (a tuning aid)
  // Worth it when the split round is at least 16 K steps (12 us) and an eighth shorter than a whole tile.
  const int steps = split_round_steps(plan, nsteps);
  return (nsteps - steps >= 16 && (nsteps - steps) * 8 >= nsteps) ? grid : 0;
}

template <class CFG>
int launch_mfma(const FusedParams& p, int device, int cu_count, hipStream_t stream, const char* name) {
  const int total = p.tiles_m * p.tiles_n;
  const int cap = cu_count * CFG::WG_PER_CU;
  const int grid = resident_grid(total, cap, p.num_xcd);
  iris_host::set_last_kernel(name);
  const bool per_tile_launch = total > grid && workgroup_per_tile(p.epi, p.world, p.sum_peers, p.all_owners);
  if constexpr (CFG::NW == 8) {
    FusedParams q = p;
    const int sk_grid = per_tile_launch ? 0 : split_tile_grid<CFG>(q, total, cu_count);
    if (sk_grid > 0) {
      q.interleave = 0;  // the plan hands out the last round of every XCD's span
      q.tile_rotate = 0;
      q.group_m = q.group_m_spans;
      constexpr long long slot_bytes = (long long)CFG::MB * CFG::NB * CFG::QUADS * CFG::NT * 16;
      // No workspace (the stream is being captured before its first split launch, or the device has
      // used up its workspaces): hand the tiles out whole.
      if (iris_host::split_tile_workspace(device, stream, sk_grid, slot_bytes, &q.sk_partials, &q.sk_flags, &q.sk_epoch) == 0) {
        char sk_name[112];
        snprintf(sk_name, sizeof(sk_name), "%s_splitk", name);
        iris_host::set_last_kernel(sk_name);
        return launch_mfma_grid<CFG, false, true>(q, device, sk_grid, stream);
      }
    }
  }
  if (total <= grid) return launch_mfma_grid<CFG, true>(p, device, grid, stream);
  // More tiles than workgroups that fit at once: the resident workgroups loop over the tiles, or get one each in turn.
  if (per_tile_launch) {
    int per_tile = total;
    if (per_tile % p.num_xcd) per_tile += p.num_xcd - per_tile % p.num_xcd;
    return launch_mfma_grid<CFG, true>(p, device, per_tile, stream);
  }
  return launch_mfma_grid<CFG, false>(p, device, grid, stream);
}

// Tile shapes of the MFMA kernel (run_fused picks one per launch).
//   big       256x256, 8 waves, 64-byte K steps, 5-slot ring: half the operand bytes per flop of the
//             128x128 tiles; from about half the CUs busy.
//   small     128x128, 4 waves, 128-byte K steps, 4-slot ring: too few big tiles.
//   small2    128x128, 4 waves, 64-byte K steps, 64 KiB ring, two workgroups per CU: more 128x128 tiles
//             than CUs (every tile resident at once instead of a half-empty second round).
//   skinny    64x128, 4 waves, 128-byte K steps, 72 KiB ring, two workgroups per CU: at most 64 rows, or at
//             most two such tiles per CU with a short K.
//   skinny64  64x64, 4 waves of one 32x32 block, 128-byte K steps, 64 KiB ring, two workgroups per CU: at
//             most two such tiles per CU.
// For the small tiles residency - every tile of the output on a CU at once - pays before fat K steps.
enum { TILE_BIG = 0, TILE_SMALL = 1, TILE_SKINNY = 2, TILE_SMALL2 = 3, TILE_DECODE = 4, TILE_SKINNY64 = 5 };
constexpr int tile_bk(int kind, int in) {  // K elements per step
  return (kind == TILE_BIG || kind == TILE_SMALL2 ? 64 : 128) / (in == IN_FP8 ? 1 : 2);
}
template <int IN, bool BKC>
using BigTile = MfmaCfg<IN, 256, 256, tile_bk(TILE_BIG, IN), 2, 4, 5, BKC>;
template <int IN, bool BKC>
using SmallTile = MfmaCfg<IN, 128, 128, tile_bk(TILE_SMALL, IN), 2, 2, 4, BKC>;
template <int IN, bool BKC>
using SkinnyTile = MfmaCfg<IN, 64, 128, tile_bk(TILE_SKINNY, IN), 2, 2, 3, BKC>;
template <int IN, bool BKC>
using Small2Tile = MfmaCfg<IN, 128, 128, tile_bk(TILE_SMALL2, IN), 2, 2, 4, BKC>;
template <int IN, bool BKC>
using Skinny64Tile = MfmaCfg<IN, 64, 64, tile_bk(TILE_SKINNY64, IN), 2, 2, 4, BKC>;

inline int tile_rows(int kind) {
  return kind == TILE_BIG ? 256 : (kind == TILE_SKINNY || kind == TILE_SKINNY64) ? 64 : kind == TILE_DECODE ? 32 : 128;
}
inline int tile_cols(int kind) { return kind == TILE_BIG ? 256 : kind == TILE_DECODE ? 32 : kind == TILE_SKINNY64 ? 64 : 128; }

// The 32x32 kernel (decode_kernel.h), in translation units of its own: what the compiler makes of a kernel depends on the other
// kernels of its module (beside the tiles the fp16 builds changed with every edit here: 32x2880x512, eight ranks, 7.20 -> 7.30 us).
// Instantiated in iris_hip_decode_<type>.hip.
template <int IN>
int dispatch_decode(FusedParams& p, bool bkc, int device, int cu, hipStream_t s);

inline TileLaunch tile_launch(const FusedParams& p, int kind, int cu) {
  const int two_per_cu = !(kind == TILE_BIG || kind == TILE_SMALL);
  return {p.M, p.N, tile_rows(kind), tile_cols(kind), p.num_xcd, (cu / p.num_xcd) * (1 + two_per_cu), two_per_cu,
          p.epi, p.world, p.rank, p.sum_peers, p.all_owners, p.flag_bm, p.flag_bn};
}

// The tiles of a launch and their order.
inline void plan_tiles(FusedParams& p, int kind, int cu) {
  const TileOrder o = tile_order(tile_launch(p, kind, cu));
  p.tiles_m = o.tiles_m;
  p.tiles_n = o.tiles_n;
  p.interleave = o.interleave;
  p.tile_rotate = o.tile_rotate;
  p.group_m_spans = o.group_m_spans;
  int g = o.group_m;
  const bool rs_band = p.epi == EPI_REDUCE_SCATTER && !p.all_owners && p.sum_peers && p.world > 1;
  static const int forced_order = [] {
    const char* e = getenv("IRIS_HIP_TILE_ORDER");  // "spans" or "dealt": a tuning aid, the same on all ranks
    return !e ? -1 : (e[0] == 'd' ? 1 : 0);
  }();
  if (forced_order >= 0) p.interleave = forced_order;
  if (!p.interleave) {
    if (rs_band) g = p.group_m_spans;
    p.tile_rotate = 0;
  }
  // IRIS_HIP_GROUP_M overrides the group height (a tuning aid; results do not depend on the tile order).
  static const int forced_group_m = [] { const char* e = getenv("IRIS_HIP_GROUP_M"); return e ? atoi(e) : 0; }();
  if (forced_group_m > 0) {
    g = forced_group_m < p.tiles_m ? forced_group_m : p.tiles_m;
    p.group_m_spans = g;
  }
  p.group_m = g;
}

template <int IN>
int dispatch_mfma_in(FusedParams& p, int kind, bool bkc, int device, int cu, hipStream_t s) {
  if (kind == TILE_DECODE) return dispatch_decode<IN>(p, bkc, device, cu, s);
  plan_tiles(p, kind, cu);
  const int bm = tile_rows(kind), bn = tile_cols(kind);
  static const char* names[3] = {"bf16", "f16", "fp8"};
  char name[96];
  snprintf(name, sizeof(name), "mfma_%s_%dx%dx%d_%s", names[IN], bm, bn, tile_bk(kind, IN), bkc ? "nt" : "nn");
  switch (kind) {
    case TILE_BIG:
      return bkc ? launch_mfma<BigTile<IN, true>>(p, device, cu, s, name) : launch_mfma<BigTile<IN, false>>(p, device, cu, s, name);
    case TILE_SMALL:
      return bkc ? launch_mfma<SmallTile<IN, true>>(p, device, cu, s, name) : launch_mfma<SmallTile<IN, false>>(p, device, cu, s, name);
    case TILE_SMALL2:
      return bkc ? launch_mfma<Small2Tile<IN, true>>(p, device, cu, s, name) : launch_mfma<Small2Tile<IN, false>>(p, device, cu, s, name);
    case TILE_SKINNY64:
      return bkc ? launch_mfma<Skinny64Tile<IN, true>>(p, device, cu, s, name) : launch_mfma<Skinny64Tile<IN, false>>(p, device, cu, s, name);
    default:
      return bkc ? launch_mfma<SkinnyTile<IN, true>>(p, device, cu, s, name) : launch_mfma<SkinnyTile<IN, false>>(p, device, cu, s, name);
  }
}

// ANY_ROWS builds, in translation units of their own (iris_hip_rows_<type>.hip): one workgroup per tile, in the order of plan_tiles.
template <class CFG>
int launch_mfma_rows(const FusedParams& p, int device, hipStream_t s, const char* name) {
  iris_host::set_last_kernel(name);
  return launch_mfma_grid<CFG, true, false, true>(p, device, cdiv(p.tiles_m * p.tiles_n, p.num_xcd) * p.num_xcd, s);
}

template <int IN>
int dispatch_mfma_rows(const FusedParams& p, int kind, bool bkc, int device, hipStream_t s) {
  static const char* names[3] = {"bf16", "f16", "fp8"};
  char name[96];
  snprintf(name, sizeof(name), "mfma_%s_%dx%dx%d_%s_rows", names[IN], tile_rows(kind), tile_cols(kind), tile_bk(kind, IN), bkc ? "nt" : "nn");
  switch (kind) {
    case TILE_BIG:
      return bkc ? launch_mfma_rows<BigTile<IN, true>>(p, device, s, name) : launch_mfma_rows<BigTile<IN, false>>(p, device, s, name);
    case TILE_SMALL:
      return bkc ? launch_mfma_rows<SmallTile<IN, true>>(p, device, s, name) : launch_mfma_rows<SmallTile<IN, false>>(p, device, s, name);
    case TILE_SMALL2:
      return bkc ? launch_mfma_rows<Small2Tile<IN, true>>(p, device, s, name) : launch_mfma_rows<Small2Tile<IN, false>>(p, device, s, name);
    default:
      return bkc ? launch_mfma_rows<Skinny64Tile<IN, true>>(p, device, s, name) : launch_mfma_rows<Skinny64Tile<IN, false>>(p, device, s, name);
  }
}
