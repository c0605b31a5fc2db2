// fused_any_kernel: every operator on operands of any alignment, stride, size and element type - what the
// direct-to-LDS kernels of fused_kernel.h do not take: rows that do not start on 16-byte boundaries (an odd N
// or K), float32 data, A or B without a unit stride, an output row stride that is not a multiple of 8.
//
// Where it differs from those kernels is the way of the operands: 16-byte pieces travel HBM -> registers ->
// LDS (global loads take any alignment; the direct-to-LDS load is used only where its pieces are
// aligned), one K step ahead in registers and one in the second LDS buffer.  The LDS layouts, the MFMA
// operand lanes and the order of the epilogue are the same.  What bounds it on the small tiles is no unit's rate but
// the K step's chain - loads, LDS, barrier, fragments, products - which two or three workgroups per CU only partly hide
// (over one launch of 64x128 tiles with its exchange: bf16 1999x2877x1371 MFMA 10 %, VALU 19 %, LDS 15 % busy; float32, as
// three bf16 pieces per operand, 2048x2880x1024 27 %, 37 %, 23 %); with peers the epilogue's HBM streams come on top.
//
// Nothing on the hot path is predicated: rows past M (or N) repeat the last row, columns of B past N are
// read as they lie in memory as long as the piece ends inside the operand - what they produce are output
// rows and columns that do not exist and are not stored.  Only k beyond K has to be zero on both sides
// (the other operand may hold NaN there); those pieces are loaded element by element in the last K step
// of a source.
#pragma once

#include "fused_kernel.h"

constexpr int IN_F32 = 3;  // next to IN_BF16, IN_F16, IN_FP8

template <int IN> struct AnyIn;
template <> struct AnyIn<IN_BF16> { static constexpr int ES = 2; };
template <> struct AnyIn<IN_F16> { static constexpr int ES = 2; };
template <> struct AnyIn<IN_FP8> { static constexpr int ES = 1; };
template <> struct AnyIn<IN_F32> { static constexpr int ES = 4; };

// [k][n] tile of B in LDS, n contiguous.  16- and 8-bit data use the transpose-read layout of ColTile; a
// float32 fragment is four 4-byte reads per lane, row k for the first half-wave and row k + 4 for the second,
// 32 consecutive columns (128 bytes) each: the 128-byte blocks of rows with bit 2 of k set change
// places, so that the halves meet on different banks (rows of 256 bytes and more).
template <int RB, int ES>
struct AnyColTile : ColTile<RB, ES> {};
template <int RB>
struct AnyColTile<RB, 4> {
  IRIS_HD static int lds_offset(int krow, int c) {
    return krow * RB + ((RB >= 256 ? c ^ (((krow >> 2) & 1) * 8) : c) * kChunkBytes);
  }
};

// A workgroup computes BM x BN outputs with WM x WN x WK waves: a wave owns a (BM/WM) x (BN/WN) block, and with
// WK > 1 every WK-th 128-byte slice of K (the partial blocks meet in LDS at the end).
template <int IN_, class Out_, int BM_, int BN_, int WM_, int WN_, int WK_, bool BKC_>
struct AnyCfg {
  static constexpr int IN = IN_;
  using Out = Out_;
  static constexpr int ES = AnyIn<IN>::ES;
  static constexpr int CE = kChunkBytes / ES;
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_;
  static constexpr bool BKC = BKC_;  // B as [n][k] (K-contiguous, or no unit stride at all), else [k][n]
  static constexpr int NW = WM * WN * WK, NT = 64 * NW;
  static constexpr int TM = BM / WM, TN = BN / WN, MB = TM / 32, NB = TN / 32;
  static constexpr int KB = 128;               // bytes of K per row and slice
  static constexpr int KE = KB / ES;           // ... in elements
  static constexpr int KSTEP = KE * WK;        // elements of K per step of the workgroup
  static constexpr int KM = IN == IN_FP8 ? 64 : IN == IN_F32 ? 8 : 16;  // k per fragment
  static constexpr int KS = KE / KM;
  static constexpr int NFRAG = IN == IN_FP8 ? 2 : 1;
  static constexpr int RBB = BKC ? KB : BN * ES;
  static constexpr int A_SLICE = BM * KB, B_SLICE = BN * KB;
  static constexpr int A_BYTES = A_SLICE * WK, B_BYTES = B_SLICE * WK;
  static constexpr int BUF_BYTES = A_BYTES + B_BYTES;
  static constexpr int LA = A_BYTES / kChunkBytes / NT, LB = B_BYTES / kChunkBytes / NT;
  static constexpr int CPR = BN * ES / kChunkBytes;  // pieces per row of a [k][n] tile
  // Staged output tile: rows padded by 16 bytes against bank conflicts of the accumulator layout.
  static constexpr int OE = kChunkBytes / Out::size;  // output elements per piece
  static constexpr int TROW = BN * Out::size + 16;
  static constexpr int TILE_BYTES = BM * TROW;
  // Partial blocks of the waves along K: fp32, one 36-float row per output row, next to each other.
  static constexpr int PART_ROW = BN * 4 + 16;
  static constexpr int PART_BYTES = WK > 1 ? WK * BM * PART_ROW : 0;
  // float32 as three bf16 pieces (where the kernel says why): a step's tiles of A and of B, three planes each.
  // Eight waves, alone on their CU, split one step while they multiply another and need two buffers; workgroups of
  // four share a CU and take turns.
  static constexpr bool SPLIT = IN == IN_F32 && WK == 1;
  static constexpr int KB16 = KE * 2;  // bytes of K per row of a plane
  static constexpr int A_PLANE = BM * KB16, B_PLANE = BN * KB16;
  static constexpr int SPLIT_BUF = 3 * (A_PLANE + B_PLANE), SPLIT_BYTES = !SPLIT ? 0 : NW == 8 ? 2 * SPLIT_BUF : SPLIT_BUF;
  static constexpr int SMEM0 = 2 * BUF_BYTES > TILE_BYTES ? 2 * BUF_BYTES : TILE_BYTES;
  static constexpr int SMEM1 = SMEM0 > TILE_BYTES + PART_BYTES ? SMEM0 : TILE_BYTES + PART_BYTES;
  static constexpr int FLAG_OFF = SMEM1 > SPLIT_BYTES ? SMEM1 : SPLIT_BYTES;  // SPLIT: the workgroup's vote
  static constexpr int SMEM_BYTES = FLAG_OFF + (SPLIT ? kChunkBytes : 0);
  static constexpr int WG_PER_CU = NW != 4 ? 1 : !SPLIT ? 2 : 160 * 1024 / SMEM_BYTES < 3 ? 160 * 1024 / SMEM_BYTES : 3;
  static_assert(SMEM_BYTES * WG_PER_CU <= 160 * 1024, "LDS budget of a gfx950 CU");
  static_assert((BM * 8) % NT == 0 && (BN * 8) % NT == 0 && NT % CPR == 0, "whole pieces per thread");
};

template <class CFG>
__global__ void __launch_bounds__(CFG::NT, CFG::WG_PER_CU * CFG::NW / 4) fused_any_kernel(const FusedParams p) {
  using Out = typename CFG::Out;
  constexpr int IN = CFG::IN, ES = CFG::ES, CE = CFG::CE, BM = CFG::BM, BN = CFG::BN, NT = CFG::NT, KE = CFG::KE, KS = CFG::KS;
  constexpr int LA = CFG::LA, LB = CFG::LB, MB = CFG::MB, NB = CFG::NB, NFRAG = CFG::NFRAG, OE = CFG::OE;
  using ATile = RowTile<CFG::KB>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (CFG::WM * CFG::WN), wm = wave / CFG::WN % CFG::WM, wn = wave % CFG::WN;

  const int tidx = xcd_tile_index(blockIdx.x, gridDim.x, 0, p.tiles_m * p.tiles_n, p.interleave ? 1 : p.num_xcd);
  if (tidx < 0) return;
#ifdef IRIS_HIP_PHASE_STAMPS
  constexpr int it = 0;  // PHASE_STAMP records the first tile of a workgroup; there is only one here
#endif
  PHASE_STAMP(0);
  int tm, tn;
  grouped_tile(tidx, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  const int nsrc = (p.gather == GATHER_K) ? p.world : 1;
  const int klocal = (p.gather == GATHER_K) ? p.K_local : p.K;
  const int nkb = cdiv(klocal, CFG::KSTEP);
  const int nsteps = nsrc * nkb;

  // ---- loaders: which pieces this thread fetches, from where, and where they live in LDS ---------------
  // Consecutive threads take consecutive pieces of a row; with a strided operand consecutive rows, so that
  // a transposed A (rows one element apart) is still read in whole lines.
  const bool a_vec = p.s_ak == 1;
  const char* ptr[LA + LB];  // (A's pieces first, then B's)
  int a_k[LA], lds_at[LA + LB];
  int f_kb, f_src;  // K step the next fetch brings
  auto point_at_a = [&](auto split_tag) INLINED {
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int id = tid + i * NT, sub = id / (BM * 8), in_sub = id - sub * (BM * 8);
      const int row = a_vec ? in_sub >> 3 : in_sub % BM, c = a_vec ? in_sub & 7 : in_sub / BM;
      a_k[i] = sub * KE + c * CE;
      if constexpr (decltype(split_tag)::value) lds_at[i] = RowTile<CFG::KB16>::lds_offset(row, c >> 1) + (c & 1) * 8;
      else lds_at[i] = sub * CFG::A_SLICE + ATile::lds_offset(row, c);
      long long gm = min(m0 + row, p.M - 1);
      int slot = p.gather == GATHER_K ? 0 : p.rank;
      if (p.gather == GATHER_M) {
        slot = (int)(gm / p.M_local);
        gm -= (long long)slot * p.M_local;
      }
      const char* base = p.gather == GATHER_NONE ? p.A : slot_ptr(p.heap_bases, p.A, p.rank, slot);
      ptr[i] = base + (gm * p.s_am + (long long)a_k[i] * p.s_ak) * ES;
    }
    f_kb = f_src = 0;
  };
  const bool b_vec = !CFG::BKC || p.s_bk == 1;
  int b_k[LB];
  int b_cols;  // [k][n] tile: columns of this thread's piece that exist
  auto point_at_b = [&](auto split_tag) INLINED {
    constexpr bool SPLIT = decltype(split_tag)::value;
    b_cols = CE;
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int id = tid + i * NT;
      if constexpr (CFG::BKC) {
        const int sub = id / (BN * 8), in_sub = id - sub * (BN * 8);
        const int row = b_vec ? in_sub >> 3 : in_sub % BN, c = b_vec ? in_sub & 7 : in_sub / BN;
        b_k[i] = sub * KE + c * CE;
        if constexpr (SPLIT) lds_at[LA + i] = 3 * CFG::A_PLANE + RowTile<CFG::KB16>::lds_offset(row, c >> 1) + (c & 1) * 8;
        else lds_at[LA + i] = CFG::A_BYTES + sub * CFG::B_SLICE + ATile::lds_offset(row, c);
        ptr[LA + i] = p.B + ((long long)min(n0 + row, p.N - 1) * p.s_bn + (long long)b_k[i] * p.s_bk) * ES;
      } else {
        const int krow = id / CFG::CPR, c = id % CFG::CPR, sub = krow / KE;
        b_k[i] = krow;
        if constexpr (SPLIT) lds_at[LA + i] = 3 * CFG::A_PLANE + ColTile<BN * 2, 2>::lds_offset(krow, c >> 1) + (c & 1) * 8;
        else lds_at[LA + i] = CFG::A_BYTES + sub * CFG::B_SLICE + AnyColTile<CFG::RBB, ES>::lds_offset(krow - sub * KE, c);
        const int gn = n0 + c * CE;
        b_cols = p.N - gn;
        ptr[LA + i] = p.B + ((long long)krow * p.s_bk + (gn < p.N ? gn : 0)) * ES;  // pieces past N: any columns do
      }
    }
    if (b_cols <= 0 || b_cols > CE) b_cols = CE;
  };
  // One past the last byte of B ([k][n]); a piece that ends beyond it is loaded element by element.  With rows
  // at least a piece apart only a piece of the last row can.
  const char* const b_end = p.B + ((long long)(p.K - 1) * p.s_bk + p.N) * ES;
  const bool b_edge = !CFG::BKC && (n0 + BN > p.N || p.N < CE);
  const int b_safe_k = !b_edge ? p.K : p.s_bk >= CE ? p.K - 1 : 0;  // rows below this one can be read in whole pieces

  // Elements [0, count) of a piece, `stride` bytes apart; the rest of it zero.
  auto load_elements = [&](const char* ptr, long long stride, int count) INLINED {
    u32x4_t v = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < CE; ++e)
      if (e < count) {
        const char* q = ptr + e * stride;
        unsigned x;
        if constexpr (ES == 4) x = *(const GLOBAL_AS unsigned*)(GLOBAL_AS const char*)q;
        else if constexpr (ES == 2) x = *(const GLOBAL_AS unsigned short*)(GLOBAL_AS const char*)q;
        else x = *(const GLOBAL_AS unsigned char*)(GLOBAL_AS const char*)q;
        v[e * ES / 4] |= x << (8 * (e * ES % 4));
      }
    return v;
  };

  const long long a_step = (long long)CFG::KSTEP * p.s_ak * ES, b_step = (long long)CFG::KSTEP * p.s_bk * ES;
  u32x4_t raw[LA + LB];
  // Whether the next fetch brings nothing but whole pieces.
  auto plain = [&]() INLINED {
    return a_vec && b_vec && klocal - f_kb * CFG::KSTEP >= CFG::KSTEP && f_src * klocal + (f_kb + 1) * CFG::KSTEP <= b_safe_k;
  };
  auto advance = [&]() INLINED {
    long long da = a_step, db = b_step;
    if (++f_kb == nkb) {  // on to the next source's columns
      f_kb = 0;
      ++f_src;
      da -= nkb * a_step;
      db += (long long)klocal * p.s_bk * ES - nkb * b_step;
      if (f_src < nsrc) da += p.heap_bases[f_src] - p.heap_bases[f_src - 1];
    }
#pragma unroll
    for (int i = 0; i < LA; ++i) ptr[i] += da;
#pragma unroll
    for (int i = 0; i < LB; ++i) ptr[LA + i] += db;
  };
  auto fetch = [&]() INLINED {
    const int left = klocal - f_kb * CFG::KSTEP;  // elements of K from this step on
    if (left >= CFG::KSTEP && a_vec) {
#pragma unroll
      for (int i = 0; i < LA; ++i) raw[i] = load16_any(ptr[i]);
    } else {
#pragma unroll
      for (int i = 0; i < LA; ++i)
        raw[i] = a_vec && a_k[i] + CE <= left ? load16_any(ptr[i]) : load_elements(ptr[i], p.s_ak * ES, left - a_k[i]);
    }
    if (left >= CFG::KSTEP && b_vec && f_src * klocal + (f_kb + 1) * CFG::KSTEP <= b_safe_k) {
#pragma unroll
      for (int i = 0; i < LB; ++i) raw[LA + i] = load16_any(ptr[LA + i]);
    } else if constexpr (CFG::BKC) {
#pragma unroll
      for (int i = 0; i < LB; ++i)
        raw[LA + i] = b_vec && b_k[i] + CE <= left ? load16_any(ptr[LA + i]) : load_elements(ptr[LA + i], p.s_bk * ES, left - b_k[i]);
    } else {
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        if (b_k[i] >= left) raw[LA + i] = (u32x4_t){0u, 0u, 0u, 0u};
        else if (ptr[LA + i] + 16 <= b_end) raw[LA + i] = load16_any(ptr[LA + i]);
        else raw[LA + i] = load_elements(ptr[LA + i], ES, min(b_cols, p.N));
      }
    }
    advance();
  };
  auto put = [&](int buf) INLINED {
    char* const s = smem + buf * CFG::BUF_BYTES;
#pragma unroll
    for (int i = 0; i < LA; ++i) *(LDS_AS u32x4_t*)(LDS_AS char*)(s + lds_at[i]) = raw[i];
#pragma unroll
    for (int i = 0; i < LB; ++i) *(LDS_AS u32x4_t*)(LDS_AS char*)(s + lds_at[LA + i]) = raw[LA + i];
  };

  // ---- fragments ------------------------------------------------------------------------------------------
  struct Frag {
    i32x4_t a[MB][NFRAG], b[NB][NFRAG];
  };
  auto load_frag = [&](Frag& f, int buf, int kk) INLINED {
    const char* const sa = smem + buf * CFG::BUF_BYTES + wk * CFG::A_SLICE;
    const char* const sb = smem + buf * CFG::BUF_BYTES + CFG::A_BYTES + wk * CFG::B_SLICE;
#pragma unroll
    for (int h = 0; h < NFRAG; ++h) {
      const int c = IN == IN_FP8 ? frag8_chunk(lane, kk, h) : frag16_chunk(lane, kk);  // float32: 4 k per half-wave
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        f.a[mb][h] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sa + ATile::lds_offset(wm * CFG::TM + frag16_row(lane), c) + mb * 32 * CFG::KB);
      if constexpr (CFG::BKC) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          f.b[nb][h] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sb + ATile::lds_offset(wn * CFG::TN + frag16_row(lane), c) + nb * 32 * CFG::KB);
      }
    }
    if constexpr (!CFG::BKC) {
      using BTile = AnyColTile<CFG::RBB, ES>;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int col = wn * CFG::TN + nb * 32;
        if constexpr (IN == IN_F32) {
          const int n = col + (lane & 31), k = kk * 8 + 4 * (lane >> 5);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            f.b[nb][0][e] = *(const LDS_AS int*)(LDS_AS char*)(sb + BTile::lds_offset(k + e, n / CE) + (n % CE) * 4);
        } else if constexpr (IN == IN_FP8) {
          const int n = col + tr8_ncol(lane);
          i32x2_t t[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            t[r] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                (LDS_AS i32x2_t*)(LDS_AS char*)(sb + BTile::lds_offset(tr8_krow(lane, kk, r), n / CE) + n % CE));
          f.b[nb][0] = (i32x4_t){t[0].x, t[0].y, t[1].x, t[1].y};
          f.b[nb][NFRAG - 1] = (i32x4_t){t[2].x, t[2].y, t[3].x, t[3].y};
        } else {
          const int n = col + tr16_ncol(lane);
          i32x2_t t[2];
#pragma unroll
          for (int j = 0; j < 2; ++j)
            t[j] = __builtin_bit_cast(i32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (LDS_AS i16x4_t*)(LDS_AS char*)(sb + BTile::lds_offset(tr16_krow(lane, kk, j), n / CE) + (n % CE) * 2)));
          f.b[nb][0] = (i32x4_t){t[0].x, t[0].y, t[1].x, t[1].y};
        }
      }
    }
  };
  f32x16_t acc[MB][NB];
  auto clear_sums = [&]() INLINED {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.f;
  };
  auto multiply = [&](const Frag& f) INLINED {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if constexpr (IN == IN_F32) {
          // (element by element through a copy: bit_cast of a vector element lvalue reads element 0)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int a = f.a[mb][0][e], b = f.b[nb][0][e];
            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(__int_as_float(b), __int_as_float(a), acc[mb][nb], 0, 0, 0);
          }
        } else {
          acc[mb][nb] = mfma_block<IN, NFRAG>(f.a[mb], f.b[nb], acc[mb][nb]);
        }
      }
  };
  // Every wave's LDS accesses done, then everybody's; loads to registers stay in flight.
  auto lds_barrier = [&]() INLINED {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((0xF) | (0x3 << 14) | (0x7 << 4));  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- K loop ---------------------------------------------------------------------------------------------
  // Step s reads LDS buffer s & 1; meanwhile step s+1 arrives in registers, is put into the other buffer half
  // way through the step's products, and the loads of step s+2 go out.
  auto k_loop = [&]() INLINED {
    point_at_a(std::false_type{});
    point_at_b(std::false_type{});
    clear_sums();
    fetch();
    put(0);
    if (nsteps > 1) fetch();
    lds_barrier();
    PHASE_STAMP(1);
    for (int s = 0; s < nsteps; ++s) {
      const int buf = s & 1;
      Frag f[2];
      load_frag(f[0], buf, 0);
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        if (kk + 1 < KS) load_frag(f[(kk + 1) & 1], buf, kk + 1);
        multiply(f[kk & 1]);
        if (kk == KS / 2 - 1 && s + 1 < nsteps) {
          put(buf ^ 1);
          if (s + 2 < nsteps) fetch();
        }
      }
      lds_barrier();
    }
  };

  if constexpr (!CFG::SPLIT) {
    k_loop();
  } else {
    // float32 on the bf16 matrix pipes.  A float of at least 2^-110 (or zero) is the exact sum of three bf16
    // numbers: the value rounded to eight bits, the remainder rounded, and the rest, which fits.  Six of the nine
    // products of the pieces are added up (hi hi, hi mid, mid hi, mid mid, hi lo, lo hi); the others are at
    // most 2^-24 of the product and 2^-27 of it in the mean, below the rounding of one fp32 addition.  The sums are
    // fp32; the five smaller products have sums of their own, 2^-8 of the others, so that one addition per 16 k rounds at
    // the size of the result instead of sixteen.  Error against 64 bits, 2-norm, 1024x1024xK, float32 MFMA -> three
    // pieces (with all six products in one sum):
    //              normal operands               normal, A's negative half zero   uniform in [0, 1)
    //   K =   64   1.44e-7 -> 0.50e-7 (1.10)     1.03e-7 -> 0.41e-7 (1.06)        1.15e-7 -> 0.49e-7 (0.84)
    //       1024   5.7e-7  -> 1.9e-7  (4.9)      4.0e-7  -> 1.4e-7  (4.6)         4.3e-7  -> 1.6e-7  (2.9)
    //       8192   1.62e-6 -> 0.57e-6 (1.44)     1.15e-6 -> 0.48e-6 (1.34)        1.19e-6 -> 0.42e-6 (0.75)
    // A sum with a single product in it is the exception: what is left out comes on top of the one rounding it has with
    // the float32 MFMA (normal operands: largest error 0.5 -> 0.98 of a last place, 2-norm 2.48e-8 -> 2.52e-8; sums of two
    // products 3.1e-8 -> 2.6e-8).  K = 1, where every sum is one, is left to the float32 MFMA.  The other products of
    // pieces would bring it back for a longer K whose other products are zeros, at 2048x2880x1024 108 -> 119 us.
    // What the pieces cannot represent is left to it too, tile by tile: a nonzero operand below
    // 2^-110 (found while splitting), and tiles with a sum that is not finite (infinities and NaN, and values
    // that round to infinity in bf16), whose pieces need not add up to what the operands do.
    // The pieces are formed once per workgroup on the way from registers to LDS, 7 VALU instructions per
    // element (15.6 of the 24.5 million of a 2048x2880x1024 launch).  What bounds it: splitting, products and LDS (6 bytes
    // written per element, 9 KiB read per 12 products of a 32x64 wave block) one behind the other in a wave, 37, 27 and
    // 23 % of the launch on the 64x128 tile.  The second sums
    // cost nothing (2048x2880x1024 two-shot 109.2 -> 108.1 us) but registers: a 256x128 tile, whose waves own 64x64, has none
    // left (169 spilled) and would have to keep one sum; it is 12 % faster (4096x4096x1536 267 us, 128x128 298) with 2.6
    // times the error, more than the float32 MFMA's where half of A is zero.
    LDS_AS int* const vote = (LDS_AS int*)(LDS_AS char*)(smem + CFG::FLAG_OFF);
    if (tid == 0) *vote = 0;
    lds_barrier();
    constexpr unsigned kSmallest = ((127u - 110u) << 24) - 1u;  // 2^-110, in the form of `low`
    unsigned low = ~0u;  // smallest magnitude of a nonzero element: its bits without the sign, doubled, less one
    // One of the six parts of the splitting of a 16-byte piece v, in which v is left as the remainder:
    // elements 2 * (part & 1) and the next, plane part / 2.
    auto split_part = [&](u32x4_t& v, u32x2_t (&w)[3], int part) INLINED {
      const int e = 2 * (part & 1), i = part / 2;
      if (i == 0) low = min(low, min((v[e] << 1) - 1u, (v[e + 1] << 1) - 1u));
      const float x = __uint_as_float(v[e]), y = __uint_as_float(v[e + 1]);
      const unsigned h = pack_bf16(x, y);
      w[i][part & 1] = h;
      if (i < 2) {
        v[e] = __float_as_uint(x - __uint_as_float(h << 16));
        v[e + 1] = __float_as_uint(y - __uint_as_float(h & 0xFFFF0000u));
      }
    };
    auto put_plane = [&](const u32x2_t (&w)[3], int at, int plane, int i) INLINED {
      *(LDS_AS u32x2_t*)(LDS_AS char*)(smem + at + i * plane) = w[i];
    };
    auto put_split = [&](u32x4_t& v, int at, int plane) INLINED {
      u32x2_t w[3];
#pragma unroll
      for (int part = 0; part < 6; ++part) split_part(v, w, part);
#pragma unroll
      for (int i = 0; i < 3; ++i) put_plane(w, at, plane, i);
    };
    struct Pieces {
      i32x4_t a[MB][1], b[NB][1];
    };
    auto load_pieces = [&](Pieces& f, int buf, int kk, int i) INLINED {  // plane i of k-slice kk
      const char* const sa = smem + buf * CFG::SPLIT_BUF + i * CFG::A_PLANE;
      const char* const sb = smem + buf * CFG::SPLIT_BUF + 3 * CFG::A_PLANE + i * CFG::B_PLANE;
      const int c = frag16_chunk(lane, kk);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        f.a[mb][0] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sa + RowTile<CFG::KB16>::lds_offset(wm * CFG::TM + frag16_row(lane), c) + mb * 32 * CFG::KB16);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if constexpr (CFG::BKC) {
          f.b[nb][0] = *(const LDS_AS i32x4_t*)(LDS_AS char*)(sb + RowTile<CFG::KB16>::lds_offset(wn * CFG::TN + frag16_row(lane), c) + nb * 32 * CFG::KB16);
        } else {
          const int n = wn * CFG::TN + nb * 32 + tr16_ncol(lane);
          i32x2_t t[2];
#pragma unroll
          for (int j = 0; j < 2; ++j)
            t[j] = __builtin_bit_cast(i32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (LDS_AS i16x4_t*)(LDS_AS char*)(sb + ColTile<BN * 2, 2>::lds_offset(tr16_krow(lane, kk, j), n / 8) + (n % 8) * 2)));
          f.b[nb][0] = (i32x4_t){t[0].x, t[0].y, t[1].x, t[1].y};
        }
      }
    };
    // Eight waves: the products of the step in buffer `buf`.  Between them, in parts of five to seven instructions that
    // issue in the shadow of a product, the step that has arrived in registers is split and put into the
    // other buffer, and the loads of the step after it go out.
    f32x16_t small[MB][NB];  // sums of the five smaller products
    constexpr int kPairs[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};  // the smallest products first
    constexpr int KS16 = CFG::KE / 16, NMUL = KS16 * 6 * MB * NB, PARTS = 6 * (LA + LB);
    auto step = [&](int buf, auto fetch_tag) INLINED {
      const int to = (buf ^ 1) * CFG::SPLIT_BUF;
      Pieces f[KS16][3];
      u32x2_t w[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) load_pieces(f[0][i], buf, 0, i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < NMUL; ++m) {
        const int kk = m / (6 * MB * NB), t = m / (MB * NB) % 6, mb = m / NB % MB, nb = m % NB;
        f32x16_t& sum = t < 5 ? small[mb][nb] : acc[mb][nb];
        sum = mfma_block<IN_BF16, 1>(f[kk][kPairs[t][0]].a[mb], f[kk][kPairs[t][1]].b[nb], sum);
        if (kk + 1 < KS16 && m % (2 * MB * NB) == 0) load_pieces(f[kk + 1][t / 2], buf, kk + 1, t / 2);
#pragma unroll
        for (int j = 0; j <= PARTS / NMUL; ++j) {
          const int q = (m * PARTS + NMUL - 1) / NMUL + j;
          if (q * NMUL / PARTS != m || q >= PARTS) continue;
          const int i = q / 6, part = q % 6;
          split_part(raw[i], w, part);
          if (part & 1) put_plane(w, to + lds_at[i], i < LA ? CFG::A_PLANE : CFG::B_PLANE, part / 2);
          if (decltype(fetch_tag)::value && part == 5) raw[i] = load16_any(ptr[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    bool redo = false;
    point_at_a(std::true_type{});
    point_at_b(std::true_type{});
    clear_sums();
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) small[mb][nb] = acc[mb][nb];
    int s = 0;
    bool stop = false;
    // Eight waves: one barrier per step.  What a wave reads of the vote behind the barrier of step s, another one may
    // already be past: nobody writes ahead of the barrier of step s + 1 then (layout.h), `tiny` keeps the answer.
    bool tiny = false;  // an operand of the steps put down so far is below 2^-110
    auto close_step = [&]() INLINED {
      if (s + 1 < nsteps) tiny = low < kSmallest;  // (the last step puts down leftovers)
      if (tiny && vote_written_before_barrier(s)) *vote = 1;
      lds_barrier();
      stop = vote_read_behind_barrier(s) && *vote != 0;
      ++s;
    };
    fetch();
    if constexpr (CFG::NW == 8) {
#pragma unroll
      for (int i = 0; i < LA + LB; ++i) put_split(raw[i], lds_at[i], i < LA ? CFG::A_PLANE : CFG::B_PLANE);
      tiny = low < kSmallest;  // (with a single step the only look at it)
      if (nsteps > 1) fetch();
      lds_barrier();
      PHASE_STAMP(1);
      while (s < nsteps && !stop) {
        // Steps that fetch whole pieces have a loop of their own: where a general fetch can reach the next step's
        // splitting, the compiler waits there for every load at once.
        while (!stop && s + 2 < nsteps && plain()) {
          step(s & 1, std::true_type{});
          advance();
          close_step();
        }
        if (stop || s >= nsteps) break;
        step(s & 1, std::false_type{});  // (behind the last step the pieces in registers are put down again, where nobody reads them)
        if (s + 2 < nsteps) fetch();
        close_step();
      }
    } else {
      while (s < nsteps && !stop) {
        if (s > 0) lds_barrier();
#pragma unroll
        for (int i = 0; i < LA + LB; ++i) put_split(raw[i], lds_at[i], i < LA ? CFG::A_PLANE : CFG::B_PLANE);
        if (low < kSmallest) *vote = 1;
        if (s + 1 < nsteps) fetch();
        lds_barrier();
        if (s == 0) PHASE_STAMP(1);
        stop = vote_read_behind_barrier(s) && *vote != 0;  // (nobody writes before the barrier in front of the next step)
#pragma unroll
        for (int kk = 0; kk < KS16; ++kk) {
          Pieces f[3];
#pragma unroll
          for (int i = 0; i < 3; ++i) load_pieces(f[i], 0, kk, i);
#pragma unroll
          for (int t = 0; t < 6; ++t)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
              for (int nb = 0; nb < NB; ++nb) {
                f32x16_t& sum = t < 5 ? small[mb][nb] : acc[mb][nb];
                sum = mfma_block<IN_BF16, 1>(f[kPairs[t][0]].a[mb], f[kPairs[t][1]].b[nb], sum);
              }
        }
        ++s;
      }
      lds_barrier();
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][nb][i] += small[mb][nb][i];
    // The vote: sums of elements that exist, and what the splitting saw.
    bool finite = true;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const bool there = n0 + wn * CFG::TN + nb * 32 + acc_row(lane, i) < p.N;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) finite = finite && (!there || __builtin_fabsf(acc[mb][nb][i]) <= 3.402823466e38f);
      }
    if (!finite || tiny || p.K == 1) *vote = 1;
    lds_barrier();
    redo = *vote;
    if (redo) k_loop();
  }

  PHASE_STAMP(2);

  // ---- the tile in the output type, in LDS ------------------------------------------------------------------
  if constexpr (CFG::WK > 1) {
    // The waves along K leave their partial blocks behind the staged tile; wave 0 of each block adds them.
    char* const part = smem + CFG::TILE_BYTES + wk * (BM * CFG::PART_ROW);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x4_t v = {__float_as_uint(acc[mb][nb][4 * q]), __float_as_uint(acc[mb][nb][4 * q + 1]),
                             __float_as_uint(acc[mb][nb][4 * q + 2]), __float_as_uint(acc[mb][nb][4 * q + 3])};
          *(LDS_AS u32x4_t*)(LDS_AS char*)(part + (wm * CFG::TM + mb * 32 + acc_col(lane)) * CFG::PART_ROW +
                                           (wn * CFG::TN + nb * 32 + acc_row(lane, 4 * q)) * 4) = v;
        }
    lds_barrier();
  }
  auto stage4 = [&](int row, int col, const float (&sum)[4], float badd) INLINED {
    char* const dst = smem + row * CFG::TROW + col * Out::size;
    float h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = sum[e] * p.scale + badd;
    if constexpr (Out::size == 4) {
      *(LDS_AS u32x4_t*)(LDS_AS char*)dst = (u32x4_t){__float_as_uint(h[0]), __float_as_uint(h[1]), __float_as_uint(h[2]), __float_as_uint(h[3])};
    } else {
      using Out16 = typename std::conditional<Out::kFp32SumInReference, OutF16, OutBF16>::type;
      *(LDS_AS u32x2_t*)(LDS_AS char*)dst = (u32x2_t){Out16::pack(h[0], h[1]), Out16::pack(h[2], h[3])};
    }
  };
  auto bias_of = [&](int row) INLINED -> float {
    return p.bias && m0 + row < p.M ? load_scalar_as_float(p.bias, (long long)(m0 + row) * p.s_bias, p.bias_dtype) : 0.f;
  };
  if constexpr (CFG::WK > 1) {
    for (int q = tid; q < BM * BN / 4; q += NT) {
      const int row = q / (BN / 4), col = q % (BN / 4) * 4;
      float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < CFG::WK; ++w) {
        const u32x4_t v = *(const LDS_AS u32x4_t*)(LDS_AS char*)(smem + CFG::TILE_BYTES + (w * BM + row) * CFG::PART_ROW + col * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[e] += __uint_as_float(v[e]);
      }
      stage4(row, col, sum, bias_of(row));
    }
  } else {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int row = wm * CFG::TM + mb * 32 + acc_col(lane);
      const float badd = bias_of(row);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float sum[4] = {acc[mb][nb][4 * q], acc[mb][nb][4 * q + 1], acc[mb][nb][4 * q + 2], acc[mb][nb][4 * q + 3]};
          stage4(row, wn * CFG::TN + nb * 32 + acc_row(lane, 4 * q), sum, badd);
        }
    }
  }
  lds_barrier();

  PHASE_STAMP(3);

  const LinearTile<CFG::TROW> tile{smem};
  finish_any<Out, BM, BN, NT, CFG::NW == 8 ? 16 : 14, CFG::WK == 1>(p, tile, m0, n0, tid);
}

// ------------------------------------------------------------------------------------------------
// Launch
// ------------------------------------------------------------------------------------------------
template <class CFG>
int launch_any(FusedParams p, int device, int cu_count, hipStream_t stream, const char* types) {
  static std::atomic<bool> attr_set[64];  // see launch_mfma_grid
  if (device < 0 || device >= 64) return iris_host::fail("device index %d out of range", device);
  if (!attr_set[device].load(std::memory_order_acquire)) {
    hipError_t e = hipFuncSetAttribute((const void*)fused_any_kernel<CFG>, hipFuncAttributeMaxDynamicSharedMemorySize, CFG::SMEM_BYTES);
    if (e != hipSuccess) return (int)e;
    attr_set[device].store(true, std::memory_order_release);
  }
  p.tiles_m = cdiv(p.M, CFG::BM);
  p.tiles_n = cdiv(p.N, CFG::BN);
  const long long total = (long long)p.tiles_m * p.tiles_n;
  if (total > (1ll << 30)) return iris_host::fail("output of %d x %d has too many tiles", p.M, p.N);
  // (A launch that takes the place of one on packed operands comes with that one's order.)
  if (p.group_m == 0) p.group_m = any_group_m(p.tiles_m, p.tiles_n, p.num_xcd, cu_count / p.num_xcd * CFG::WG_PER_CU);
  const int grid = cdiv((int)total, p.num_xcd) * p.num_xcd;
  char name[96];
  snprintf(name, sizeof(name), "generic_%s_%dx%d_%s", types, CFG::BM, CFG::BN, CFG::BKC ? "nt" : "nn");
  iris_host::set_last_kernel(name);
  hipLaunchKernelGGL((fused_any_kernel<CFG>), dim3(grid), dim3(CFG::NT), CFG::SMEM_BYTES, stream, p);
  return (int)hipGetLastError();
}

// Tile choice: the tile with the least expected time, area x (tiles the busiest CU gets) / rate.  The rates (TFLOP/s, plain
// GEMM 4095x4095x4095 bf16 and 4096x4096x1536 float32, every CU busy) fall with the tile because LDS reads, operand
// bytes and splitting per flop rise; the 32x32 tile of float32 multiplies on the float32 MFMA.  A CU with a single
// workgroup of four waves has nothing to run while it waits (bf16 1024x4095x2049 on 256 tiles of 128x128: 40 us, where
// the full rate would give 26).  Checked against forced tiles, us for 256x256 / 128x128 / 64x128 / 64x64 / 32x32, the
// choice first (float32 without the largest): bf16 1999x2877x1371 64x128 41 (53 / 40 / - / 51 / 119), 1024x4095x2049 64x128 38 (68 / 40 /
// - / 48 / 105), one-shot with seven peers 500x2877x1371 64x64 30 (92 / 46 / 32 / - / 51), 33x2877x1371 32x32 13 (49 / 31 / 25 / 20 / -);
// float32 2048x2880x1024 64x128 98 (108 / - / 113 / 174), 2048x2048x4096 128x128 199 (- / 236 / 260 / 381), 512x2880x1024 64x64 40
// (47 / 45 / - / 44), 300x4096x4096 32x32 129 (159 / 153 / 138 / -), and, the one miss, 1536x2880x1024 64x64 87 (100 / 80 / - / 121).
// (e4m3 goes by the rates of bf16; they have not been measured for it.)
struct AnyTile {
  int bm, bn;
  float rate;
};
constexpr AnyTile kAnyTiles[] = {{256, 256, 855.f}, {128, 128, 654.f}, {64, 128, 508.f}, {64, 64, 395.f}, {32, 32, 195.f}};
constexpr AnyTile kAnyTilesF32[] = {{0, 0, 0.f}, {128, 128, 163.f}, {64, 128, 160.f}, {64, 64, 140.f}, {32, 32, 98.f}};  // the largest of eight waves

inline int choose_any_tile(int M, int N, int cu, bool f32_in, bool f32_out, float* expected = nullptr) {
  int best = 1;
  float best_time = 0.f;
  long long best_per_cu = 1;
  for (int i = f32_out ? 1 : 0; i < 5; ++i) {
    const AnyTile& t = f32_in ? kAnyTilesF32[i] : kAnyTiles[i];
    const long long per_cu = ((long long)cdiv(M, t.bm) * cdiv(N, t.bn) + cu - 1) / cu;
    const float alone = i == 0 || per_cu > 1 || (f32_in && i == 1) ? 1.f : f32_in ? 1.15f : 1.5f;
    const float time = (float)t.bm * t.bn * per_cu * alone / t.rate;
    if (best_time == 0.f || time < best_time) {
      best = i;
      best_time = time;
      best_per_cu = per_cu;
    }
  }
  // For a comparison with other kernels (times 2e-6 cu K: microseconds): of an odd number of 128x128 tiles, two to a CU, the last
  // one runs alone (bf16 8000x1501x1371, three per CU: 71.8 us).
  if (expected) *expected = best_time * (best == 1 && !f32_in && best_per_cu > 1 && best_per_cu % 2 ? (best_per_cu + 0.5f) / best_per_cu : 1.f);
  return best;
}

template <int IN, class Out, bool BKC>
int dispatch_any_layout(const FusedParams& p, int device, int cu, hipStream_t s, const char* types, int tile) {
  constexpr bool F32_IN = AnyIn<IN>::ES == 4, F32_OUT = Out::size == 4;
  switch (tile >= 0 ? tile : choose_any_tile(p.M, p.N, cu, F32_IN, F32_OUT)) {
    case 0:  // (a staged 256x256 tile of float32 would not fit the LDS)
      if constexpr (!F32_OUT) return launch_any<AnyCfg<IN, Out, 256, 256, 2, 4, 1, BKC>>(p, device, cu, s, types);
      break;
    case 2: return launch_any<AnyCfg<IN, Out, 64, 128, 2, 2, 1, BKC>>(p, device, cu, s, types);
    case 3: return launch_any<AnyCfg<IN, Out, 64, 64, 2, 2, 1, BKC>>(p, device, cu, s, types);
    case 4: return launch_any<AnyCfg<IN, Out, 32, 32, 1, 1, 4, BKC>>(p, device, cu, s, types);
  }
  return launch_any<AnyCfg<IN, Out, 128, 128, 2, F32_IN ? 4 : 2, 1, BKC>>(p, device, cu, s, types);
}

// The layout of B in LDS follows its unit stride: [k][n] when N is contiguous, else [n][k].  tile: index into kAnyTiles, or -1 for the choice.
template <int IN, class Out>
int dispatch_any(const FusedParams& p, int device, int cu, hipStream_t s, const char* types, int tile) {
  return p.s_bn == 1 ? dispatch_any_layout<IN, Out, false>(p, device, cu, s, types, tile)
                     : dispatch_any_layout<IN, Out, true>(p, device, cu, s, types, tile);
}
