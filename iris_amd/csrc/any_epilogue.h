// The end of a tile whose output rows may start and end anywhere: from the tile in the output type, staged in LDS, to
// aux, the flags, the slot sum and C.  fused_any_kernel always ends here, fused_mfma_kernel in its ANY_ROWS builds.
#pragma once

#include "fused_params.h"

// For the lambdas that the kernel is made of.  They keep their arrays in the kernel's registers only where they are inlined,
// which the compiler's cost limit did not allow where a piece has sixteen elements: e4m3 operands were worked on in
// scratch memory (1999x2877x1371 as a plain GEMM 200 -> 31 us, 4095x4095x2047 223 -> 75, 200x1001x3001 56 -> 12.5).  On the
// 256x256 tile (the 4095x4095x2047) 19 to 25 registers still do not fit and are spilled, 80 to 88 bytes a lane.
#define INLINED __attribute__((always_inline))

// Results: past the caches' keep policy when the rows are whole 16-byte pieces, through them otherwise, where the L2 puts
// the pieces of a line together first (bf16 4096x4095x352 27.3 -> 25.0 us; the aligned 4096x4096x352 23.5 against 24.5).
__device__ __forceinline__ void store16_result(char* p, u32x4_t v, bool aligned) {
  if (aligned) __builtin_nontemporal_store(v, (GLOBAL_AS u32x4_t*)(GLOBAL_AS char*)p);
  else *(GLOBAL_AS u32x4_any_t*)(GLOBAL_AS char*)p = v;
}

// One 16-byte piece of output elements as floats.
template <class Out>
struct OutPiece;
template <class Out16>
struct OutPiece16 {
  static __device__ __forceinline__ void unpack(u32x4_t v, float (&f)[8]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = Out16::to_float((unsigned short)(v[e] & 0xFFFF));
      f[2 * e + 1] = Out16::to_float((unsigned short)(v[e] >> 16));
    }
  }
  static __device__ __forceinline__ u32x4_t pack(const float (&f)[8]) {
    return (u32x4_t){Out16::pack(f[0], f[1]), Out16::pack(f[2], f[3]), Out16::pack(f[4], f[5]), Out16::pack(f[6], f[7])};
  }
};
template <> struct OutPiece<ElemBF16> : OutPiece16<OutBF16> {};
template <> struct OutPiece<ElemF16> : OutPiece16<OutF16> {};
template <>
struct OutPiece<ElemF32> {
  static __device__ __forceinline__ void unpack(u32x4_t v, float (&f)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = __uint_as_float(v[e]);
  }
  static __device__ __forceinline__ u32x4_t pack(const float (&f)[4]) {
    return (u32x4_t){__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
  }
};

// Element stores that are written through to memory at system scope (see store16_system).
template <class Out>
__device__ __forceinline__ void store_element_system(char* p, const char* from) {
  if constexpr (Out::size == 2)
    __hip_atomic_store((unsigned short*)p, *(const LDS_AS unsigned short*)(LDS_AS const char*)from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  else
    __hip_atomic_store((unsigned*)p, *(const LDS_AS unsigned*)(LDS_AS const char*)from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}


// A staged tile as this epilogue reads it: the address of an element, and 16 bytes from there on.
template <int TROW>
struct LinearTile {  // rows of TROW bytes
  char* base;
  __device__ __forceinline__ char* at(int row, int byte) const { return base + row * TROW + byte; }
  __device__ __forceinline__ u32x4_t piece(int row, int byte) const { return *(const LDS_AS u32x4_any_t*)(LDS_AS char*)at(row, byte); }
};

// IN_FLIGHT: 16-byte pieces of the peers per thread that are loaded together; with more, fewer workgroups share a CU.  LARGE: with
// both ways to read them (FusedParams::stream_peers), owned flag tiles as rectangles and the distances to the slots in registers.  The
// 32x32 tile, for small outputs, goes without: it starts anew for every launch, and more code took it 0.1 to 0.3 us of 6 to 10.
template <class Out, int BM, int BN, int NT, int IN_FLIGHT, bool LARGE, class Tile>
__device__ __forceinline__ void finish_any(const FusedParams& p, const Tile& tile, const int m0, const int n0, const int tid) {
#ifdef IRIS_HIP_PHASE_STAMPS
  constexpr int it = 0;  // PHASE_STAMP records the first tile of a workgroup; there is only one here
#endif
  constexpr int OE = kChunkBytes / Out::size;  // output elements per piece
  // ---- epilogue: pieces of OE consecutive columns, handed out row by row ---------------------------------------
  constexpr int PPR = BN / OE;             // pieces per tile row
  constexpr int RPP = NT / PPR;            // tile rows per pass of the workgroup
  constexpr int PASSES = BM > RPP ? BM / RPP : 1;
  static_assert(NT % PPR == 0 && (BM % RPP == 0 || BM < RPP), "epilogue pass shape");
  const int m_end = min(m0 + BM, p.M);  // one past the tile's last row (threads may have no row in a 32x32 tile)
  // A piece that would reach past the last column starts further left (both its threads then write the same
  // values twice), as long as the tile has that many columns.
  const int t_row = tid / PPR, tile_cols = min(BN, p.N - n0);
  int t_col = tid % PPR * OE;
  if (p.s_cn == 1 && t_col < tile_cols && t_col + OE > tile_cols && tile_cols >= OE) t_col = tile_cols - OE;
  const int gn = n0 + t_col;
  const int cols = min(p.N - gn, OE);           // columns of this thread's pieces that exist (may be <= 0)
  const bool whole = cols == OE && p.s_cn == 1;  // moved as 16 bytes, else element by element
  const int ftn = cdiv(p.N, p.flag_bn);
  const int ftotal = cdiv(p.M, p.flag_bm) * ftn;
  auto staged_piece = [&](int row, int col) INLINED { return tile.piece(row, col * Out::size); };
  auto staged_element = [&](int row, int col) INLINED -> float {
    if constexpr (Out::size == 4) {
      return *(const LDS_AS float*)(LDS_AS char*)tile.at(row, col * 4);
    } else {
      const unsigned short b = *(const LDS_AS unsigned short*)(LDS_AS char*)tile.at(row, col * 2);
      return Out::kFp32SumInReference ? f16_bits_to_float(b) : bf16_bits_to_float(b);
    }
  };
  auto offset = [&](int row, int col) INLINED {  // bytes into C (or aux) of an element of the tile
    return ((long long)(m0 + row + p.row_offset) * p.s_cm + (long long)(n0 + col) * p.s_cn) * Out::size;
  };
  auto owner_at = [&](int gm, int g) INLINED { return owner_of(p.epi, (gm / p.flag_bm) * ftn + g / p.flag_bn, ftotal, p.world, p.rank); };
  // Bytes from the own slot to the others, in scalar registers: read where they are used, behind stores that the compiler cannot
  // see into, every one of them is a load that the wave waits for (matmul_all_gather, bf16 1041x7521x65 of eight ranks 39.5 -> 35.2 us,
  // atomic 4000x2877x1371 386 -> 244).
  long long to_slot[kMaxCachedSlots] = {};
  if (LARGE && p.epi != EPI_STORE) {
    unsigned long long base[kMaxCachedSlots], own = 0;
    if (p.hb_in_args) {
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r) base[r] = (unsigned long long)p.hb_arg[r];
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r) own = r == p.rank ? base[r] : own;
    } else {
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r) base[r] = (unsigned long long)p.heap_bases[min(r, p.world - 1)];
      own = (unsigned long long)p.heap_bases[p.rank];
    }
#pragma unroll
    for (int r = 0; r < kMaxCachedSlots; ++r) to_slot[r] = (long long)uniform64(base[r] - own);
  }
  auto in_slot = [&](const char* at, int r) INLINED {  // r known when this is compiled, or beyond the cached slots
    return LARGE && r < kMaxCachedSlots ? (char*)at + to_slot[r] : slot_ptr(p.heap_bases, at, p.rank, r);
  };
  auto every_slot = [&](auto&& f) INLINED {
    if constexpr (LARGE) {
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r)
        if (r < p.world) f(r);
    }
    for (int r = LARGE ? kMaxCachedSlots : 0; r < p.world; ++r) f(r);
  };

  if (p.epi == EPI_ATOMIC) {
    if constexpr (Out::size == 4) {
      for (int d = tid; d < BM * BN; d += NT) {
        const int row = d / BN, col = d % BN;
        if (m0 + row >= p.M || n0 + col >= p.N) continue;
        const float v = *(const LDS_AS float*)(LDS_AS char*)tile.at(row, col * 4);
        const long long eoff = ((long long)(m0 + row) * p.s_cm + (long long)(n0 + col) * p.s_cn) * 4;
        every_slot([&](int pr) INLINED {
          if (p.clear_c && pr == p.rank) *(float*)(p.C + eoff) = 0.f + v;
          else atomicAdd((float*)(in_slot(p.C, pr) + eoff), v);
        });
      }
    } else if (p.s_cn == 1) {
      // Packed adds of aligned dwords, one per thread.  A row that starts in the middle of a dword is shifted by
      // one element against them; the half of a dword that is not this tile's gets -0 added, which leaves
      // every value of C as it is.  What lies next to C need not be a number (-0 makes a signalling NaN quiet): dwords
      // that reach past the first or the last column are for the element of C alone.
      using Out16 = typename std::conditional<Out::kFp32SumInReference, OutF16, OutBF16>::type;
      constexpr int DPR = BN / 2 + 1;
      for (int d = tid; d < BM * DPR; d += NT) {
        const int row = d / DPR;
        if (m0 + row >= p.M) continue;
        char* const at = p.C + ((long long)(m0 + row) * p.s_cm + n0) * 2;
        const int e = 2 * (d - row * DPR) - (int)(((unsigned long long)at >> 1) & 1);
        const bool lo = e >= 0 && e < BN && n0 + e < p.N, hi = e + 1 < BN && n0 + e + 1 < p.N;
        if (!lo && !hi) continue;
        const bool inside = n0 + e >= 0 && n0 + e + 1 < p.N;
        const unsigned w = (lo ? *(const LDS_AS unsigned short*)(LDS_AS char*)tile.at(row, e * 2) : 0x8000u) |
                           (hi ? (unsigned)*(const LDS_AS unsigned short*)(LDS_AS char*)tile.at(row, e * 2 + 2) : 0x8000u) << 16;
        every_slot([&](int pr) INLINED {
          if (p.clear_c && pr == p.rank) {
            const unsigned z = added_to_zero(w);
            if (lo) *(unsigned short*)(at + e * 2) = (unsigned short)z;
            if (hi) *(unsigned short*)(at + e * 2 + 2) = (unsigned short)(z >> 16);
          } else if (inside) {
            atomic_add_packed<Out16>(in_slot(at, pr) + e * 2, w);
          }
        });
      }
      // The elements of C in dwords that reach past it, a row and a rank per thread: each is a load and an exchange one behind
      // the other (fp16 3693x5963x258, eight ranks: 581 us with the ranks in turn above, 530 us).
      if (n0 == 0 || n0 + BN >= p.N) {
        for (int i = tid; i < BM * 2 * p.world; i += NT) {
          const int row = i % BM, last = i / BM & 1, pr = i / (2 * BM), e = last ? p.N - 1 - n0 : 0;
          if (m0 + row >= p.M || e >= BN || (n0 > 0 && !last) || (p.clear_c && pr == p.rank)) continue;
          char* const at = p.C + ((long long)(m0 + row) * p.s_cm + n0 + e) * 2;
          if ((int)(((unsigned long long)at >> 1) & 1) == last) continue;  // inside: not the high half, not the low half
          Out::atomic_add(slot_ptr(p.heap_bases, at, p.rank, pr),
                          Out16::to_float(*(const LDS_AS unsigned short*)(LDS_AS char*)tile.at(row, e * 2)));
        }
      }
    } else {
      for (int ps = 0; ps < PASSES; ++ps) {
        const int row = ps * RPP + t_row;
        if (m0 + row >= m_end) continue;
        for (int e = 0; e < cols; ++e)
          for (int pr = 0; pr < p.world; ++pr) {
            if (p.clear_c && pr == p.rank) Out::store(p.C + offset(row, t_col + e), 0.f + staged_element(row, t_col + e));
            else Out::atomic_add(slot_ptr(p.heap_bases, p.C, p.rank, pr) + offset(row, t_col + e), staged_element(row, t_col + e));
          }
      }
    }
    return;
  }

  const bool flags = epi_has_flags(p.epi);
  const bool solo = flags && (!p.sum_peers || p.world == 1);  // no peer contributes: the sum is the own tile
  // Stores of a result piece (or its elements) to wherever the operator wants it.
  auto each_destination = [&](int gm, int g, auto&& store) INLINED {
    if (p.epi == EPI_STORE) {
      store(p.C);
    } else if (p.epi == EPI_ALL_GATHER) {
      every_slot([&](int pr) INLINED { store(in_slot(p.C, pr)); });
    } else if (p.epi == EPI_ONE_SHOT) {
      store(p.C);
    } else {
      const int owner = owner_at(gm, g);
      if (!p.all_owners && owner != p.rank) return;
      if (p.epi == EPI_TWO_SHOT) {
        every_slot([&](int pr) INLINED { store(in_slot(p.C, pr)); });
      } else {
        store(slot_ptr(p.heap_bases, p.C, p.rank, p.all_owners ? owner : p.rank));
      }
    }
  };
  const bool aligned = (((unsigned long long)p.C | (unsigned long long)(p.s_cm * Out::size)) & 15) == 0 && p.N % OE == 0;
  const bool owners = flags && p.epi != EPI_ONE_SHOT;
  // A piece may be moved whole when all of it has one owner.
  const bool piece_ok = whole && (!owners || gn / p.flag_bn == (gn + OE - 1) / p.flag_bn);

  // Elements that no piece takes, in one place of the code.  Those of the last columns - fewer than a piece, or a piece that was moved to
  // the left over the edge of a flag tile - are dealt to all threads: with one thread per row the 7 columns that N = 3207
  // leaves for the last 128x128 tiles took longer than the rest of a bf16 product 691x3207x849, and the owners of the elements of the moved
  // pieces 30 to 40 us of a two-shot sum 1124x7618x1965.  Strided columns and flag tiles that are no whole pieces stay with the thread that has them.
  const int tail = p.s_cn != 1 ? 0 : tile_cols < OE ? tile_cols : owners && tile_cols % OE && p.flag_bn % OE == 0 && (n0 + tile_cols - OE) / p.flag_bn != (n0 + tile_cols - 1) / p.flag_bn ? OE : 0;
  auto each_element = [&](auto&& f) INLINED {
    if (!tail && (piece_ok || cols <= 0)) return;
    const int per_row = tail ? tail : cols, first = tail ? tile_cols - tail : t_col;
    const int row_step = tail ? NT / tail : 0, col_step = tail ? NT % tail : 1, next_row = tail ? 1 : RPP;
    int row = tail ? tid / tail : t_row, col = tail ? tid % tail : 0;
#pragma unroll 1
    while (row < m_end - m0) {
      f(row, first + col);
      row += row_step;
      col += col_step;
      if (col >= per_row) {
        col -= per_row;
        row += next_row;
      }
    }
  };
#pragma unroll 2
  for (int ps = 0; ps < PASSES; ++ps) {
    const int row = ps * RPP + t_row, gm = m0 + row;
    if (gm >= m_end) break;
    if (flags) {
      if (whole) store16_system_of_valu_data(p.aux + offset(row, t_col), staged_piece(row, t_col));
      if (p.clear_c && owners && piece_ok && owner_at(gm, gn) != p.rank)  // other ranks' tiles: zeros
        store16_result(p.C + offset(row, t_col), (u32x4_t){0u, 0u, 0u, 0u}, aligned);
      if (!solo) continue;
    }
    if (piece_ok) {
      const u32x4_t v = staged_piece(row, t_col);
      each_destination(gm, gn, [&](char* base) { store16_result(base + offset(row, t_col), v, aligned); });
    }
  }
  // A thread's own elements where little is to be done with them: all of a row at one time (two-shot of two ranks, bf16
  // 4000x2877x200, flag tiles of 70 columns, 88.9 -> 55.8 us).  64x64 and 32x32 tiles go without: launches of 10 us were 1 to 2 % slower for
  // the longer code.
  constexpr bool OWN_ROWS = LARGE && BM * BN > 64 * 64;
  auto my_elements = [&](auto&& f) INLINED {
    if (piece_ok || cols <= 0) return;
#pragma unroll 1
    for (int row = t_row; row < m_end - m0; row += RPP) {
#pragma unroll
      for (int e = 0; e < OE; ++e)
        if (e < cols) f(row, t_col + e);
    }
  };
  if (OWN_ROWS && !tail && p.epi == EPI_STORE) {
    my_elements([&](int row, int col) INLINED { Out::store(p.C + offset(row, col), staged_element(row, col)); });
  } else if (OWN_ROWS && !tail && flags && !solo) {
    if (p.s_cn != 1) my_elements([&](int row, int col) INLINED { store_element_system<Out>(p.aux + offset(row, col), tile.at(row, col * Out::size)); });
    if (p.clear_c && owners && !piece_ok && cols > 0) {
      const int split = (gn + cols - 1) / p.flag_bn * p.flag_bn - gn;  // columns left of the last flag tile
#pragma unroll 1
      for (int row = t_row; row < m_end - m0; row += RPP) {
        const int left = owner_at(m0 + row, gn), right = owner_at(m0 + row, gn + cols - 1);
        if (p.flag_bn >= OE) {
#pragma unroll
          for (int e = 0; e < OE; ++e)
            if (e < cols && (e < split ? left : right) != p.rank) Out::store(p.C + offset(row, t_col + e), 0.f);
        } else {
#pragma unroll 1
          for (int e = 0; e < cols; ++e)
            if (owner_at(m0 + row, gn + e) != p.rank) Out::store(p.C + offset(row, t_col + e), 0.f);
        }
      }
    }
  } else if (!flags || solo || (p.clear_c && owners) || tile_cols < OE || p.s_cn != 1) {  // (else there is nothing to do for them)
    each_element([&](int row, int col) INLINED {
      const int gm = m0 + row, g = n0 + col;
      if (flags) {
        if (tile_cols < OE || p.s_cn != 1) store_element_system<Out>(p.aux + offset(row, col), tile.at(row, col * Out::size));
        if (p.clear_c && owners && owner_at(gm, g) != p.rank) Out::store(p.C + offset(row, col), 0.f);
        if (!solo) return;
      }
      each_destination(gm, g, [&](char* base) { Out::store(base + offset(row, col), staged_element(row, col)); });
    });
  }
  PHASE_STAMP(4);
  if (!flags) return;

  // Publish and wait, as in the tiled kernel: aux is written through, so relaxed flag stores behind the
  // acknowledgement are enough.
  const bool up_already = solo ? true : probe_peer_flags<BM, BN, NT>(p, m0, n0, tid);
  wait_vmcnt<0>();
  __syncthreads();
  PHASE_STAMP(5);
  raise_flags<BM, BN, NT, true>(p, m0, n0, tid);
  if (solo) return;
  if (!up_already) wait_peer_flags<BM, BN, NT>(p, m0, n0, tid);
  __syncthreads();
  PHASE_STAMP(6);

  // Slot sum in ascending rank order from the own (already rounded) value, in fp32 or by the reference's rule.
  const bool ref_chain = (p.acc_mode == IRIS_HIP_ACC_REFERENCE) && !Out::kFp32SumInReference;
  auto add = [&](float sum, float x) INLINED {
    sum += x;
    return ref_chain ? Out::round(sum) : sum;
  };
  // Both ways to read the peers' tiles differ in nothing but the loads.  (32x32 tiles are for outputs of at most 5.2 MB, of which
  // seven peers' are 37 MB: the line of peers_past_caches, and one way is enough.)
  const bool stream = LARGE && p.stream_peers;
  // The pieces of the tile are handed out row by row (RECT false: each thread keeps its column, what another rank reduces is
  // left out), or those of one rectangle of it, rows [r0, r1) and columns [c0, c1) of the tile, all with one owner (RECT true).
  auto reduce = [&](auto np_tag, auto rect_tag, int r0, int r1, int c0, int c1) INLINED {
    constexpr int NP = decltype(np_tag)::value;  // peers, all of whose loads go out together; 0: any number
    constexpr bool RECT = decltype(rect_tag)::value;
    constexpr int NPV = NP > 0 ? NP : 1;
    // Passes whose loads are in flight together: as many as the registers hold (the sums are staged and their
    // accumulators free), every group of passes is a round trip to memory.
    constexpr int G = PASSES % 8 == 0 && 8 * NPV <= IN_FLIGHT ? 8 : PASSES % 4 == 0 && 4 * NPV <= IN_FLIGHT ? 4 : PASSES % 2 == 0 ? 2 : 1;
    const int per_row = RECT ? cdiv(c1 - c0, OE) : PPR;
    const int passes = RECT ? cdiv((r1 - r0) * per_row, NT) : PASSES;
    for (int pg = 0; pg < passes; pg += G) {
      if (!RECT && m0 + pg * RPP >= p.M) break;
      bool act[G];
      int row[G], col[G];
      u32x4_t pv[G][NPV];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if constexpr (RECT) {
          const unsigned i = (unsigned)((pg + g) * NT + tid), r = i / (unsigned)per_row;
          row[g] = r0 + (int)r;
          col[g] = rect_piece_col(c0, c1, (int)(i - r * per_row), OE);
          act[g] = row[g] < r1;
        } else {
          row[g] = (pg + g) * RPP + t_row;
          col[g] = t_col;
          act[g] = m0 + row[g] < m_end && piece_ok;
          if (act[g] && owners && !p.all_owners) act[g] = owner_at(m0 + row[g], gn) == p.rank;
        }
        if constexpr (NP > 0) {
          if (act[g]) {
            auto at = [&](int i) INLINED {
              return (LARGE ? p.aux + (i < p.rank ? to_slot[i] : to_slot[i + 1]) : slot_ptr(p.heap_bases, p.aux, p.rank, i < p.rank ? i : i + 1)) + offset(row[g], col[g]);
            };
            if (stream) {
              KEEP_BRANCHES_APART();
#pragma unroll
              for (int i = 0; i < NP; ++i) pv[g][i] = load16_any_nt(at(i));
              KEEP_BRANCHES_APART();
            } else {
#pragma unroll
              for (int i = 0; i < NP; ++i) pv[g][i] = load16_any(at(i));
            }
          }
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (!act[g]) continue;
        const int gm = m0 + row[g];
        float sum[OE], x[OE];
        OutPiece<Out>::unpack(staged_piece(row[g], col[g]), sum);
        if constexpr (NP > 0) {
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            OutPiece<Out>::unpack(pv[g][i], x);
#pragma unroll
            for (int e = 0; e < OE; ++e) sum[e] = add(sum[e], x[e]);
          }
        } else {
          for (int pr = 0; pr < p.world; ++pr) {
            if (pr == p.rank) continue;
            const char* const at = slot_ptr(p.heap_bases, p.aux, p.rank, pr) + offset(row[g], col[g]);
            u32x4_t v;
            if (p.stream_peers) {
              KEEP_BRANCHES_APART();
              v = load16_any_nt(at);
              KEEP_BRANCHES_APART();
            } else {
              v = load16_any(at);
            }
            OutPiece<Out>::unpack(v, x);
#pragma unroll
            for (int e = 0; e < OE; ++e) sum[e] = add(sum[e], x[e]);
          }
        }
        const u32x4_t v = OutPiece<Out>::pack(sum);
        each_destination(gm, n0 + col[g], [&](char* base) { store16_result(base + offset(row[g], col[g]), v, RECT ? rect_pieces_aligned(aligned, p.flag_bn, OE) : aligned); });
      }
    }
  };
  // Fewer columns than a piece, strided columns or several owners: all elements of a peer in one go.
  auto reduce_elements = [&](int row) INLINED {
    float sum[OE];
#pragma unroll
    for (int e = 0; e < OE; ++e) sum[e] = e < cols ? staged_element(row, t_col + e) : 0.f;
    for (int pr = 0; pr < p.world; ++pr) {
      if (pr == p.rank) continue;
      const char* const src = slot_ptr(p.heap_bases, p.aux, p.rank, pr);
      float x[OE];
#pragma unroll
      for (int e = 0; e < OE; ++e) x[e] = e < cols ? Out::load(src + offset(row, t_col + e)) : 0.f;
#pragma unroll
      for (int e = 0; e < OE; ++e) sum[e] = add(sum[e], x[e]);
    }
#pragma unroll
    for (int e = 0; e < OE; ++e)
      if (e < cols) each_destination(m0 + row, gn + e, [&](char* base) { Out::store(base + offset(row, t_col + e), sum[e]); });
  };
  // What a flag tile has in this tile, or the tile itself, when that is narrower than a piece: an element per thread, all peers of it in one go.
  auto reduce_sliver = [&](int r0, int r1, int c0, int c1) INLINED {
    const int wide = c1 - c0;
#pragma unroll 1
    for (int i = tid; i < (r1 - r0) * wide; i += NT) {
      const int row = r0 + i / wide, col = c0 + i % wide;
      if (owners && !p.all_owners && owner_at(m0 + row, n0 + col) != p.rank) continue;
      const char* const own = p.aux + offset(row, col);
      float sum = staged_element(row, col), x[kMaxCachedSlots];
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r)  // (slots that there are not: the own one)
        x[r] = Out::load(LARGE ? own + (r < p.world ? to_slot[r] : 0) : slot_ptr(p.heap_bases, own, p.rank, r < p.world ? r : p.rank));
#pragma unroll
      for (int r = 0; r < kMaxCachedSlots; ++r)
        if (r < p.world && r != p.rank) sum = add(sum, x[r]);
      for (int r = kMaxCachedSlots; r < p.world; ++r)
        if (r != p.rank) sum = add(sum, Out::load(slot_ptr(p.heap_bases, own, p.rank, r)));
      each_destination(m0 + row, n0 + col, [&](char* base) { Out::store(base + offset(row, col), sum); });
    }
  };
  // Variants with owners: a thread that keeps its column has nothing to do in most rows, so flag tiles that keep half of the
  // threads busy are streamed one after the other by all of them (two-shot, eight ranks, bf16 1999x2877x1371 59.8 -> 50.7 us,
  // 4000x2877x2501 160 -> 143; float32 2048x2880x1024 of four ranks 102.8 -> 100.5).
  const bool by_rect = LARGE && owners && p.s_cn == 1 && p.flag_bn >= OE && (long long)min(p.flag_bm, BM) * (min(p.flag_bn, BN) / OE) * 2 >= NT;
  auto each_owned = [&](auto&& f) INLINED {
    const int n1 = min(n0 + BN, p.N);
    for (int fr = m0 / p.flag_bm; fr * p.flag_bm < m_end; ++fr)
      for (int fc = n0 / p.flag_bn; fc * p.flag_bn < n1; ++fc) {
        if (!p.all_owners && owner_of(p.epi, fr * ftn + fc, ftotal, p.world, p.rank) != p.rank) continue;
        f(max(m0, fr * p.flag_bm) - m0, min(m_end, (fr + 1) * p.flag_bm) - m0, max(n0, fc * p.flag_bn) - n0, min(n1, (fc + 1) * p.flag_bn) - n0);
      }
  };
  auto reduce_pieces = [&](auto np_tag) INLINED {
    if (!by_rect) {
      reduce(np_tag, std::false_type{}, 0, 0, 0, 0);
    } else {
      if constexpr (LARGE)
        each_owned([&](int r0, int r1, int c0, int c1) INLINED {
          if (c1 - c0 >= OE) reduce(np_tag, std::true_type{}, r0, r1, c0, c1);
        });
    }
  };
  if (tile_cols < OE && p.s_cn == 1) {
    reduce_sliver(0, m_end - m0, 0, tile_cols);
    return;
  }
  if (by_rect) {
    // Only the first and the last flag tile of a row can be that narrow here.
    const int first = p.flag_bn - n0 % p.flag_bn, last = (n0 + tile_cols - 1) % p.flag_bn + 1;
    if (LARGE && min(first, last) < OE)
      each_owned([&](int r0, int r1, int c0, int c1) INLINED {
        if (c1 - c0 < OE) reduce_sliver(r0, r1, c0, c1);
      });
  } else if (tail) {
    reduce_sliver(0, m_end - m0, tile_cols - tail, tile_cols);
  } else if (!piece_ok && cols > 0) {
#pragma unroll 1
    for (int row = t_row; row < m_end - m0; row += RPP) reduce_elements(row);
  }
  switch (p.world - 1) {
    case 1: reduce_pieces(std::integral_constant<int, 1>{}); break;
    case 3: reduce_pieces(std::integral_constant<int, 3>{}); break;
    case 7: reduce_pieces(std::integral_constant<int, 7>{}); break;
    default: reduce_pieces(std::integral_constant<int, 0>{}); break;
  }
  PHASE_STAMP(7);
}
