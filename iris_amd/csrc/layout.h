// Index math shared by the gfx950 GEMM kernels and the host-side layout simulator.
//
// Everything here is a pure function of small integers, usable from host and device code.
// The kernels move operand tiles from HBM into LDS with 16-byte direct-to-LDS buffer loads
// (one wave instruction deposits 64 lanes x 16 B = 1 KiB of contiguous LDS), read the
// K-contiguous operand with 16-byte LDS reads and the N-contiguous operand with the gfx950
// LDS transpose reads, and feed 32x32 or 16x16 MFMA blocks.  The functions below say, for every lane,
// which global 16-byte chunk it fetches, where that chunk lives in LDS, and which LDS address
// a lane presents when it assembles an MFMA operand.
//
// Conventions
//   ES     element size in bytes (2 for bf16/fp16, 1 for fp8)
//   chunk  16 bytes = CE elements (8 or 16)
//   "row tile"   an operand tile stored as [rows][BK elements], K contiguous  (A, or B given as B^T)
//   "col tile"   an operand tile stored as [BK rows (k)][BN elements], N contiguous (row-major B)
#pragma once

#if defined(__HIPCC__)
#define IRIS_HD __host__ __device__ __forceinline__
#else
#define IRIS_HD inline
#endif

namespace iris_layout {

constexpr int kChunkBytes = 16;
constexpr int kWave = 64;
constexpr int kDmaBytes = kWave * kChunkBytes;  // LDS bytes written by one wave-level load

// ---------------------------------------------------------------------------------------------
// Row tile: [rows][RB bytes], RB = BK*ES in {64, 128}.  16-byte chunks are XOR-swizzled so that
// 16 lanes reading the same logical chunk of 16 consecutive rows touch 16 distinct 16-byte
// bank groups (one full sweep of the 64 four-byte banks).
// ---------------------------------------------------------------------------------------------
template <int RB>
struct RowTile {
  static_assert(RB == 64 || RB == 128 || RB == 256, "row bytes must be 64, 128 or 256");
  static constexpr int kChunksPerRow = RB / kChunkBytes;
  static constexpr int kRowsPer256 = (256 / RB) > 0 ? (256 / RB) : 1;

  IRIS_HD static int swizzle(int row) { return (row / kRowsPer256) % kChunksPerRow; }
  // LDS byte offset of logical chunk c of a row.
  IRIS_HD static int lds_offset(int row, int c) { return row * RB + ((c ^ swizzle(row)) * kChunkBytes); }
  // Inverse used by the loader: LDS byte offset (multiple of 16) -> (row, logical chunk).
  IRIS_HD static void from_lds(int off, int& row, int& c) {
    row = off / RB;
    c = ((off % RB) / kChunkBytes) ^ swizzle(row);
  }
};

// ---------------------------------------------------------------------------------------------
// Col tile: [BK rows][RB bytes], RB = BN*ES >= 256 (16-bit) or >= 128 (8-bit).  LDS serves a
// transpose read one half-wave (32 lanes x 8 bytes = 256 bytes = all 64 banks) at a time.  A half-wave
// touches 4 k-rows x 64 contiguous bytes (16-bit) or 8 k-rows x 32 bytes (8-bit); the other half-wave
// reads the same columns 8 (32) k-rows further down.  XOR-ing the index of that 64- (32-) byte block
// with the k-row puts the rows of a half-wave on distinct blocks of a 256-byte bank line.  When a
// 256-byte bank line holds two tile rows (RB = 128) the row parity already separates them and the
// XOR uses k-row / 2.  (Rotating 32-byte blocks by k-row % 8 for 16-bit data, as an earlier layout
// did, is conflict-free per 16 lanes but lets rows 2i and 2i+1 of a half-wave share a block: the
// hardware counted bank conflicts on half of the cycles of these reads.)
// ---------------------------------------------------------------------------------------------
template <int RB, int ES>
struct ColTile {
  static_assert(ES == 1 || ES == 2, "element size must be 1 or 2 bytes");
  static constexpr int kChunksPerRow = RB / kChunkBytes;
  static constexpr int kBlockChunks = (ES == 2) ? 4 : 2;        // 16-byte chunks per swizzled block
  static constexpr int kRowsPerLine = RB >= 256 ? 1 : 256 / RB;  // tile rows per 256-byte bank line
  static constexpr int kSwRows = ((ES == 2) ? 4 : 8) / kRowsPerLine;
  static_assert(kChunksPerRow >= kSwRows * kBlockChunks, "tile row too short for the swizzle");

  IRIS_HD static int swizzle(int krow) { return ((krow / kRowsPerLine) % kSwRows) * kBlockChunks; }
  IRIS_HD static int lds_offset(int krow, int c) { return krow * RB + ((c ^ swizzle(krow)) * kChunkBytes); }
  IRIS_HD static void from_lds(int off, int& krow, int& c) {
    krow = off / RB;
    c = ((off % RB) / kChunkBytes) ^ swizzle(krow);
  }
};

// ---------------------------------------------------------------------------------------------
// MFMA 32x32 operand lanes.  For v_mfma_f32_32x32x16_{bf16,f16} lane l supplies, for row (or
// column) l%32, the 8 k-values 8*(l/32)..+7 of the 16-wide k-slice; for the 8-bit 32x32x64 form
// it supplies the 32 k-values 32*(l/32)..+31.  Only the pairing of A and B k-slots matters for
// the product, so both operands simply use the same rule.
// ---------------------------------------------------------------------------------------------

// 16-bit, K-contiguous operand: one 16-byte read per 32x32x16 MFMA.
//   row  = block_row0 + lane%32 ; chunk = kk*2 + lane/32        (kk = k-slice of 16 within the tile)
IRIS_HD int frag16_row(int lane) { return lane % 32; }
IRIS_HD int frag16_chunk(int lane, int kk) { return kk * 2 + lane / 32; }

// 8-bit, K-contiguous operand: two 16-byte reads per 32x32x64 MFMA (h = 0,1).
IRIS_HD int frag8_chunk(int lane, int kk, int h) { return kk * 4 + 2 * (lane / 32) + h; }

// LDS transpose read, 16-bit (ds_read_b64_tr_b16).  Within each 16-lane group, lane p presents
// the address of 4 consecutive n at k-row p/4, n = 4*(p%4); it receives, for n = p, the 4 k-rows.
// For read j (0,1) of the k-slice kk, lane l of the wave addresses:
IRIS_HD int tr16_krow(int lane, int kk, int j) {
  int g = lane / 16, p = lane % 16;
  return kk * 16 + 8 * (g / 2) + 4 * j + p / 4;
}
IRIS_HD int tr16_ncol(int lane) {  // first of 4 consecutive n, relative to the 32-wide block
  int g = lane / 16, p = lane % 16;
  return 16 * (g % 2) + 4 * (p % 4);
}

// LDS transpose read, 8-bit (ds_read_b64_tr_b8).  Lane p of a 16-lane group presents 8
// consecutive n at k-row p/2, n = 8*(p%2); it receives, for n = p, the 8 k-rows.
// For read r (0..3) of the 64-wide k-slice kk:
IRIS_HD int tr8_krow(int lane, int kk, int r) {
  int g = lane / 16, p = lane % 16;
  return kk * 64 + 32 * (g / 2) + 8 * r + p / 2;
}
IRIS_HD int tr8_ncol(int lane) {
  int g = lane / 16, p = lane % 16;
  return 16 * (g % 2) + 8 * (p % 2);
}

// ---------------------------------------------------------------------------------------------
// MFMA 16x16 operand lanes, 16-bit (v_mfma_f32_16x16x32_{bf16,f16}): lane l supplies, for row (or column)
// l%16, the 8 k-values 8*(l/16)..+7 of the 32-wide k-slice.
// ---------------------------------------------------------------------------------------------
IRIS_HD int mma16_row(int lane) { return lane % 16; }
IRIS_HD int mma16_chunk(int lane, int kk) { return kk * 4 + lane / 16; }

// The row tile those reads want.  LDS serves a 16-byte read 16 lanes at a time, and not 16 in a row: lanes {0-3, 12-15,
// 20-27}, then {4-11, 16-19, 28-31}, then the same of the upper half-wave (measured with address patterns of an MI355X:
// 4.2 cycles per read and CU where these meet on 16 distinct chunks of a 256-byte bank line, 8 with RowTile<64>, whose
// rows 0-3 of one chunk and 4-7 of the next share theirs).
template <int RB>
struct RowTile16 : RowTile<RB> {};
template <>
struct RowTile16<64> {
  static constexpr int kChunksPerRow = 4;
  IRIS_HD static int swizzle(int row) { return (row >> 1) & 2; }
  IRIS_HD static int lds_offset(int row, int c) { return row * 64 + ((c ^ swizzle(row)) * kChunkBytes); }
  IRIS_HD static void from_lds(int off, int& row, int& c) {
    row = off / 64;
    c = ((off % 64) / kChunkBytes) ^ swizzle(row);
  }
};

// Transpose read j (0,1) of k-slice kk of a 16-wide column block: as tr16_* above, but the 16-lane groups of a
// wave all take the same 16 columns, 8 k-rows apart.
IRIS_HD int mma16_tr_krow(int lane, int kk, int j) { return kk * 32 + 8 * (lane / 16) + 4 * j + lane % 16 / 4; }
IRIS_HD int mma16_tr_ncol(int lane) { return 4 * (lane % 4); }

// The column tile those reads want: a half-wave touches k-rows {0..3, 8..11} (plus a multiple of 4) x 32 contiguous
// bytes, so 32-byte blocks are XORed with the k-row's bits 0, 1 and 3: eight blocks, one 256-byte bank line.  With two
// tile rows to a bank line (RB = 128) the row parity already separates rows, and bits 1 and 3 are left.
template <int RB>
struct ColTile16 {
  static constexpr int kChunksPerRow = RB / kChunkBytes;
  static_assert(RB == 128 || RB >= 256, "tile row too short for the swizzle");
  IRIS_HD static int swizzle(int krow) {
    return RB >= 256 ? 2 * ((krow & 3) | ((krow >> 1) & 4)) : 2 * (((krow >> 1) & 1) | ((krow >> 2) & 2));
  }
  IRIS_HD static int lds_offset(int krow, int c) { return krow * RB + ((c ^ swizzle(krow)) * kChunkBytes); }
  IRIS_HD static void from_lds(int off, int& krow, int& c) {
    krow = off / RB;
    c = ((off % RB) / kChunkBytes) ^ swizzle(krow);
  }
};

// Accumulator of D = X * Y for the 16x16 MFMA: register i (0..3) of lane l holds D[4*(l/16) + i][l%16].
IRIS_HD int mma16_acc_row(int lane, int i) { return 4 * (lane / 16) + i; }
IRIS_HD int mma16_acc_col(int lane) { return lane % 16; }

// Block i of a k-slice's products over MB x NB blocks: quadrant by quadrant (upper left, upper right, lower right, lower
// left), row by row inside one, every other row backwards, so that consecutive products mostly share an operand (less
// switching, a few percent of the power) and the first quadrant needs only half of the fragments.
template <int MB, int NB>
IRIS_HD constexpr void quad_block(int i, int& mb, int& nb) {
  constexpr int QM = MB / 2, QN = NB / 2, Q = QM * QN;
  const int q = i / Q, r = i % Q, row = r / QN, col = r % QN;
  mb = (q >= 2 ? QM : 0) + row;
  nb = (q == 1 || q == 2 ? QN : 0) + ((row & 1) ? QN - 1 - col : col);
}

// Accumulator of D = X * Y for the 32x32 MFMA: register i (0..15) of lane l holds
//   D[row = 8*(i/4) + 4*(l/32) + i%4][col = l%32].
// The kernels issue mfma(Bfrag, Afrag) so that D rows run along n and columns along m: every
// lane then owns 4 consecutive n for one m, which packs into one 8-byte LDS write.
IRIS_HD int acc_row(int lane, int i) { return 8 * (i / 4) + 4 * (lane / 32) + (i % 4); }
IRIS_HD int acc_col(int lane) { return lane % 32; }

// ---------------------------------------------------------------------------------------------
// Tile order.  Workgroup b of a launch lands on XCD b % num_xcd (round-robin dispatch).  Tiles
// are first put in a grouped order (group_m tile-rows at a time, walking down the group's
// column before moving right) and each XCD is handed one contiguous span of that order, so the
// tiles that share A row-panels and B column-panels meet in the same L2.
// ---------------------------------------------------------------------------------------------
IRIS_HD void grouped_tile(int idx, int tiles_m, int tiles_n, int group_m, int& tm, int& tn) {
  int per_group = group_m * tiles_n;
  int g = idx / per_group;
  int first_m = g * group_m;
  int rows = tiles_m - first_m < group_m ? tiles_m - first_m : group_m;
  int r = idx - g * per_group;
  tm = first_m + r % rows;
  tn = r / rows;
}

// Position in the grouped order of the it-th tile processed by workgroup `wg` of `nwg`.
// Returns -1 when that workgroup has no it-th tile.
IRIS_HD int xcd_tile_index(int wg, int nwg, int it, int total, int num_xcd) {
  if (nwg % num_xcd != 0 || nwg < num_xcd) {  // plain round-robin
    long idx = (long)wg + (long)it * nwg;
    return idx < total ? (int)idx : -1;
  }
  int xcd = wg % num_xcd;
  int local = wg / num_xcd;
  int wg_per_xcd = nwg / num_xcd;
  int span = (total + num_xcd - 1) / num_xcd;
  long in_span = (long)local + (long)it * wg_per_xcd;
  if (in_span >= span) return -1;
  long idx = (long)xcd * span + in_span;
  return idx < total ? (int)idx : -1;
}

// ---------------------------------------------------------------------------------------------
// Flag tiles (the reference's BLOCK_SIZE_M x BLOCK_SIZE_N tiles) and their owners.
// ---------------------------------------------------------------------------------------------
IRIS_HD int cdiv(int a, int b) { return (a + b - 1) / b; }

// Owner of flag tile t under interleaved (two-shot all-reduce) distribution.
IRIS_HD int owner_interleaved(int t, int world) { return t % world; }

// Owner of flag tile t under contiguous (reduce-scatter) distribution: each rank takes
// total/world tiles, the last rank also the remainder.
IRIS_HD int owner_contiguous(int t, int total, int world) {
  int per = total / world;
  if (per == 0) return world - 1;
  int o = t / per;
  return o < world - 1 ? o : world - 1;
}

// A flag tile's columns [c0, c1) of a tile in pieces of `oe` elements, the last one from as far left as it takes: the column of
// piece i, and whether all such pieces of a launch start on 16-byte boundaries when its rows do (tiles always do, flag tiles
// start at multiples of flag_bn).
IRIS_HD int rect_piece_col(int c0, int c1, int i, int oe) { return c0 + i * oe < c1 - oe ? c0 + i * oe : c1 - oe; }
IRIS_HD bool rect_pieces_aligned(bool rows_aligned, int flag_bn, int oe) { return rows_aligned && flag_bn % oe == 0; }

// How many kernel macro-tiles (KM x KN) overlap flag tile (fm, fn) of size (FM x FN) in an
// M x N matrix.  A flag is raised by the last of them to finish.
IRIS_HD int macro_tiles_over_flag_tile(int fm, int fn, int FM, int FN, int KM, int KN, int M, int N) {
  int r0 = fm * FM, r1 = (fm + 1) * FM < M ? (fm + 1) * FM : M;
  int c0 = fn * FN, c1 = (fn + 1) * FN < N ? (fn + 1) * FN : N;
  int nm = (r1 - 1) / KM - r0 / KM + 1;
  int nn = (c1 - 1) / KN - c0 / KN + 1;
  return nm * nn;
}

// ---------------------------------------------------------------------------------------------
// Order of a launch's tiles, and what it has to guarantee.
//
// Epilogues with flags publish their tile and then wait in place for the peers' flags: a waiting workgroup keeps its CU.  A
// launch with more tiles than workgroups that run at one time therefore needs an order that lets the ranks finish together.
//   - The same order on every rank does: the first unfinished tile of that order is running, and published, on all of them.
//   - A rank whose waiting workgroups leave others room to run (publishes_alone) publishes everything whatever the
//     others do.  It may take any order, and no order of its own can hold up anybody else.
// What only one rank knows - whether it got memory, whether its stream is captured - may choose the kernel of such a rank, and for
// the others only between kernels that take the same tiles in the same order (run_packed in iris_hip.hip).
// tests/host_sim/layout_sim.cpp replays the launches of all ranks, with what fits at one time, until they end.
// ---------------------------------------------------------------------------------------------
enum { EPI_STORE = 0, EPI_ONE_SHOT = 1, EPI_TWO_SHOT = 2, EPI_REDUCE_SCATTER = 3, EPI_ALL_GATHER = 4, EPI_ATOMIC = 5 };

// Epilogues that publish aux + flags and then reduce over the slots.
IRIS_HD bool epi_has_flags(int epi) { return epi == EPI_ONE_SHOT || epi == EPI_TWO_SHOT || epi == EPI_REDUCE_SCATTER; }

struct TileLaunch {
  int M, N, tile_m, tile_n;
  int num_xcd;
  int resident;    // workgroups that run at one time on an XCD
  int two_per_cu;  // ... two of them on a CU
  int epi, world, rank;
  int sum_peers;   // 0: the peers' tiles are neither waited for nor read
  int all_owners;  // reduce-scatter: this rank sums the tiles of every owner
  int flag_bm, flag_bn;
};

struct TileOrder {
  int tiles_m, tiles_n;
  int group_m, group_m_spans;  // group height; the one to use if the launch falls back to spans (split tiles)
  int interleave, tile_rotate;  // see FusedParams
};

// This rank's band of a reduce-scatter as rows [first, last] of kernel tiles; false when it owns no flag tile.
IRIS_HD bool band_tile_rows(const TileLaunch& t, int& first, int& last) {
  const int ftn = cdiv(t.N, t.flag_bn), ftotal = cdiv(t.M, t.flag_bm) * ftn, per = ftotal / t.world;
  const int lo = t.rank * per, hi = t.rank == t.world - 1 ? ftotal : lo + per;
  if (lo >= hi) return false;
  const long end = (long)((hi - 1) / ftn + 1) * t.flag_bm;
  first = (int)((long)(lo / ftn) * t.flag_bm / t.tile_m);
  last = (int)(((end < t.M ? end : t.M) - 1) / t.tile_m);
  return true;
}

// Whether the workgroups of a launch on this rank that wait for peers leave room for the others to run and publish.  The order
// is the one of tile_order with a reduce-scatter's tiles dealt out, in groups of `group_m` rows.
IRIS_HD bool publishes_alone(const TileLaunch& t, int group_m) {
  if (!epi_has_flags(t.epi) || !t.sum_peers || t.world == 1) return true;
  const int tiles_m = cdiv(t.M, t.tile_m), tiles_n = cdiv(t.N, t.tile_n);
  if (cdiv(tiles_m * tiles_n, t.num_xcd) <= t.resident) return true;
  if (t.epi != EPI_REDUCE_SCATTER || t.all_owners) return false;
  int first, last;
  if (!band_tile_rows(t, first, last)) return true;
  // The groups that hold the band (its tiles may be every second one of a group's), at most five eighths of what runs at one time:
  // CUs may be busy with other launches.  (At a half the last of four ranks no longer starts with its band of 140 tiles: bf16
  // 3128x7162x1270, 256 CUs, 112 -> 143 us.)
  first = first / group_m * group_m;
  last = last / group_m * group_m + group_m - 1;
  if (last >= tiles_m) last = tiles_m - 1;
  return cdiv((last - first + 1) * tiles_n, t.num_xcd) * 8 <= t.resident * 5;
}

IRIS_HD TileOrder tile_order(const TileLaunch& t) {
  TileOrder o;
  o.tiles_m = cdiv(t.M, t.tile_m);
  o.tiles_n = cdiv(t.N, t.tile_n);
  // Group height: tile-rows walked together so that the tiles an XCD works on at one time - its whole
  // span, or one round of it when the span is longer than its resident workgroups - are close to a
  // square (fewest operand panels per L2).
  const int span = cdiv(o.tiles_m * o.tiles_n, t.num_xcd);
  const bool rounds = span > t.resident, peers = t.sum_peers && t.world > 1;
  const int at_once = rounds ? t.resident : span;
  int g = 1;
  while (g * g * 2 <= at_once && g * 2 <= o.tiles_m) g *= 2;
  // Two-shot launches of several rounds (one workgroup per tile, handed out in this order) do better with
  // groups of at most four rows (eight ranks, fp16: 16384x3584x8192 1006 -> 977 us, 8192x8192x2752 441 -> 428).
  if (rounds && peers && t.epi == EPI_TWO_SHOT) g = g < 4 ? g : 4;
  // A reduce-scatter rank sums the slots only for its own band of rows.  With XCD spans that are
  // close to square that band falls to one or two XCDs, whose CUs then carry all the slow tiles;
  // taller groups spread it over more XCDs at the price of more operand panels per L2
  // (8192 x 4096 x 1376, 8 ranks, seven peers, on one box: 131 us at the default height 8, 114 at
  // 16, 119 at 32; fetched by the L2s: 207, 290 and 443 MB).
  const bool rs_band = t.epi == EPI_REDUCE_SCATTER && !t.all_owners && peers;
  if (rs_band) g = g * 2 < o.tiles_m ? g * 2 : o.tiles_m;
  o.interleave = 0;
  o.tile_rotate = 0;
  // Launches whose epilogue streams whole tiles from or to every rank - the one-shot all-reduce with peers
  // spends half its time reading the peers' tiles, matmul_all_gather and the atomic variant write every
  // tile into all slots - want the workgroups that run together to touch long pieces of the same rows
  // (DRAM pages stay open): flat groups of two rows - more for narrow outputs, so that g x tiles_n stays
  // near 32 (64 with two workgroups per CU) and an L2 still sees as few operand panels as with a square
  // span.  When the launch fills at least three quarters of the chip the grouped order is also dealt out
  // workgroup by workgroup instead of in one span per XCD: XCD x then holds the tiles at positions x modulo
  // the XCD count, 1/g of the rows and g/8 of the columns of one band of rows that the whole chip works on.
  // Measured, eight ranks, one box, square spans -> this rule; one-shot: fp8 16384x8192x1024 568 -> 496 us
  // (520 with flat spans), bf16 8192x4096x1376 216 -> 194, 4096x4096x1376 98.0 -> 96.8, 2048x8192x1376
  // 108 -> 99, 2048x4096x1376 (128x128 tiles) 64.6 -> 60.4, 256x4096x4096 (64x64 tiles, chip half full:
  // spans) 39.3 -> 32.2; atomic fp16 8192x4096x1376 566 -> 520; matmul_all_gather fp16 2048x3584x8192
  // 175 -> 168, 512x4096x1376 22.9 -> 21.4.  Dealt out with one-row groups or spans of eight rows are the
  // outliers (+9 % on 1536x6144x2048), and a chip that is little more than half full does better with spans
  // (3072x3072x1024: 67.9 against 70.6).  Two-shot launches lose 3-5 % when dealt out; launches that
  // neither read nor write other ranks' tiles do not care.
  const bool streams_tiles = t.world > 1 && ((t.epi == EPI_ONE_SHOT && t.sum_peers) || t.epi == EPI_ALL_GATHER || t.epi == EPI_ATOMIC);
  if (streams_tiles) {
    g = 2;
    while (g < 8 && g * 2 * o.tiles_n <= (t.two_per_cu ? 64 : 32)) g *= 2;
    while (g > o.tiles_m && g > 1) g /= 2;
    o.interleave = (long long)o.tiles_m * o.tiles_n * 4 >= (long long)t.resident * t.num_xcd * 3;
  }
  o.group_m_spans = g;
  // The reduce-scatter with peers is dealt out as well (its launches hand one workgroup per tile to the
  // hardware in this order), starting with the band of rows this rank sums: those tiles take half as long
  // again as the others, so they go first and spread over every XCD (8192x4096x1376, eight ranks, rank 0:
  // 111.8 -> 106.6 us against spans of sixteen rows).  A band that would fill more than five eighths of the chip with workgroups
  // that wait - for tiles that the other ranks only reach behind theirs - has to keep its place in the common order (last of
  // eight ranks, own band first -> common order, us: 16384x8192x512, bands of 256 tiles, 228 -> 244; of two ranks 8192x8192x1024
  // 156 -> 159, 8192x4096x1376 97 -> 97).
  if (rs_band) {
    o.interleave = 1;
    g = o.tiles_m >= 2 ? 2 : 1;
    int first = 0, last = 0;
    if (band_tile_rows(t, first, last) && publishes_alone(t, g)) o.tile_rotate = first / g * g * o.tiles_n;
  }
  o.group_m = g;
  return o;
}

// Workgroups of a launch whose tiles are walked by the resident workgroups: as many as run at one time (`cap`), or the
// tiles if these are fewer.  A multiple of the XCD count keeps the XCD mapping exact.  Rounded up when the tiles fit in one
// round (the surplus workgroups find no tile and leave), so that no tile waits for a second round.
IRIS_HD int resident_grid(int total, int cap, int num_xcd) {
  int grid = total < cap ? total : cap;
  if (grid % num_xcd) {
    const int up = grid + num_xcd - grid % num_xcd;
    grid = up <= cap ? up : grid - grid % num_xcd;
  }
  return grid < 1 ? 1 : grid;
}

// Whether a launch of several rounds has one workgroup per tile, handed out by the hardware as CUs free up.  The two-shot
// all-reduce does better that way (measured at W = 8: 16384x4096x1376 322 -> 273 us, 8192x8192x2752 461 -> 417 us,
// 8192x8192x8192 1059 -> 1009 us); the one-shot variant does worse (+3-7 %), launches
// without peers do not care.  The same goes for a reduce-scatter whose rank owns one block of
// rows: the few tiles that carry the slot sum take half as long again as the others, and a fixed
// tile-to-workgroup assignment gives some workgroups two of them.
IRIS_HD bool workgroup_per_tile(int epi, int world, int sum_peers, int all_owners) {
  return world > 1 && sum_peers && (epi == EPI_TWO_SHOT || (epi == EPI_REDUCE_SCATTER && !all_owners));
}

// Group height of the any-shape kernel's spans (one workgroup per tile, xcd_tile_index): close to square groups of the tiles an XCD
// works on at one time, the same on every rank.
IRIS_HD int any_group_m(int tiles_m, int tiles_n, int num_xcd, int resident) {
  const int span = cdiv(tiles_m * tiles_n, num_xcd), at_once = span < resident ? span : resident;
  int g = 1;
  while (g * g * 2 <= at_once && g * 2 <= tiles_m) g *= 2;
  return g;
}

// ---------------------------------------------------------------------------------------------
// Tail policy of the 256x256 tile: how the tiles of a partly filled last round are split along K.
//
// An XCD's `wgs` workgroups meet `left` (< wgs) tiles in the last round.  When at most half of them
// would get a tile, workgroup h < left HELPS tile h: the tile's MAIN workgroup (the last `left`
// workgroups of the XCD) multiplies the K steps [0, main_steps) and owns the epilogue, the helper
// multiplies [main_steps, nsteps) and passes its fp32 accumulators on as a partial sum.  Helpers beyond
// `left` stay idle.
// All mains walk K from step 0 at the same pace and all helpers from main_steps, as the whole tiles of
// the earlier rounds do, so the operand panels they share keep meeting in the XCD's L2.  What was measured
// and left out (bf16, one rank, kernel time whole -> split):
//   - the textbook scheme, the round's K steps cut into equal consecutive shares: every workgroup sits at
//     another K offset and the operand traffic from the last-level cache grows ninefold
//     (8192 x 1792 x 4096, 28 of 32 tiles left: 116 -> 154 us);
//   - several helpers per tile: the main adds their partial sums one after the other
//     (5120 x 3840 x 4096, 6 of 32 left, four helpers each: 187 -> 192 us; one helper each: 186 -> 163);
//   - a helper serving several tiles in a row when more than half of the round is filled
//     (4096 x 2880 x 4096, 24 of 32 left, three tiles per helper: 91 -> 102 us).
// main_steps balances the main's work (its steps, then `gather_cost` steps' worth of loading the partial
// sum) against the helper's (its steps, `pass_cost` steps' worth of pipeline fill and storing the partial
// sum).  per_tile = 0 means: do not split (nothing to gain).  With both costs at 0 (a test setting) every
// round of at least 4 K steps that can be split is split.
// ---------------------------------------------------------------------------------------------
struct SplitPlan {
  int per_tile;     // helper pieces per tile (0: tiles stay whole)
  int per_helper;   // tiles a helper serves
  int main_steps;   // K steps [0, main_steps) stay with the main
  int piece_steps;  // K steps of a helper piece (the last piece of a tile may be shorter)
};
// In K steps of the 256x256 tile (about 0.75 us each), from time stamps inside a split launch
// (8192 x 2880 x 4096 bf16): a helper's 256 KiB of partial sums are stored and acknowledged 4.7 us after
// its last K step, and the next tile's first operands land 3 us later; the main has the partial sum in
// its staged tile 6 us after the helper's flag went up, 4.5 us more than staging alone takes.
constexpr int kSplitGatherCost = 8;
constexpr int kSplitPassCost = 10;

IRIS_HD SplitPlan split_plan(int left, int wgs, int nsteps, int gather_cost = kSplitGatherCost, int pass_cost = kSplitPassCost) {
  SplitPlan s = {0, 1, nsteps, 0};
  const int helpers = wgs - left;
  if (left <= 0 || helpers <= 0 || nsteps < 4) return s;
  if (helpers < left) return s;  // more than half of the round is filled
  const int n = 1, m = 1;
  // main_steps + n * gather = m * ((nsteps - main_steps) / n + pass)
  long num = (long)m * nsteps + (long)n * m * pass_cost - (long)n * n * gather_cost;
  int main_steps = (int)(num / (n + m));
  if (main_steps < 1) main_steps = 1;
  if (main_steps > nsteps - n) return s;        // every helper piece needs a step
  const int piece = (nsteps - main_steps + n - 1) / n;
  // The round as its slowest workgroup sees it, in K steps; a split that does not beat a whole tile is none.
  const int main_cost = main_steps + n * gather_cost;
  const int helper_cost = m * (piece + pass_cost);
  if ((main_cost > helper_cost ? main_cost : helper_cost) >= nsteps) return s;
  s.per_tile = n;
  s.per_helper = m;
  s.main_steps = main_steps;
  s.piece_steps = piece;
  return s;
}
// K steps the slowest workgroup of the round spends, split or not (what the launch code compares).
IRIS_HD int split_round_steps(const SplitPlan& s, int nsteps, int gather_cost = kSplitGatherCost, int pass_cost = kSplitPassCost) {
  if (s.per_tile == 0) return nsteps;
  const int main_cost = s.main_steps + s.per_tile * gather_cost;
  const int helper_cost = s.per_helper * (s.piece_steps + pass_cost);
  return main_cost > helper_cost ? main_cost : helper_cost;
}

// What workgroup `local` (0 .. wgs-1) of an XCD does in the split round as its `served`-th item (0, 1, ...).
// Returns false when it has nothing (more) to do.  Otherwise tile j (0 .. left-1) of the round, the K
// steps [k_begin, k_end), and
//   kind 0: a whole tile (the plan does not split),
//   kind 1: a helper piece - the accumulators go to partial-sum slot `slot`,
//   kind 2: the main's piece - the partial sum in slot `slot` is added before the epilogue (partners = 1).
// Slots count from 0 within the XCD (all below wgs).  Helpers are the first
// wgs - left workgroups, mains the last `left`.
IRIS_HD bool split_item(const SplitPlan& s, int left, int wgs, int nsteps, int local, int served,
                        int& j, int& k_begin, int& k_end, int& kind, int& partners, int& slot) {
  const int helpers = wgs - left;
  k_begin = 0; k_end = nsteps; kind = 0; partners = 0; slot = 0;
  if (local >= helpers) {  // main
    if (served > 0) return false;
    j = local - helpers;
    if (s.per_tile > 0) {
      kind = 2;
      k_end = s.main_steps;
      const int pieces = (nsteps - s.main_steps + s.piece_steps - 1) / s.piece_steps;
      partners = pieces < s.per_tile ? pieces : s.per_tile;
      slot = j * s.per_tile;
    }
    return true;
  }
  if (s.per_tile == 0 || served >= s.per_helper) return false;
  int piece = 1;
  if (s.per_helper > 1) {
    j = local * s.per_helper + served;
  } else {
    j = local % left;
    piece = 1 + local / left;
  }
  k_begin = s.main_steps + (piece - 1) * s.piece_steps;
  if (j >= left || piece > s.per_tile || k_begin >= nsteps) return false;
  k_end = k_begin + s.piece_steps < nsteps ? k_begin + s.piece_steps : nsteps;
  kind = 1;
  slot = j * s.per_tile + piece - 1;
  return true;
}

// The 32x32 small-output kernel addresses A from the operand's first row (of the slot that holds it) and
// the peers' aux tiles from the buffer's first element, with 32-bit byte offsets into a buffer resource
// of 2^31 bytes: an offset at or beyond 2^31 would read zeros.  True when every offset the kernel can
// form stays below that: a_rows rows of A (the rows one slot holds) with a stride of s_am elements of es
// bytes and K elements per row; M x N outputs of 2-byte elements with a row stride of s_cm elements.
// Launches that fail the test take the tiled kernels, which rebase their resources per tile.
IRIS_HD bool decode_offsets_fit(long long a_rows, long long s_am, long long K, int es, long long M, long long s_cm, long long N) {
  const long long limit = 1ll << 31;
  const long long a_last = (a_rows - 1) * s_am * es + K * es;  // one past the last byte of A
  const long long c_last = ((M - 1) * s_cm + N) * 2;            // ... of aux / C
  return a_rows > 0 && s_am >= 0 && s_cm >= 0 && a_last < limit && c_last < limit;
}

// ---------------------------------------------------------------------------------------------
// The vote of a workgroup on a word in LDS, where the K loop has one barrier per step: in which steps the word is read
// behind the barrier (to leave the loop early, the same step for every wave), and in which it may be written in front
// of it.  Between two barriers there is either a read or a write: a wave that has read behind the barrier of step s may
// run through step s + 1 while another one has yet to read.
// ---------------------------------------------------------------------------------------------
IRIS_HD bool vote_read_behind_barrier(int step) { return (step & 7) == 7; }
IRIS_HD bool vote_written_before_barrier(int step) { return (step & 7) != 0; }

// ---------------------------------------------------------------------------------------------
// Stand-alone collectives: a consecutive run of tiles of the grouped order (groups of group_m tile rows walked column
// by column) is the rest of a column, some columns of a group, whole groups, and the mirror image at the end - at most
// five rectangles.  Walked row by row, a workgroup moves kilobytes of every row instead of tiles' 128-byte rows (bf16
// 8192x2880 two-shot, eight ranks: 22.2 -> 19.8 us).
// ---------------------------------------------------------------------------------------------
struct RowRect {
  int pm0, pn0, width;  // first tile row and column, units per row
  long long base;       // index of the rectangle's first unit
};
constexpr int kMaxRowRects = 5;

// The rectangles of tiles [first, first + n) of a tiles_m x tiles_n grid, group_m <= tiles_m; a tile has bm rows of upr
// units.  Returns how many there are.
inline int row_rects(RowRect (&rect)[kMaxRowRects], int first, int n, int tiles_m, int tiles_n, int group_m, int bm, int upr) {
  int count = 0;
  long long base = 0;
  auto add = [&](int pm0, int rows, int pn0, int cols) {
    if (rows <= 0 || cols <= 0) return;
    rect[count++] = {pm0, pn0, cols * upr, base};
    base += (long long)rows * bm * cols * upr;
  };
  const int per_group = group_m * tiles_n, total = tiles_m * tiles_n;
  const int end = first + n;
  int t = first;
  auto inside_group = [&](int stop) {  // tiles [t, stop) of one group
    const int m0 = t / per_group * group_m, gs = tiles_m - m0 < group_m ? tiles_m - m0 : group_m;
    const int a = t - m0 * tiles_n, b = stop - m0 * tiles_n;  // positions in the group, column by column
    const int first_col = (a + gs - 1) / gs, last_col = b / gs;  // whole columns [first_col, last_col)
    if (first_col > last_col) {                                  // all in one column
      add(m0 + a % gs, b - a, a / gs, 1);
    } else {
      if (a % gs) add(m0 + a % gs, gs - a % gs, a / gs, 1);
      add(m0, gs, first_col, last_col - first_col);
      if (b % gs) add(m0, b % gs, last_col, 1);
    }
    t = stop;
  };
  if (t % per_group) {
    const long long next = ((long long)t / per_group + 1) * per_group;
    inside_group(next < end ? (int)next : end);
  }
  const int whole_end = end == total ? end : end / per_group * per_group;
  if (t < whole_end) {
    const int m0 = t / per_group * group_m, m1 = whole_end == total ? tiles_m : whole_end / per_group * group_m;
    add(m0, m1 - m0, 0, tiles_n);
    t = whole_end;
  }
  if (t < end) inside_group(end);
  return count;
}

// Tile (pm, pn) and unit inside it of unit g, for fewer than 2^31 units.
IRIS_HD void row_rect_unit(const RowRect (&rect)[kMaxRowRects], int n_rects, long long g, int bm, int upr, int& pm, int& pn, int& unit) {
  int pm0 = rect[0].pm0, pn0 = rect[0].pn0, width = rect[0].width;
  long long first_unit = 0;
#pragma unroll
  for (int i = 1; i < kMaxRowRects; ++i) {
    if (i < n_rects && g >= rect[i].base) {
      pm0 = rect[i].pm0, pn0 = rect[i].pn0, width = rect[i].width;
      first_unit = rect[i].base;
    }
  }
  const unsigned in_rect = (unsigned)(g - first_unit), r = in_rect / (unsigned)width, across = in_rect - r * (unsigned)width;
  pm = pm0 + (int)(r / (unsigned)bm);
  pn = pn0 + (int)(across / (unsigned)upr);
  unit = (int)(r % (unsigned)bm) * upr + (int)(across % (unsigned)upr);
}

// Position of a tile in the grouped order.
IRIS_HD int grouped_tile_id(int pm, int pn, int tiles_m, int tiles_n, int group_m) {
  const int first_m = pm / group_m * group_m, gs = tiles_m - first_m < group_m ? tiles_m - first_m : group_m;
  return first_m * tiles_n + pn * gs + pm - first_m;
}

}  // namespace iris_layout
