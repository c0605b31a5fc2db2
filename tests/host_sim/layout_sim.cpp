// Host-side check of iris_amd/csrc/layout.h: replays, on the CPU, what the gfx950 kernels do with the
// index functions - direct-to-LDS deposits, 16-byte fragment reads, LDS transpose reads - and checks
// that every MFMA operand slot receives the element the kernel assumes, that the LDS swizzles are
// bijections without bank conflicts inside a 16-lane group, and that the tile orders and flag-tile
// counts are exact.  The transpose-read semantics used here (within each 16-lane group, output lane i
// element e comes from input lane 4e + i/4, element i%4 for 16-bit data; input lane 2e + i/8, byte
// i%8 for 8-bit data) were measured on an MI355X.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <vector>

#include "layout.h"

using namespace iris_layout;

static int failures = 0;
#define CHECK(cond, ...)                         \
  do {                                           \
    if (!(cond)) {                               \
      if (failures < 20) { printf("FAIL %s:%d: ", __FILE__, __LINE__); printf(__VA_ARGS__); printf("\n"); } \
      ++failures;                                \
    }                                            \
  } while (0)

// ---- swizzle bijection + bank spread -------------------------------------------------------------
template <int RB>
void check_row_tile(int rows) {
  using T = RowTile<RB>;
  std::set<int> seen;
  for (int r = 0; r < rows; ++r)
    for (int c = 0; c < T::kChunksPerRow; ++c) {
      int off = T::lds_offset(r, c);
      CHECK(off >= 0 && off < rows * RB && off % 16 == 0, "row tile offset out of range");
      CHECK(seen.insert(off).second, "row tile offset reused");
      int r2, c2;
      T::from_lds(off, r2, c2);
      CHECK(r2 == r && c2 == c, "row tile inverse mismatch RB=%d r=%d c=%d", RB, r, c);
    }
  // 16 lanes reading the same logical chunk of 16 consecutive rows: 16 distinct 16-byte bank groups
  for (int r0 = 0; r0 + 16 <= rows; r0 += 16)
    for (int c = 0; c < T::kChunksPerRow; ++c) {
      std::set<int> banks;
      for (int i = 0; i < 16; ++i) banks.insert((T::lds_offset(r0 + i, c) % 256) / 16);
      CHECK(banks.size() == 16, "row tile RB=%d bank conflict at rows %d.., chunk %d (%zu groups)", RB, r0, c, banks.size());
    }
}

template <int RB, int ES>
void check_col_tile(int krows) {
  using T = ColTile<RB, ES>;
  std::set<int> seen;
  for (int k = 0; k < krows; ++k)
    for (int c = 0; c < T::kChunksPerRow; ++c) {
      int off = T::lds_offset(k, c);
      CHECK(off >= 0 && off < krows * RB, "col tile offset out of range");
      CHECK(seen.insert(off).second, "col tile offset reused");
      int k2, c2;
      T::from_lds(off, k2, c2);
      CHECK(k2 == k && c2 == c, "col tile inverse mismatch");
    }
}

// ---- simulate loader + fragment reads for one operand tile -----------------------------------------
// Element identity: (row-or-k, col) packed in an int; the simulated LDS stores one id per element.
struct Lds {
  std::vector<int> id;  // per byte/ES element slot
  int es;
  Lds(int bytes, int es_) : id(bytes / es_, -1), es(es_) {}
  int& at(int byte_off) { return id[byte_off / es]; }
};

// K-contiguous operand (A, or B^T): tile [rows][BK], fragment lanes per frag16_*/frag8_*.
template <int RB, int ES>
void sim_row_operand(int rows, int nwaves) {
  using T = RowTile<RB>;
  const int CE = 16 / ES, BK = RB / ES;
  Lds lds(rows * RB, ES);
  // loader: wave w, instruction i deposits 1 KiB at (w + i*nwaves)*1024; lane l its 16 bytes
  const int ninstr = rows * RB / kDmaBytes;
  for (int q = 0; q < ninstr; ++q)
    for (int lane = 0; lane < 64; ++lane) {
      int off = q * kDmaBytes + lane * 16, row, c;
      T::from_lds(off, row, c);
      for (int e = 0; e < CE; ++e) lds.at(off + e * ES) = row * 4096 + (c * CE + e);  // global (row, k)
    }
  for (int x : lds.id) CHECK(x >= 0, "row operand: LDS element never written");
  // fragment reads: block of 32 rows starting at r0, every k-slice
  const int KM = ES == 2 ? 16 : 64;
  for (int r0 = 0; r0 + 32 <= rows; r0 += 32)
    for (int kk = 0; kk < BK / KM; ++kk)
      for (int lane = 0; lane < 64; ++lane) {
        const int nfrag = ES == 2 ? 1 : 2;
        for (int h = 0; h < nfrag; ++h) {
          int c = ES == 2 ? frag16_chunk(lane, kk) : frag8_chunk(lane, kk, h);
          int off = T::lds_offset(r0 + frag16_row(lane), c);
          for (int e = 0; e < CE; ++e) {
            int got = lds.at(off + e * ES);
            // MFMA slot: row lane%32, k = kk*KM + (KM/2)*(lane/32) + h*CE + e
            int want = (r0 + lane % 32) * 4096 + kk * KM + (KM / 2) * (lane / 32) + h * CE + e;
            CHECK(got == want, "row operand ES=%d lane %d kk %d: got (%d,%d) want (%d,%d)", ES, lane, kk, got / 4096, got % 4096, want / 4096, want % 4096);
          }
        }
      }
}

// N-contiguous operand (row-major B): tile [BK][BN], transpose reads.
template <int RB, int ES>
void sim_col_operand(int BK) {
  using T = ColTile<RB, ES>;
  const int CE = 16 / ES, BN = RB / ES;
  Lds lds(BK * RB, ES);
  const int ninstr = BK * RB / kDmaBytes;
  for (int q = 0; q < ninstr; ++q)
    for (int lane = 0; lane < 64; ++lane) {
      int off = q * kDmaBytes + lane * 16, k, c;
      T::from_lds(off, k, c);
      for (int e = 0; e < CE; ++e) lds.at(off + e * ES) = k * 4096 + (c * CE + e);  // global (k, n)
    }
  for (int x : lds.id) CHECK(x >= 0, "col operand: LDS element never written");
  const int KM = ES == 2 ? 16 : 64;
  const int per_read = ES == 2 ? 4 : 8;     // elements a lane contributes / receives per transpose read
  const int nreads = ES == 2 ? 2 : 4;
  for (int n0 = 0; n0 + 32 <= BN; n0 += 32)
    for (int kk = 0; kk < BK / KM; ++kk)
      for (int rd = 0; rd < nreads; ++rd) {
        // every lane presents an address; the hardware redistributes within 16-lane groups
        int addr[64];
        std::set<int> banks_by_group[2];  // LDS serves a transpose read one half-wave (256 bytes) at a time
        for (int lane = 0; lane < 64; ++lane) {
          int krow = ES == 2 ? tr16_krow(lane, kk, rd) : tr8_krow(lane, kk, rd);
          int n = n0 + (ES == 2 ? tr16_ncol(lane) : tr8_ncol(lane));
          addr[lane] = T::lds_offset(krow, n / CE) + (n % CE) * ES;
          for (int b = 0; b < 8; b += 4) banks_by_group[lane / 32].insert(((addr[lane] + b) % 256) / 4);
        }
        for (int g = 0; g < 2; ++g)
          CHECK(banks_by_group[g].size() == 64, "col operand ES=%d RB=%d: bank conflict in half-wave %d (%zu banks)", ES, RB, g, banks_by_group[g].size());
        for (int lane = 0; lane < 64; ++lane) {
          int grp = lane / 16, i = lane % 16;
          for (int e = 0; e < per_read; ++e) {
            int src_lane = grp * 16 + (ES == 2 ? 4 * e + i / 4 : 2 * e + i / 8);
            int src_elem = ES == 2 ? i % 4 : i % 8;
            int got = lds.at(addr[src_lane] + src_elem * ES);
            // MFMA slot of lane: n = lane%32, k = kk*KM + (KM/2)*(lane/32) + rd*per_read + e
            int want = (kk * KM + (KM / 2) * (lane / 32) + rd * per_read + e) * 4096 + n0 + lane % 32;
            CHECK(got == want, "col operand ES=%d lane %d kk %d read %d elem %d: got (k%d,n%d) want (k%d,n%d)", ES, lane, kk, rd, e,
                  got / 4096, got % 4096, want / 4096, want % 4096);
          }
        }
      }
}

// The 16x16x32 products of 16-bit data: fragments of 16 rows (mma16_*), [k][n] tiles in ColTile16.
template <int RB>
void check_col_tile16(int krows) {
  using T = ColTile16<RB>;
  std::set<int> seen;
  for (int k = 0; k < krows; ++k)
    for (int c = 0; c < T::kChunksPerRow; ++c) {
      int off = T::lds_offset(k, c), k2, c2;
      CHECK(off >= 0 && off < krows * RB && seen.insert(off).second, "col tile 16 offset out of range or reused");
      T::from_lds(off, k2, c2);
      CHECK(k2 == k && c2 == c, "col tile 16 inverse mismatch");
    }
}

template <int RB>
void sim_row_operand16(int rows) {
  using T = RowTile16<RB>;
  std::set<int> seen;
  for (int off = 0; off < rows * RB; off += 16) {
    int row, c;
    T::from_lds(off, row, c);
    CHECK(row < rows && T::lds_offset(row, c) == off && seen.insert(row * T::kChunksPerRow + c).second, "row tile 16 inverse mismatch RB=%d", RB);
  }
  for (int r0 = 0; r0 + 16 <= rows; r0 += 16)
    for (int kk = 0; kk < RB / 64; ++kk) {
      std::set<int> banks[4];  // the lanes that LDS serves together
      for (int lane = 0; lane < 64; ++lane) {
        // the kernel adds the block's first row to the address of row lane % 16: the swizzle must repeat every 16 rows
        const int off = T::lds_offset(mma16_row(lane), mma16_chunk(lane, kk)) + r0 * RB;
        int row, c;
        T::from_lds(off, row, c);
        CHECK(row == r0 + lane % 16 && c == kk * 4 + lane / 16, "row operand 16: RB=%d lane %d", RB, lane);
        const int l = lane % 32, second = (l >= 4 && l < 12) || (l >= 16 && l < 20) || l >= 28;
        banks[lane / 32 * 2 + second].insert(off % 256 / 16);
      }
      for (int g = 0; g < 4; ++g) CHECK(banks[g].size() == 16, "row operand 16: bank conflict RB=%d group %d (%zu)", RB, g, banks[g].size());
    }
}

template <int RB>
void sim_col_operand16(int BK) {
  using T = ColTile16<RB>;
  for (int n0 = 0; n0 + 16 <= RB / 2; n0 += 16)
    for (int kk = 0; kk < BK / 32; ++kk)
      for (int j = 0; j < 2; ++j) {
        int addr[64];
        std::set<int> banks[2];
        for (int lane = 0; lane < 64; ++lane) {
          // one address per column block, read j and slice kk at constant distances from it
          const int n = n0 + mma16_tr_ncol(lane);
          addr[lane] = T::lds_offset(mma16_tr_krow(lane, 0, 0), n / 8) + n % 8 * 2 + (kk * 32 + 4 * j) * RB;
          CHECK(addr[lane] == T::lds_offset(mma16_tr_krow(lane, kk, j), n / 8) + n % 8 * 2, "col operand 16: swizzle of read %d", j);
          for (int b = 0; b < 8; b += 4) banks[lane / 32].insert((addr[lane] + b) % 256 / 4);
        }
        for (int g = 0; g < 2; ++g) CHECK(banks[g].size() == 64, "col operand 16: bank conflict RB=%d half-wave %d (%zu)", RB, g, banks[g].size());
        for (int lane = 0; lane < 64; ++lane)
          for (int e = 0; e < 4; ++e) {
            const int i = lane % 16, src = lane / 16 * 16 + 4 * e + i / 4;  // the transpose within 16 lanes
            int k, c;
            T::from_lds(addr[src] / 16 * 16, k, c);
            const int n = c * 8 + addr[src] % 16 / 2 + i % 4;
            CHECK(k == kk * 32 + 8 * (lane / 16) + 4 * j + e && n == n0 + i, "col operand 16: lane %d elem %d got (k%d,n%d)", lane, e, k, n);
          }
      }
}

// The order of a k-slice's products: every block once, the first quadrant from the first half of the fragments, the first
// half of the products from half of A's.
template <int MB, int NB>
void check_quad_blocks() {
  std::set<int> seen;
  for (int i = 0; i < MB * NB; ++i) {
    int mb, nb;
    quad_block<MB, NB>(i, mb, nb);
    CHECK(mb >= 0 && mb < MB && nb >= 0 && nb < NB && seen.insert(mb * NB + nb).second, "quad_block<%d,%d>(%d)", MB, NB, i);
    if (i < MB * NB / 4) CHECK(mb < MB / 2 && nb < NB / 2, "quad_block: first quadrant");
    if (i < MB * NB / 2) CHECK(mb < MB / 2, "quad_block: first half");
  }
}

void check_acc_layout16() {
  std::set<int> seen;
  for (int lane = 0; lane < 64; ++lane)
    for (int i = 0; i < 4; ++i) seen.insert(mma16_acc_row(lane, i) * 16 + mma16_acc_col(lane));
  CHECK(seen.size() == 256 && *seen.rbegin() == 255, "acc layout 16 must cover the block");
}

// ---- accumulator layout: every (n, m) of a 32x32 block owned exactly once -----------------------------
void check_acc_layout() {
  std::set<int> seen;
  for (int lane = 0; lane < 64; ++lane)
    for (int i = 0; i < 16; ++i) {
      int r = acc_row(lane, i), c = acc_col(lane);
      CHECK(r >= 0 && r < 32 && c >= 0 && c < 32, "acc index range");
      CHECK(seen.insert(r * 32 + c).second, "acc element owned twice");
      if (i % 4) CHECK(acc_row(lane, i) == acc_row(lane, i - 1) + 1, "acc rows of a register quad must be consecutive");
    }
  CHECK(seen.size() == 1024, "acc layout must cover the block");
}

// ---- tile orders ---------------------------------------------------------------------------------------
void check_tile_orders() {
  for (int tm = 1; tm <= 40; tm += 3)
    for (int tn = 1; tn <= 40; tn += 5)
      for (int g : {1, 2, 4, 8, 16}) {
        std::set<int> seen;
        for (int idx = 0; idx < tm * tn; ++idx) {
          int a, b;
          grouped_tile(idx, tm, tn, g, a, b);
          CHECK(a >= 0 && a < tm && b >= 0 && b < tn, "grouped_tile out of range tm=%d tn=%d g=%d idx=%d -> (%d,%d)", tm, tn, g, idx, a, b);
          seen.insert(a * tn + b);
        }
        CHECK((int)seen.size() == tm * tn, "grouped_tile is not a bijection tm=%d tn=%d g=%d", tm, tn, g);
      }
  for (int total : {1, 7, 8, 10, 224, 255, 256, 257, 1000, 2048})
    for (int nwg : {1, 5, 8, 16, 224, 256})
      for (int xcd : {1, 8}) {
        std::map<int, int> count;
        for (int wg = 0; wg < nwg; ++wg) {
          bool ended = false;
          for (int it = 0; it < total + 2; ++it) {
            int idx = xcd_tile_index(wg, nwg, it, total, xcd);
            if (idx < 0) { ended = true; continue; }
            CHECK(!ended, "xcd_tile_index resumed after it ended (total=%d nwg=%d)", total, nwg);
            CHECK(idx < total, "xcd_tile_index out of range");
            count[idx]++;
          }
        }
        CHECK((int)count.size() == total, "xcd_tile_index misses tiles: total=%d nwg=%d xcd=%d covered=%zu", total, nwg, xcd, count.size());
        for (auto& kv : count) CHECK(kv.second == 1, "tile %d processed %d times", kv.first, kv.second);
      }
}

// The order launches that stream whole tiles use: the grouped order dealt out workgroup by workgroup
// (xcd_tile_index with one "XCD"), optionally started `rotate` positions in (the reduce-scatter starts
// at the rank's own band of rows).  Every tile exactly once; and with groups of g rows, XCD x (workgroup
// index modulo 8) of a full first round meets 1/g of the round's tile rows and g/8 of its tile columns.
void check_dealt_order() {
  struct Case { int tm, tn, g, nwg, rotate; };
  for (Case c : {Case{16, 16, 2, 256, 0}, Case{64, 32, 2, 256, 0}, Case{32, 16, 2, 256, 2 * 16 * 5}, Case{32, 16, 2, 512, 2 * 16 * 15},
                 Case{7, 23, 2, 168, 46}, Case{32, 8, 4, 256, 0}}) {
    const int total = c.tm * c.tn;
    std::vector<int> count(total, 0);
    for (int wg = 0; wg < c.nwg; ++wg)
      for (int it = 0;; ++it) {
        int idx = xcd_tile_index(wg, c.nwg, it, total, 1);
        if (idx < 0) break;
        idx += c.rotate;
        if (idx >= total) idx -= total;
        CHECK(idx >= 0 && idx < total, "dealt order out of range");
        count[idx]++;
      }
    for (int t = 0; t < total; ++t) CHECK(count[t] == 1, "dealt order: tile %d taken %d times (tm=%d tn=%d)", t, count[t], c.tm, c.tn);
  }
  // 16 x 16 tiles, groups of two rows, 256 workgroups on 8 XCDs: each XCD sees 8 of the 16 tile rows and 4 of the 16 tile columns
  for (int xcd = 0; xcd < 8; ++xcd) {
    std::set<int> rows, cols;
    for (int wg = xcd; wg < 256; wg += 8) {
      int a, b;
      grouped_tile(xcd_tile_index(wg, 256, 0, 256, 1), 16, 16, 2, a, b);
      rows.insert(a);
      cols.insert(b);
    }
    CHECK(rows.size() == 8 && cols.size() == 4, "dealt order: XCD %d meets %zu tile rows and %zu tile columns", xcd, rows.size(), cols.size());
  }
}

// ---- flag tiles ----------------------------------------------------------------------------------------
void check_flag_counts() {
  struct Case { int M, N, FM, FN, KM, KN; };
  for (Case c : {Case{4096, 4096, 256, 64, 256, 256}, Case{1024, 1024, 512, 512, 128, 128}, Case{1024, 1024, 384, 200, 128, 128},
                 Case{100, 72, 32, 24, 64, 64}, Case{257, 129, 64, 64, 64, 64}, Case{1000, 600, 96, 96, 256, 256}}) {
    int ftm = cdiv(c.M, c.FM), ftn = cdiv(c.N, c.FN);
    for (int fm = 0; fm < ftm; ++fm)
      for (int fn = 0; fn < ftn; ++fn) {
        std::set<int> macro;
        for (int m = fm * c.FM; m < (fm + 1) * c.FM && m < c.M; ++m)
          for (int n = fn * c.FN; n < (fn + 1) * c.FN && n < c.N; n += 1) macro.insert((m / c.KM) * 100000 + n / c.KN);
        int got = macro_tiles_over_flag_tile(fm, fn, c.FM, c.FN, c.KM, c.KN, c.M, c.N);
        CHECK(got == (int)macro.size(), "macro_tiles_over_flag_tile(%d,%d) = %d, brute force %zu", fm, fn, got, macro.size());
      }
  }
  for (int world : {1, 2, 3, 4, 8})
    for (int total : {1, 4, 7, 40, 64, 2048}) {
      int per = total / world;
      for (int t = 0; t < total; ++t) {
        int want = -1;
        for (int r = 0; r < world; ++r) {
          int s = r * per, e = (r == world - 1) ? total : s + per;
          if (t >= s && t < e) want = r;
        }
        CHECK(owner_contiguous(t, total, world) == want, "owner_contiguous(%d,%d,%d)", t, total, world);
        CHECK(owner_interleaved(t, world) == t % world, "owner_interleaved");
      }
    }
}

// Flag tiles summed as rectangles: their pieces cover the columns, stay inside, and start on 16-byte boundaries of rows that do
// wherever the rule says so.
void check_rect_pieces() {
  for (int oe : {4, 8})
    for (int bn : {64, 128, 256})
      for (int N : {bn, 2 * bn + oe, 5 * bn - oe})
        for (int flag_bn = oe; flag_bn <= 300; ++flag_bn)
          for (int n0 = 0; n0 < N; n0 += bn)
            for (int n1 = std::min(n0 + bn, N), fc = n0 / flag_bn; fc * flag_bn < n1; ++fc) {
              const int c0 = std::max(n0, fc * flag_bn) - n0, c1 = std::min(n1, (fc + 1) * flag_bn) - n0;
              if (c1 - c0 < oe) continue;
              int covered = c0;
              for (int i = 0; i < cdiv(c1 - c0, oe); ++i) {
                const int col = rect_piece_col(c0, c1, i, oe);
                CHECK(col >= c0 && col <= covered && col + oe <= c1, "piece %d of columns [%d, %d) at %d", i, c0, c1, col);
                CHECK(!rect_pieces_aligned(true, flag_bn, oe) || (n0 + col) % oe == 0, "flag tiles of %d columns, pieces of %d: one at column %d", flag_bn, oe, n0 + col);
                covered = col + oe;
              }
              CHECK(covered == c1, "pieces end at %d of [%d, %d)", covered, c0, c1);
            }
}

// The rule that keeps launches away from the 32x32 kernel when its 32-bit offsets would not reach.
void check_decode_offsets() {
  CHECK(decode_offsets_fit(32, 1024, 1024, 1, 32, 8192, 8192), "decode shape 32 x 8192 x 1024 fp8");
  CHECK(decode_offsets_fit(16384, 4096, 4096, 2, 16384, 32, 32), "tall output, 128 MiB of A");
  CHECK(!decode_offsets_fit(16384, 65536, 65536, 2, 16384, 32, 32), "16384 x 65536 bf16 is 2 GiB of A");
  CHECK(decode_offsets_fit(16384, 65536, 65536, 1, 16384, 32, 32), "the same in fp8 is 1 GiB");
  CHECK(!decode_offsets_fit(2048, 1 << 20, 512, 2, 2048, 32, 32), "padded A rows: 2048 rows of 2 MiB");
  CHECK(decode_offsets_fit(1023, 1 << 20, 512, 2, 1023, 32, 32), "1023 rows of 2 MiB end below 2 GiB");
  CHECK(!decode_offsets_fit(1025, 1 << 20, 512, 2, 1025, 32, 32), "1025 rows of 2 MiB do not");
  CHECK(!decode_offsets_fit(64, 512, 512, 2, 16385, 1 << 16, 32), "strided C view: 16385 rows of 128 KiB");
  CHECK(decode_offsets_fit(64, 512, 512, 2, 16384, 1 << 15, 32), "16384 rows of 64 KiB end below 2 GiB");
  CHECK(!decode_offsets_fit(0, 512, 512, 2, 64, 64, 64), "no rows");
}

// The tail policy: for every (tiles left in the last round, workgroups, K steps) the items of all
// workgroups must cover every K step of every tile exactly once, helpers must come before the mains that
// wait for them, slots must be distinct and within the XCD's share of the workspace, the main must expect
// exactly the partial sums that get written, in ascending K order, and the predicted round must never
// be longer than a whole tile.
void check_split_plan() {
  for (int wgs : {4, 32, 38})
    for (int left = 1; left < wgs; ++left)
      for (int nsteps : {1, 3, 4, 5, 10, 11, 43, 128, 129, 256, 1000})
      for (int costs = 0; costs < 2; ++costs) {  // planned with the measured costs, and with none (the test setting)
        const int gc = costs ? kSplitGatherCost : 0, pc = costs ? kSplitPassCost : 0;
        const SplitPlan s = split_plan(left, wgs, nsteps, gc, pc);
        CHECK(split_round_steps(s, nsteps, gc, pc) < nsteps || s.per_tile == 0, "split round not shorter than a tile: %d %d %d", left, wgs, nsteps);
        std::vector<std::vector<int>> covered(left, std::vector<int>(nsteps, 0));
        std::vector<int> slot_writer(wgs, -1), slot_begin(wgs, -1);
        std::vector<int> expects(left, 0), first_slot(left, 0), main_end(left, nsteps);
        for (int local = 0; local < wgs; ++local)
          for (int served = 0;; ++served) {
            int j, kb, ke, kind, partners, slot;
            if (!split_item(s, left, wgs, nsteps, local, served, j, kb, ke, kind, partners, slot)) break;
            CHECK(served < 64, "a workgroup never runs out of items");
            if (served >= 64) break;
            CHECK(j >= 0 && j < left && kb >= 0 && kb < ke && ke <= nsteps, "item out of range: %d %d %d wg %d", left, wgs, nsteps, local);
            for (int k = kb; k < ke; ++k) covered[j][k]++;
            if (kind == 1) {
              CHECK(local < wgs - left, "helper among the mains");
              CHECK(slot >= 0 && slot < wgs && slot_writer[slot] < 0, "slot %d reused or out of range (%d %d %d)", slot, left, wgs, nsteps);
              if (slot >= 0 && slot < wgs) { slot_writer[slot] = j; slot_begin[slot] = kb; }
            } else {
              CHECK(local >= wgs - left && kb == 0, "main among the helpers");
              CHECK((kind == 2) == (s.per_tile > 0), "kind of the main's item");
              expects[j] = partners; first_slot[j] = slot; main_end[j] = ke;
            }
          }
        for (int j = 0; j < left; ++j) {
          bool once = true;
          for (int k = 0; k < nsteps; ++k) once = once && covered[j][k] == 1;
          CHECK(once, "K steps of tile %d not covered exactly once (%d %d %d)", j, left, wgs, nsteps);
          int prev = main_end[j];
          for (int i = 0; i < expects[j]; ++i) {
            const int sl = first_slot[j] + i;
            CHECK(sl < wgs && slot_writer[sl] == j && slot_begin[sl] == prev, "main %d expects a partial sum nobody writes (%d %d %d)", j, left, wgs, nsteps);
            if (sl < wgs && slot_writer[sl] == j) prev = slot_begin[sl] + s.piece_steps;
          }
          int written = 0;
          for (int sl = 0; sl < wgs; ++sl) written += slot_writer[sl] == j;
          CHECK(written == expects[j], "tile %d: %d partial sums written, %d expected (%d %d %d)", j, written, expects[j], left, wgs, nsteps);
        }
      }
  // worked examples (32 workgroups per XCD).  More than half of the round filled: the tiles stay whole
  CHECK(split_plan(28, 32, 128).per_tile == 0 && split_plan(28, 32, 1024).per_tile == 0 && split_plan(17, 32, 1024).per_tile == 0,
        "a round that is more than half full stays whole");
  const SplitPlan h = split_plan(16, 32, 256);  // half a round: one helper per tile, about equal halves
  CHECK(h.per_tile == 1 && h.per_helper == 1 && h.main_steps == 129 && h.piece_steps == 127, "plan for 16/32/256: %d %d %d %d", h.per_tile, h.per_helper, h.main_steps, h.piece_steps);
  CHECK(split_round_steps(h, 256) == 137, "round of 16/32/256");
  const SplitPlan q = split_plan(6, 32, 256);   // a fifth of a round: still one helper per tile, twenty stay idle
  CHECK(q.per_tile == 1 && q.per_helper == 1 && q.main_steps == h.main_steps, "plan for 6/32/256: %d %d %d %d", q.per_tile, q.per_helper, q.main_steps, q.piece_steps);
  CHECK(split_plan(16, 32, 16).per_tile == 0, "16 K steps: the partial sum costs more than it saves");
}

// ---- row walk of the collectives -------------------------------------------------------------------
// Units walked by rectangles are exactly the units of the owned tiles, each once, and lead back to their tile's id:
// every grid of up to 7 x 6 tiles, every group height, every run of tiles.
void check_row_rects() {
  for (int tm = 1; tm <= 7; ++tm)
    for (int tn = 1; tn <= 6; ++tn)
      for (int g = 1; g <= tm; ++g) {
        std::vector<std::pair<int, int>> tile;  // the grouped order, written down
        for (int m0 = 0; m0 < tm; m0 += g)
          for (int n = 0; n < tn; ++n)
            for (int m = m0; m < tm && m < m0 + g; ++m) tile.push_back({m, n});
        for (int first = 0; first < tm * tn; ++first)
          for (int n = 1; first + n <= tm * tn; ++n) {
            const int bm = 1 + (first + n) % 3, upr = 1 + n % 3, upt = bm * upr;
            RowRect rect[kMaxRowRects];
            const int count = row_rects(rect, first, n, tm, tn, g, bm, upr);
            CHECK(count >= 1 && count <= kMaxRowRects, "%d rectangles (%d x %d, group %d, tiles %d + %d)", count, tm, tn, g, first, n);
            std::vector<int> seen(n * upt);
            for (long long u = 0; u < (long long)n * upt; ++u) {
              int pm, pn, unit;
              row_rect_unit(rect, count, u, bm, upr, pm, pn, unit);
              const int j = grouped_tile_id(pm, pn, tm, tn, g) - first;
              const bool owned = j >= 0 && j < n && unit >= 0 && unit < upt && tile[first + j] == std::make_pair(pm, pn);
              CHECK(owned && seen[j * upt + unit]++ == 0, "unit %lld: tile %d unit %d (%d x %d, group %d, tiles %d + %d)", u, j, unit, tm, tn, g, first, n);
            }
          }
      }
}

// ---- ranks that wait for each other ------------------------------------------------------------------
// One rank's launch: the tiles of every workgroup in turn, and the flag tiles that a tile publishes and waits for.
struct RankLaunch {
  TileLaunch t;
  std::vector<std::vector<int>> chain;  // kernel tiles (row * tiles_n + column) of workgroup b
  int resident;                         // workgroups that run at one time on an XCD
};

RankLaunch make_launch(const TileLaunch& t, const TileOrder& o, bool one_each, int xcds_of_order) {
  RankLaunch l;
  l.t = t;
  l.resident = t.resident;
  const int total = o.tiles_m * o.tiles_n;
  const int grid = one_each ? cdiv(total, t.num_xcd) * t.num_xcd : resident_grid(total, t.resident * t.num_xcd, t.num_xcd);
  l.chain.resize(grid);
  for (int wg = 0; wg < grid; ++wg)
    for (int it = 0; it == 0 || !one_each; ++it) {
      int idx = xcd_tile_index(wg, grid, it, total, xcds_of_order);
      if (idx < 0) break;
      idx = (idx + o.tile_rotate) % total;
      int tm, tn;
      grouped_tile(idx, o.tiles_m, o.tiles_n, o.group_m, tm, tn);
      l.chain[wg].push_back(tm * o.tiles_n + tn);
    }
  return l;
}

// fused_mfma_kernel as launch_mfma launches it.
RankLaunch tiled_launch(const TileLaunch& t) {
  const TileOrder o = tile_order(t);
  const bool rounds = o.tiles_m * o.tiles_n > resident_grid(o.tiles_m * o.tiles_n, t.resident * t.num_xcd, t.num_xcd);
  return make_launch(t, o, rounds && workgroup_per_tile(t.epi, t.world, t.sum_peers, t.all_owners), o.interleave ? 1 : t.num_xcd);
}

// The same tiles on packed operands (launch_mfma_rows), or the any-shape kernel in their place: as always, with a tile and an
// order of its own, or with the tiles and the order of the packed launch.
RankLaunch packed_launch(const TileLaunch& t, bool has_memory, int any_m, int any_n, int any_resident) {
  const TileOrder o = tile_order(t);
  if (has_memory || !publishes_alone(t, o.group_m)) return make_launch(t, o, true, o.interleave ? 1 : t.num_xcd);
  TileLaunch a = t;
  a.tile_m = any_m;
  a.tile_n = any_n;
  a.resident = any_resident;
  TileOrder own = {cdiv(a.M, any_m), cdiv(a.N, any_n), 0, 0, 0, 0};
  own.group_m = any_group_m(own.tiles_m, own.tiles_n, a.num_xcd, a.resident);
  return make_launch(a, own, true, a.num_xcd);
}

// How many workgroups of all ranks are left when nobody can go on.  Workgroup b runs on XCD b % num_xcd, in order, as
// soon as one in front of it has left (`in_order`: and not before all workgroups below b have started).
int replay(const std::vector<RankLaunch>& ranks, bool in_order) {
  struct State {
    std::vector<int> at, needed, published;  // tile of its chain a workgroup is at; per flag tile: kernel tiles over it, those done
    std::vector<char> told;
    std::vector<int> next, running;          // per XCD
    std::vector<int> live;                   // workgroups that run
    int started = 0;
  };
  std::vector<State> st(ranks.size());
  int left = 0;
  const TileLaunch& t0 = ranks[0].t;
  const int ftm = cdiv(t0.M, t0.flag_bm), ftn = cdiv(t0.N, t0.flag_bn);
  for (size_t r = 0; r < ranks.size(); ++r) {
    const RankLaunch& l = ranks[r];
    st[r].at.assign(l.chain.size(), 0);
    st[r].told.assign(l.chain.size(), 0);
    st[r].next.resize(l.t.num_xcd);
    for (int x = 0; x < l.t.num_xcd; ++x) st[r].next[x] = x;
    st[r].running.assign(l.t.num_xcd, 0);
    st[r].published.assign(ftm * ftn, 0);
    for (int f = 0; f < ftm * ftn; ++f)
      st[r].needed.push_back(macro_tiles_over_flag_tile(f / ftn, f % ftn, l.t.flag_bm, l.t.flag_bn, l.t.tile_m, l.t.tile_n, l.t.M, l.t.N));
    left += (int)l.chain.size();
  }
  for (bool moved = true; moved;) {
    moved = false;
    for (size_t r = 0; r < ranks.size(); ++r) {
      const RankLaunch& l = ranks[r];
      State& s = st[r];
      const TileLaunch& t = l.t;
      const int tiles_n = cdiv(t.N, t.tile_n), nwg = (int)l.chain.size();
      for (bool any = true; any;) {
        any = false;
        for (int x = 0; x < t.num_xcd; ++x)
          while (s.next[x] < nwg && s.running[x] < l.resident && (!in_order || s.next[x] == s.started)) {
            s.live.push_back(s.next[x]);
            s.next[x] += t.num_xcd;
            ++s.running[x];
            ++s.started;
            any = moved = true;
          }
      }
      std::vector<int> still;
      for (int wg : s.live) {
        bool waits = false;
        while (!waits && s.at[wg] < (int)l.chain[wg].size()) {
          const int tile = l.chain[wg][s.at[wg]], m0 = tile / tiles_n * t.tile_m, n0 = tile % tiles_n * t.tile_n;
          const int m1 = std::min(m0 + t.tile_m, t.M), n1 = std::min(n0 + t.tile_n, t.N);
          for (int fm = m0 / t.flag_bm; fm <= (m1 - 1) / t.flag_bm; ++fm)
            for (int fn = n0 / t.flag_bn; fn <= (n1 - 1) / t.flag_bn; ++fn) {
              const int f = fm * ftn + fn;
              if (!s.told[wg]) ++s.published[f], moved = true;
              const int owner = t.epi == EPI_TWO_SHOT ? owner_interleaved(f, t.world) : t.epi == EPI_REDUCE_SCATTER ? owner_contiguous(f, ftm * ftn, t.world) : t.rank;
              if (owner != t.rank && !t.all_owners) continue;
              for (size_t peer = 0; peer < ranks.size(); ++peer) waits |= peer != r && st[peer].published[f] < st[peer].needed[f];
            }
          s.told[wg] = 1;
          if (waits) break;
          s.told[wg] = 0;
          ++s.at[wg];
          moved = true;
        }
        if (waits) {
          still.push_back(wg);
        } else {
          --s.running[wg % t.num_xcd];
          --left;
        }
      }
      s.live = still;
    }
  }
  return left;
}

TileLaunch launch_of(int epi, int M, int N, int tile_m, int tile_n, int two_per_cu, int world, int rank, int flag_bm, int flag_bn) {
  return {M, N, tile_m, tile_n, 8, 32 * (1 + two_per_cu), two_per_cu, epi, world, rank, 1, 0, flag_bm, flag_bn};
}

// Launches of several rounds end on every rank, whatever they wait for.
void check_ranks_finish() {
  struct Case { int epi, M, N, tile_m, tile_n, two_per_cu, world, flag_bm, flag_bn; };
  for (Case c : {Case{EPI_REDUCE_SCATTER, 8192, 4096, 256, 256, 0, 2, 256, 64}, Case{EPI_REDUCE_SCATTER, 8192, 4096, 256, 256, 0, 4, 256, 64},
                 Case{EPI_REDUCE_SCATTER, 8192, 4096, 256, 256, 0, 8, 256, 64}, Case{EPI_REDUCE_SCATTER, 8001, 4095, 256, 256, 0, 2, 256, 64},
                 Case{EPI_REDUCE_SCATTER, 8192, 4097, 256, 256, 0, 2, 256, 64}, Case{EPI_REDUCE_SCATTER, 16383, 4093, 256, 256, 0, 4, 256, 64},
                 Case{EPI_REDUCE_SCATTER, 16383, 8191, 256, 256, 0, 8, 128, 64}, Case{EPI_REDUCE_SCATTER, 16384, 8192, 256, 256, 0, 2, 96, 80},
                 Case{EPI_REDUCE_SCATTER, 8192, 1024, 128, 128, 1, 2, 64, 64}, Case{EPI_REDUCE_SCATTER, 16384, 256, 128, 128, 1, 3, 128, 64},
                 Case{EPI_REDUCE_SCATTER, 3128, 7162, 256, 256, 0, 4, 256, 64},
                 Case{EPI_REDUCE_SCATTER, 16384, 2048, 256, 256, 0, 8, 8192, 64}, Case{EPI_REDUCE_SCATTER, 8192, 8192, 256, 256, 0, 8, 4096, 4096},
                 Case{EPI_ONE_SHOT, 16384, 8192, 256, 256, 0, 8, 256, 64}, Case{EPI_ONE_SHOT, 8191, 4097, 256, 256, 0, 2, 96, 80},
                 Case{EPI_TWO_SHOT, 16384, 4096, 256, 256, 0, 8, 256, 64}, Case{EPI_TWO_SHOT, 8191, 4097, 256, 256, 0, 2, 96, 80}})
    for (bool in_order : {false, true}) {
      std::vector<RankLaunch> ranks;
      for (int r = 0; r < c.world; ++r) ranks.push_back(tiled_launch(launch_of(c.epi, c.M, c.N, c.tile_m, c.tile_n, c.two_per_cu, c.world, r, c.flag_bm, c.flag_bn)));
      const int left = replay(ranks, in_order);
      CHECK(left == 0, "%d workgroups wait for ever: epilogue %d of %d ranks, %dx%d, tiles %dx%d, flag tiles %dx%d", left, c.epi, c.world, c.M, c.N, c.tile_m, c.tile_n, c.flag_bm, c.flag_bn);
    }
  // Some ranks multiply packed operands, the others had no memory for them.
  struct Tile { int m, n, resident; };
  for (Tile any : {Tile{256, 256, 32}, Tile{128, 128, 64}, Tile{64, 128, 64}, Tile{64, 64, 64}})
  for (Case c : {Case{EPI_TWO_SHOT, 16001, 4097, 256, 256, 0, 2, 256, 64}, Case{EPI_ONE_SHOT, 16001, 4097, 256, 256, 0, 3, 256, 64},
                 Case{EPI_ONE_SHOT, 4001, 2877, 256, 256, 0, 8, 256, 64}, Case{EPI_TWO_SHOT, 1999, 2877, 128, 128, 1, 4, 128, 64},
                 Case{EPI_REDUCE_SCATTER, 8001, 4095, 256, 256, 0, 2, 256, 64}, Case{EPI_REDUCE_SCATTER, 8001, 4095, 256, 256, 0, 4, 256, 64},
                 Case{EPI_REDUCE_SCATTER, 16383, 8191, 256, 256, 0, 8, 128, 64}, Case{EPI_REDUCE_SCATTER, 4001, 2877, 256, 256, 0, 8, 256, 64}})
    for (int memory = 0; memory < 1 << c.world; memory += c.world > 4 ? 37 : 1) {
      std::vector<RankLaunch> ranks;
      for (int r = 0; r < c.world; ++r)
        ranks.push_back(packed_launch(launch_of(c.epi, c.M, c.N, c.tile_m, c.tile_n, c.two_per_cu, c.world, r, c.flag_bm, c.flag_bn), memory >> r & 1, any.m, any.n, any.resident));
      const int left = replay(ranks, false);
      CHECK(left == 0, "%d workgroups wait for ever: epilogue %d of %d ranks, %dx%d, tiles %dx%d, packed on ranks %x, else %dx%d", left, c.epi, c.world, c.M, c.N, c.tile_m, c.tile_n, memory, any.m, any.n);
    }
  // A rank starts with its own band of rows while that leaves room for the others.
  CHECK(tile_order(launch_of(EPI_REDUCE_SCATTER, 8192, 4096, 256, 256, 0, 8, 3, 256, 64)).tile_rotate == 12 * 16, "reduce-scatter of eight ranks starts with its band");
  CHECK(tile_order(launch_of(EPI_REDUCE_SCATTER, 8192, 4096, 256, 256, 0, 2, 1, 256, 64)).tile_rotate == 0, "reduce-scatter of two ranks: the same order on both");
  CHECK(tile_order(launch_of(EPI_REDUCE_SCATTER, 3128, 7162, 256, 256, 0, 4, 3, 256, 64)).tile_rotate == 8 * 28, "the last of four ranks starts with its 140 tiles");
}

// ---- vote of a workgroup in a loop with one barrier per step -----------------------------------------
// A wave meets the first reason to leave in step `seen`.  Reads behind the barrier of step s may come as early as right
// behind it or as late as right in front of the next one, when votes written in step s + 1 are there too: both have to
// leave the loop in the same step, and before long.
void check_vote() {
  for (int nsteps = 1; nsteps <= 40; ++nsteps)
    for (int seen = 0; seen < nsteps; ++seen) {
      auto leaves = [&](bool late) {
        for (int s = 0; s < nsteps; ++s) {
          if (!vote_read_behind_barrier(s)) continue;
          for (int w = seen; w <= s + (late && s + 1 < nsteps); ++w)
            if (vote_written_before_barrier(w)) return s;
        }
        return nsteps;
      };
      CHECK(leaves(false) == leaves(true), "%d steps, reason met in step %d: early readers leave in step %d, late ones in step %d", nsteps, seen, leaves(false), leaves(true));
      CHECK(leaves(false) <= seen + 8 || leaves(false) == nsteps, "%d steps, reason met in step %d: left in step %d", nsteps, seen, leaves(false));
    }
}

int main() {
  check_row_tile<64>(256);
  check_row_tile<128>(256);
  check_row_tile<256>(64);
  check_col_tile<512, 2>(32);
  check_col_tile<256, 2>(32);
  check_col_tile<256, 1>(64);
  check_col_tile<128, 1>(64);
  sim_row_operand<64, 2>(256, 8);   // bf16/fp16 A tile 256 x 32
  sim_row_operand<64, 2>(128, 4);
  sim_row_operand<64, 1>(256, 8);   // fp8 A tile 256 x 64
  sim_col_operand<512, 2>(32);      // bf16 B tile 32 x 256
  sim_col_operand<256, 2>(32);      // bf16 B tile 32 x 128
  sim_col_operand<256, 1>(64);      // fp8 B tile 64 x 256
  sim_col_operand<128, 1>(64);      // fp8 B tile 64 x 128
  check_acc_layout();
  check_col_tile16<512>(32);
  check_col_tile16<256>(64);
  check_col_tile16<128>(64);
  sim_row_operand16<64>(256);
  sim_row_operand16<128>(128);
  sim_col_operand16<512>(32);
  sim_col_operand16<256>(64);
  sim_col_operand16<128>(64);
  check_acc_layout16();
  check_quad_blocks<8, 4>();
  check_quad_blocks<4, 2>();
  check_tile_orders();
  check_dealt_order();
  check_flag_counts();
  check_rect_pieces();
  check_decode_offsets();
  check_split_plan();
  check_row_rects();
  check_vote();
  check_ranks_finish();
  if (failures) { printf("%d check(s) failed\n", failures); return 1; }
  printf("layout_sim: all checks passed\n");
  return 0;
}
