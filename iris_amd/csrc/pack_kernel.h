// pack_kernel: operands whose rows start anywhere, laid out once per launch as whole 16-byte pieces (the K of every source padded
// with zeros), so that the direct-to-LDS loads of fused_mfma_kernel can fetch them.
//
// The any-shape kernel fetches such rows through registers, every tile again: 16-byte loads that straddle lines, LDS writes
// and a barrier chain per K step.  With more than a few tiles to a row or column of the output one pass over the
// operands costs less than that (which launches: worth_packing in iris_hip.hip).  It is bound by memory: one 16-byte load and
// one 16-byte store per piece, two of each in flight per thread.
#pragma once

#include "fused_params.h"

// One operand: rows of `segments` runs of elements.  Gathered along K, a row of A has a run per source slot.
struct PackJob {
  const char* src;
  char* dst;
  long long src_row;      // bytes from row to row
  long long src_segment;  // ... and from run to run, where they lie in one slot
  int rows;               // rows written
  int segments;
  int run, run_pieces;    // elements of a run that exist, 16-byte pieces of it written (the rest of them is zero)
  int row_period, row_run;  // of every row_period rows written the first row_run exist (B's rows, K of several sources)
  int slots_of_rows;      // != 0: rows come from the slots, so many from each
  int slots_of_segments;  // != 0: run i comes from slot i
};

struct PackParams {
  PackJob job[2];
  int blocks[2];  // workgroups of each job (0: nothing to do)
  const long long* heap_bases;
  int rank;
};

constexpr int kPackThreads = 256, kPackPieces = 2;  // per workgroup, per thread

template <int ES>
__global__ void __launch_bounds__(kPackThreads) pack_kernel(const PackParams q) {
  constexpr int CE = kChunkBytes / ES;
  const bool second = (int)blockIdx.x >= q.blocks[0];
  const PackJob& j = q.job[second];
  const unsigned block = blockIdx.x - (second ? q.blocks[0] : 0);
  const unsigned per_row = (unsigned)j.segments * j.run_pieces, total = per_row * j.rows;
  const bool short_run = j.run < CE;
  u32x4_t v[kPackPieces];
  int shift[kPackPieces];  // elements to drop from the front: the last piece of a run is loaded from further left
#pragma unroll
  for (int u = 0; u < kPackPieces; ++u) {
    const unsigned i = (block * kPackPieces + u) * kPackThreads + threadIdx.x;
    v[u] = (u32x4_t){0u, 0u, 0u, 0u};
    shift[u] = 0;
    if (i >= total) continue;
    unsigned row = i / per_row;
    const unsigned c = i - row * per_row;
    const unsigned segment = j.segments > 1 ? c / j.run_pieces : 0, at = (c - segment * j.run_pieces) * CE;
    if (j.row_period) {
      const unsigned period = row / j.row_period, in = row - period * j.row_period;
      if (in >= (unsigned)j.row_run) continue;
      row = period * j.row_run + in;
    }
    const char* base = j.src;
    if (j.slots_of_rows) {
      const unsigned slot = row / j.slots_of_rows;
      row -= slot * j.slots_of_rows;
      base = slot_ptr(q.heap_bases, base, q.rank, slot);
    }
    if (j.slots_of_segments) base = slot_ptr(q.heap_bases, base, q.rank, segment);
    else base += segment * j.src_segment;
    base += row * j.src_row;
    if (at >= (unsigned)j.run) continue;
    if (short_run) {
#pragma unroll
      for (int e = 0; e < CE; ++e)
        if (e < j.run) {
          unsigned x;
          if constexpr (ES == 2) x = *(const GLOBAL_AS unsigned short*)(GLOBAL_AS const char*)(base + e * ES);
          else x = *(const GLOBAL_AS unsigned char*)(GLOBAL_AS const char*)(base + e);
          v[u][e * ES / 4] |= x << (8 * (e * ES % 4));
        }
    } else {
      const int from = min((int)at, j.run - CE);
      shift[u] = (int)at - from;
      v[u] = load16_any(base + (long long)from * ES);
    }
  }
#pragma unroll
  for (int u = 0; u < kPackPieces; ++u) {
    const unsigned i = (block * kPackPieces + u) * kPackThreads + threadIdx.x;
    if (i >= total) continue;
    if (shift[u]) {  // zeros follow behind the run
      const int bits = shift[u] * ES * 8;
      unsigned long long lo = v[u][0] | (unsigned long long)v[u][1] << 32, hi = v[u][2] | (unsigned long long)v[u][3] << 32;
      if (bits >= 64) {
        lo = hi >> (bits - 64);
        hi = 0;
      } else {
        lo = lo >> bits | hi << (64 - bits);
        hi >>= bits;
      }
      v[u] = (u32x4_t){(unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32)};
    }
    *(u32x4_t*)(j.dst + (long long)i * kChunkBytes) = v[u];
  }
}
