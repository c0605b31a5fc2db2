// What the kernels of the fused operators share: their arguments (FusedParams), the phase stamps of the diagnostic build, and the
// flags of the tiles.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <type_traits>

#include "iris_hip.h"
#include "layout.h"
#include "device_util.h"
#include "host_common.h"

using namespace iris_layout;

#define LDS_AS __attribute__((address_space(3)))

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) int i32x2_t;
typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(8))) int i32x8_t;
typedef __attribute__((ext_vector_type(4))) short i16x4_t;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2_t;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4_t;

enum { GATHER_NONE = 0, GATHER_K = 1, GATHER_M = 2 };

struct FusedParams {
  const char* A;
  const char* B;
  char* C;
  char* aux;
  int* locks;
  const char* bias;
  int M, N, K;
  int K_local;  // K extent held by one source slot (== K unless gathered along K)
  int M_local;  // rows held by one source slot when gathered along M
  int gather;
  long long s_am, s_ak, s_bk, s_bn, s_cm, s_cn, s_bias;  // element strides
  const long long* heap_bases;
  int rank, world;
  int flag_bm, flag_bn;
  int epi;
  int acc_mode;
  int clear_c;  // IRIS_HIP_CLEAR_C: the own slot's C ends up as if it had been zeroed before the launch
  int all_owners;
  int sum_peers;
  int bias_dtype;
  float scale;
  long long spin_limit;
  int* status;
  int tiles_m, tiles_n, group_m, num_xcd;
  // Tile order: 0 gives every XCD one contiguous span of the grouped order (tiles that share operand
  // panels share an L2), 1 deals the grouped order out workgroup by workgroup (the chip works on one
  // contiguous band of rows at a time; launches that stream the peers' tiles, see tile_order in layout.h).
  int interleave;
  int tile_rotate;  // with interleave: the workgroups start this many positions into the grouped order (and wrap)
  int group_m_spans;  // host only: the group height to use if the launch falls back to spans (split tiles)
  int row_offset;  // all-gather: first row of this rank's block in the gathered output
  // Heap bases as kernel arguments (slots 0..7), valid when hb_in_args is set: the host knew the contents
  // of the context tensor (iris_hip_register_context), which spares the kernels a dependent scalar load
  // on the way to the peers' flags and tiles.
  long long hb_arg[8];
  int hb_in_args;
  // Split tiles (see the STREAMK builds of fused_mfma_kernel): one slot of partial sums and one flag per
  // workgroup, and the value a flag takes in this launch.  NULL / 0 when the launch does not split tiles.
  char* sk_partials;
  int* sk_flags;
  int sk_epoch;
  int sk_gather_cost, sk_pass_cost;  // the costs the host planned the split with (iris_layout::split_plan)
  int no_workspace_alloc;  // host only: the caller must not trigger an allocation (split tiles need one)
  // (Behind the arguments of the small kernel, which is 1 % slower with anything in between.)
  int whole_lines;   // rows of C and aux start and end with 128-byte lines (see store16_system_nt)
  // The peers' tiles are read past the caches (peers_past_caches in iris_hip.hip).  The tiled kernel with other numbers of ranks than 2,
  // 4 and 8 always does, the any-shape kernel's 32x32 tile does only with such.
  int stream_peers;
#ifdef IRIS_HIP_PHASE_STAMPS
  unsigned long long* stamps;  // diagnostic build: rows of 16 time stamps (see PHASE_STAMP)
  long long stamp_rows;        // rows the buffer holds; rows beyond it are not written
#endif
};

// Diagnostic build (-DIRIS_HIP_PHASE_STAMPS): thread 0 of every workgroup records the constant-rate
// 100 MHz counter at the phase boundaries of its first eight tiles, into row it * gridDim.x + blockIdx.x
// of p.stamps (16 slots per row, slot i):
//   0 kernel entry, 1 first operands in LDS, 2 K loop done, 3 tile staged in LDS, 4 phase-1 stores
//   issued, 5 phase-1 stores acknowledged, 6 own flags raised and peers' flags seen, 7 phase-2 stores
//   issued, 8 last store acknowledged.  The regular build compiles the macro away.
#ifdef IRIS_HIP_PHASE_STAMPS
#define PHASE_STAMP(i)                                                                         \
  do {                                                                                         \
    if (p.stamps && threadIdx.x == 0 && it < 8 && (long long)it * gridDim.x + blockIdx.x < p.stamp_rows)     \
      p.stamps[((long long)it * gridDim.x + blockIdx.x) * 16 + (i)] = wall_clock64();                       \
  } while (0)
#else
#define PHASE_STAMP(i) \
  do {                 \
  } while (0)
#endif

// ------------------------------------------------------------------------------------------------
// Small device helpers
// ------------------------------------------------------------------------------------------------

__device__ __forceinline__ int owner_of(int epi, int t, int total, int world, int rank) {
  if (epi == EPI_TWO_SHOT) return owner_interleaved(t, world);
  if (epi == EPI_REDUCE_SCATTER) return owner_contiguous(t, total, world);
  return rank;
}

// Raise the flags of the flag tiles covered by the macro tile at (m0, n0) of KM x KN elements.
// Must be called by every thread of the workgroup after the workgroup's aux stores have completed
// (vmcnt(0)) and a workgroup barrier.
// WRITTEN_THROUGH = false: the aux stores were ordinary stores (dirty lines in L2), so the flag is
//   raised with system-scope release, which writes the L2 back first.
// WRITTEN_THROUGH = true: the aux stores were system-scope write-through stores (store16_system) that
//   have been acknowledged, so the data is already where a peer reads it and a relaxed system-scope
//   flag store after them is enough; this spares one whole-L2 write-back per workgroup (measured 5-11 %
//   of the fused launch).
template <int KM, int KN, int NT, bool WRITTEN_THROUGH>
__device__ __forceinline__ void raise_flags(const FusedParams& p, int m0, int n0, int tid) {
  const int m1 = min(m0 + KM, p.M), n1 = min(n0 + KN, p.N);
  const int ftn = cdiv(p.N, p.flag_bn);
  const int fm_lo = m0 / p.flag_bm, fm_hi = (m1 - 1) / p.flag_bm;
  const int fn_lo = n0 / p.flag_bn, fn_hi = (n1 - 1) / p.flag_bn;
  const int nfn = fn_hi - fn_lo + 1;
  const int nft = (fm_hi - fm_lo + 1) * nfn;
  for (int i = tid; i < nft; i += NT) {
    const int fm = fm_lo + i / nfn, fn = fn_lo + i % nfn;
    int* flag = p.locks + (fm * ftn + fn);
    const int needed = macro_tiles_over_flag_tile(fm, fn, p.flag_bm, p.flag_bn, KM, KN, p.M, p.N);
    bool last = true;
    if (needed > 1) {
      // Arrivals are counted in steps of 2 so that the flag never reads 1 before the last one.
      int old = WRITTEN_THROUGH ? __hip_atomic_fetch_add(flag, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM)
                                : __hip_atomic_fetch_add(flag, 2, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_SYSTEM);
      last = ((old >> 1) + 1) == needed;
    }
    if (last) {
      if (WRITTEN_THROUGH) __hip_atomic_exchange(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      else __hip_atomic_exchange(flag, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// Wait until the peers' flags of every flag tile this workgroup reduces are 1.
template <int KM, int KN, int NT>
__device__ __forceinline__ void wait_peer_flags(const FusedParams& p, int m0, int n0, int tid) {
  const int m1 = min(m0 + KM, p.M), n1 = min(n0 + KN, p.N);
  const int ftn = cdiv(p.N, p.flag_bn);
  const int ftotal = cdiv(p.M, p.flag_bm) * ftn;
  const int fm_lo = m0 / p.flag_bm, fm_hi = (m1 - 1) / p.flag_bm;
  const int fn_lo = n0 / p.flag_bn, fn_hi = (n1 - 1) / p.flag_bn;
  const int nfn = fn_hi - fn_lo + 1;
  const int nft = (fm_hi - fm_lo + 1) * nfn;
  const int items = nft * p.world;
  bool waited = false;
  for (int i = tid; i < items; i += NT) {
    const int r = i % p.world;
    const int f = i / p.world;
    if (r == p.rank) continue;
    const int t = (fm_lo + f / nfn) * ftn + fn_lo + f % nfn;
    if (!p.all_owners && owner_of(p.epi, t, ftotal, p.world, p.rank) != p.rank) continue;
    const int* flag = (const int*)slot_ptr(p.heap_bases, p.locks + t, p.rank, r);
    // Relaxed system-scope polls (they bypass the caches) and one acquire fence once the flag is up: an
    // acquire per poll would invalidate the XCD's L2 on every turn of the wait, under the feet of every
    // workgroup that is still multiplying or storing.
    long long polls = 0;
    while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) != 1) {
      if (p.spin_limit > 0 && ++polls >= p.spin_limit) {
        // A plain system-scope store (one status code, every writer stores the same word): the word
        // may live in pinned host memory.
        if (p.status) __hip_atomic_store(p.status, IRIS_HIP_STATUS_SPIN_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
    waited = true;
  }
  if (waited) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
}

// One look at the peers' flags that wait_peer_flags would wait for, without waiting: true when
// every flag this thread looked at was already 1, in which case the thread has also passed an
// acquire fence at system scope.  A workgroup barrier must follow before anybody reads the peers' data.
template <int KM, int KN, int NT>
__device__ __forceinline__ bool probe_peer_flags(const FusedParams& p, int m0, int n0, int tid) {
  const int m1 = min(m0 + KM, p.M), n1 = min(n0 + KN, p.N);
  const int ftn = cdiv(p.N, p.flag_bn);
  const int ftotal = cdiv(p.M, p.flag_bm) * ftn;
  const int fm_lo = m0 / p.flag_bm, fm_hi = (m1 - 1) / p.flag_bm;
  const int fn_lo = n0 / p.flag_bn, fn_hi = (n1 - 1) / p.flag_bn;
  const int nfn = fn_hi - fn_lo + 1;
  const int nft = (fm_hi - fm_lo + 1) * nfn;
  const int items = nft * p.world;
  bool up = true, looked = false;
  for (int i = tid; i < items; i += NT) {
    const int r = i % p.world;
    const int f = i / p.world;
    if (r == p.rank) continue;
    const int t = (fm_lo + f / nfn) * ftn + fn_lo + f % nfn;
    if (!p.all_owners && owner_of(p.epi, t, ftotal, p.world, p.rank) != p.rank) continue;
    const int* flag = (const int*)slot_ptr(p.heap_bases, p.locks + t, p.rank, r);
    up = up && (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM) == 1);
    looked = true;
  }
  // Only the threads that looked at a flag invalidate the caches (as only the polling threads do in
  // wait_peer_flags): the caches are the compute unit's, and an invalidation per wave of every
  // workgroup costs more than the probe saves.
  if (looked && up) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
  return up;
}

// s_waitcnt vmcnt(n) with the other counters left unconstrained (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// 16-byte store that is written through to memory at system scope (sc0 sc1): once vmcnt reports it
// done, every agent that reads the address with a coherent load sees it, without an L2 write-back.
__device__ __forceinline__ void store16_system(char* p, u32x4_t v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1" : : "v"(p), "v"(v) : "memory");
}

// The same for rows that are whole lines, past the caches' keep policy as well: own tiles on their way to the peers do not push
// everything else out of the last-level cache (bf16, eight ranks, six workspaces in turn: reduce-scatter 8192x4096x1376
// 118.6 -> 104.9 us, two-shot 8192x4096x1376 126.6 -> 112.2; with one workspace, which the cache holds, 103.4 -> 104.4 and 107 ->
// 111).  It is done at every size: launches whose slots the cache holds lose 0 to 2 % by it with one or two workspaces in turn and gain 4
// to 20 % with six (two-shot 2048x4096x512 31.2 -> 26.1 us, 4096x4096x1376 of four ranks 66.5 -> 61.0, reduce-scatter 2048x4096x1376
// 42.9 -> 38.8).  A line that two workgroups write in parts does better in the cache (2000x2896x1376 51.2 us, this way 53.8).
__device__ __forceinline__ void store16_system_nt(char* p, u32x4_t v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1 nt" : : "v"(p), "v"(v) : "memory");
}

// store16_system for data that the next instructions overwrite with VALU results (accumulator reads, say):
// a store of more than 8 bytes is still fetching its data registers for the last lanes when the next
// instruction issues, and a VALU write to them in that slot reaches memory for those lanes.  The
// compiler pads this hazard between instructions it can see; it cannot see into the asm statement, so
// the wait states are part of it.
__device__ __forceinline__ void store16_system_of_valu_data(char* p, u32x4_t v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
}

typedef u32x4_t u32x4_any_t __attribute__((aligned(1)));  // 16 bytes at any address
#define GLOBAL_AS __attribute__((address_space(1)))
// (Addresses computed from heap bases are integers to the compiler: without the address space it emits flat
// accesses, which also wait on, and are waited for with, the LDS counter.)
__device__ __forceinline__ u32x4_t load16_any(const char* p) { return *(const GLOBAL_AS u32x4_any_t*)(GLOBAL_AS const char*)p; }
__device__ __forceinline__ u32x4_t load16_any_nt(const char* p) {
  return __builtin_nontemporal_load((const GLOBAL_AS u32x4_any_t*)(GLOBAL_AS const char*)p);
}

// Around the loads on one side of a branch: the compiler takes loads that both sides make for one, and drops the cache policy that
// only one of them has.
#define KEEP_BRANCHES_APART() asm volatile("" ::: "memory")

constexpr int kMaxCachedSlots = 8;  // heap bases kept in registers; larger worlds re-load them

// A 64-bit value that is the same in every lane, moved to scalar registers.
__device__ __forceinline__ unsigned long long uniform64(unsigned long long x) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)x), hi = __builtin_amdgcn_readfirstlane((unsigned)(x >> 32));
  return ((unsigned long long)hi << 32) | lo;
}
