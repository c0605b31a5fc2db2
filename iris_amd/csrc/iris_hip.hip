// libiris_hip: gfx950 (MI355X) kernels for the rank-local compute of the fused GEMM+collective
// operators, and the C ABI declared in include/iris_hip.h.
//
// Two kernels implement every operator (the first lives in fused_kernel.h and is compiled in the
// iris_hip_mfma_<type>.hip translation units; small outputs have one of their own, decode_kernel.h; the entry points are in this file):
//
//  * fused_mfma_kernel  - persistent tiled GEMM on the matrix cores of CDNA4 (16x16 products of 16-bit data on the
//    256x256 tile, 32x32 products otherwise).  Operand tiles travel HBM -> LDS with 16-byte direct-to-LDS buffer
//    loads into a ring of STAGES buffers (four-wave tiles: STAGES-1 K steps in flight, one workgroup barrier per
//    step; the eight-wave tile, whose wave groups run half a step apart: two or three, and two barriers); the K-contiguous operand is
//    read back with 16-byte LDS reads, the N-contiguous one with LDS transpose reads.  The waves of
//    a workgroup (8 as 2x4 for the 256x256 tile, 4 as 2x2 for the smaller ones) each own a block of
//    fp32 accumulators that stays in the accumulation registers.  Requires 16-byte aligned,
//    unit-stride rows (see mfma_ineligible()).
//  * fused_any_kernel (any_kernel.h, compiled in the iris_hip_any_<type>.hip translation units) - any alignment,
//    stride, size and element type, operands through registers: everything the first does not take (fp32
//    data, odd strides, sizes that are not multiples of 8 elements) - unless it is large enough that the first is
//    ahead behind one pass that lays the operands out anew (pack_kernel.h, iris_hip_rows_<type>.hip; worth_packing below).
//
// The flag-less operators (all_gather_matmul, matmul_all_gather, the atomic all-reduce) store or add
// the tile directly.  The others end in the same epilogue protocol, which follows the reference kernels
// (iris/ops/matmul_all_reduce.py:111-144, iris/ops/matmul_reduce_scatter.py:98-118,
//  iris/mem/triton/context.py:733-764, 801-839, 953-997):
//    1. cast the fp32 tile to the output type and store it to aux in the own slot,
//    2. make those stores visible (aux is written through to memory), then raise the flag of every finished
//       flag tile,
//    3. for the flag tiles this rank reduces: wait for the peers' flags, add the peers' aux tiles
//       in ascending rank order, cast once, store to C (own slot; two-shot: every slot).

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include "any_kernel.h"
#include "fused_kernel.h"
#include "pack_kernel.h"

// ------------------------------------------------------------------------------------------------
// Host side
// ------------------------------------------------------------------------------------------------
namespace {

thread_local char g_last_error[512] = "";
thread_local char g_last_kernel[128] = "";

using iris_host::fail;  // defined below, shared with the other translation units

// Device memory for the length of a launch, from the caller's allocator (iris_hip_set_scratch_allocator).
struct ScratchAllocator {
  std::atomic<iris_hip_allocate_fn> allocate{nullptr};
  std::atomic<iris_hip_release_fn> release{nullptr};
  // NULL: there is none, none is left, or the stream is being captured (what a graph holds has to outlive the call).
  void* take(size_t bytes, hipStream_t stream) const {
    const iris_hip_allocate_fn f = allocate.load(std::memory_order_acquire);
    if (!f) return nullptr;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      return nullptr;
    }
    return f(bytes, (void*)stream);
  }
  void give_back(void* memory) const {
    if (memory) release.load(std::memory_order_acquire)(memory);
  }
};

struct DeviceFacts {
  int cu_count = 0;
  int xcc_count = 0;
  int lds_per_block = 0;
  bool ok = false;
};

DeviceFacts g_facts[64];
std::mutex g_facts_mutex;  // entry points may be called from several host threads

int facts_for(int device, DeviceFacts** out) {
  if (device < 0 || device >= 64) return fail("device index %d out of range", device);
  std::lock_guard<std::mutex> lock(g_facts_mutex);
  DeviceFacts& f = g_facts[device];
  if (!f.ok) {
    hipDeviceProp_t prop;
    hipError_t e = hipGetDeviceProperties(&prop, device);
    if (e != hipSuccess) return (int)e;
    f.cu_count = prop.multiProcessorCount;
    f.lds_per_block = (int)prop.sharedMemPerBlock;
    // XCD count as the runtime reports it (the reference asks the same attribute,
    // iris/host/platform/hip.py:218-231); a runtime that does not know the attribute means one XCD.
    int xcc = 0;
    if (hipDeviceGetAttribute(&xcc, hipDeviceAttributeNumberOfXccs, device) != hipSuccess || xcc < 1) {
      (void)hipGetLastError();
      xcc = 1;
    }
    f.xcc_count = xcc;
    f.ok = true;
  }
  *out = &f;
  return 0;
}

int elem_size(int dtype) {
  switch (dtype) {
    case IRIS_HIP_BF16: case IRIS_HIP_FP16: return 2;
    case IRIS_HIP_FP32: return 4;
    case IRIS_HIP_FP8_E4M3: return 1;
  }
  return 0;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Reasons (if any) the MFMA kernel cannot take these operands.
const char* mfma_ineligible(const FusedParams& p, int in_dtype, int out_dtype, int bm, int bn) {
  if (in_dtype == IRIS_HIP_FP32) return "fp32 inputs";
  const int es = elem_size(in_dtype);
  const int ce = 16 / es;
  const int want_out = (in_dtype == IRIS_HIP_FP16) ? IRIS_HIP_FP16 : IRIS_HIP_BF16;
  if (out_dtype != want_out) return "output type not paired with the input type";
  if (p.s_ak != 1) return "A is not K-contiguous";
  if (p.s_bn != 1 && p.s_bk != 1) return "B has no unit stride";
  if (p.s_cn != 1) return "C is not N-contiguous";
  if (!aligned16(p.A) || !aligned16(p.B) || !aligned16(p.C)) return "base pointers not 16-byte aligned";
  if (p.aux && !aligned16(p.aux)) return "aux not 16-byte aligned";
  if (p.K % ce || p.K_local % ce) return "K not a multiple of 16 bytes";
  if ((p.s_am * es) % 16) return "A rows not 16-byte aligned";
  if (p.s_bn == 1) {
    if (p.N % ce) return "N not a multiple of 16 bytes of B";
    if ((p.s_bk * es) % 16) return "B rows not 16-byte aligned";
  } else {
    if ((p.s_bn * es) % 16) return "B columns not 16-byte aligned";
  }
  if (p.N % 8 || p.s_cm % 8) return "C rows not 16-byte aligned";
  if (p.flag_bn % 8) return "flag tile width not a multiple of 8";
  // 32-bit buffer offsets: per-lane offset + per-step offset must stay below 2^31.
  const long long a_span = (long long)bm * p.s_am * es + (long long)p.K * es;
  const long long b_span = (p.s_bn == 1) ? (long long)p.K * p.s_bk * es + (long long)bn * es
                                         : (long long)bn * p.s_bn * es + (long long)p.K * es;
  if (a_span >= (1ll << 31) || b_span >= (1ll << 31)) return "operand too large for 32-bit tile offsets";
  if (p.gather == GATHER_M && (p.M_local % bm)) return "M_local not a multiple of the tile height";
  return nullptr;
}

// Type pairs the any-shape kernel is built for (the list of dispatch_generic below).
bool generic_supported(int in_dtype, int out_dtype) {
  switch (in_dtype) {
    case IRIS_HIP_BF16: return out_dtype == IRIS_HIP_BF16 || out_dtype == IRIS_HIP_FP32;
    case IRIS_HIP_FP16: return out_dtype == IRIS_HIP_FP16 || out_dtype == IRIS_HIP_FP32;
    case IRIS_HIP_FP32: return out_dtype == IRIS_HIP_FP32;
    case IRIS_HIP_FP8_E4M3: return out_dtype == IRIS_HIP_BF16 || out_dtype == IRIS_HIP_FP16;
  }
  return false;
}

}  // namespace

// Instantiated in iris_hip_mfma_bf16.hip, iris_hip_mfma_f16.hip and iris_hip_mfma_fp8.hip.
extern template int dispatch_mfma_in<IN_BF16>(FusedParams&, int, bool, int, int, hipStream_t);
extern template int dispatch_mfma_in<IN_F16>(FusedParams&, int, bool, int, int, hipStream_t);
extern template int dispatch_mfma_in<IN_FP8>(FusedParams&, int, bool, int, int, hipStream_t);
// Instantiated in iris_hip_rows_<type>.hip.
extern template int dispatch_mfma_rows<IN_BF16>(const FusedParams&, int, bool, int, hipStream_t);
extern template int dispatch_mfma_rows<IN_F16>(const FusedParams&, int, bool, int, hipStream_t);
extern template int dispatch_mfma_rows<IN_FP8>(const FusedParams&, int, bool, int, hipStream_t);
// Instantiated in iris_hip_any_<type>.hip.
extern template int dispatch_any<IN_BF16, ElemBF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_BF16, ElemF32>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_F16, ElemF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_F16, ElemF32>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_F32, ElemF32>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_FP8, ElemBF16>(const FusedParams&, int, int, hipStream_t, const char*, int);
extern template int dispatch_any<IN_FP8, ElemF16>(const FusedParams&, int, int, hipStream_t, const char*, int);

namespace {

int dispatch_generic(const FusedParams& p, int in_dtype, int out_dtype, int device, int cu, hipStream_t s, int tile = -1) {
  const bool out_f32 = out_dtype == IRIS_HIP_FP32;
  switch (in_dtype) {
    case IRIS_HIP_BF16:
      return out_f32 ? dispatch_any<IN_BF16, ElemF32>(p, device, cu, s, "bf16_f32", tile) : dispatch_any<IN_BF16, ElemBF16>(p, device, cu, s, "bf16", tile);
    case IRIS_HIP_FP16:
      return out_f32 ? dispatch_any<IN_F16, ElemF32>(p, device, cu, s, "f16_f32", tile) : dispatch_any<IN_F16, ElemF16>(p, device, cu, s, "f16", tile);
    case IRIS_HIP_FP32: return dispatch_any<IN_F32, ElemF32>(p, device, cu, s, "f32", tile);
    default:
      return out_dtype == IRIS_HIP_BF16 ? dispatch_any<IN_FP8, ElemBF16>(p, device, cu, s, "fp8_bf16", tile)
                                        : dispatch_any<IN_FP8, ElemF16>(p, device, cu, s, "fp8_f16", tile);
  }
}

// ------------------------------------------------------------------------------------------------
// Library-owned workspace of iris_hip_matmul_all_reduce_noalloc
// ------------------------------------------------------------------------------------------------
// Layout of the array: [0, 256) a one-rank context (rank 0, world 1, heap base 0: every address
// translates to itself), [256, 256 + 64 KiB) the tile flags, then the aux buffer.
constexpr size_t kScratchContextBytes = 256;
constexpr size_t kScratchFlagBytes = (size_t)IRIS_HIP_NOALLOC_MAX_FLAGS * sizeof(int32_t);
constexpr size_t kScratchAuxOffset = kScratchContextBytes + kScratchFlagBytes;
constexpr size_t kScratchBytes = kScratchAuxOffset + (size_t)IRIS_HIP_NOALLOC_MAX_AUX_BYTES;
static_assert(kScratchAuxOffset % 256 == 0, "aux buffer alignment");

// Device memory of its own on every GPU the library runs on, from module load to process end.  The
// name below is a host-side handle only: device code and HIP calls get the address that
// hipGetSymbolAddress reports for the current device (scratch_for_current_device).
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

void* g_scratch_ptr[64] = {};
std::mutex g_scratch_mutex;

// Address of the scratch array on the current device (looked up once per device).
int scratch_for_current_device(unsigned char** out) {
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return (int)e;
  if (device < 0 || device >= 64) return fail("device index %d out of range", device);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[device]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!ptr) return fail("the library's workspace has no address on device %d", device);
    g_scratch_ptr[device] = ptr;
  }
  *out = (unsigned char*)g_scratch_ptr[device];
  return 0;
}

// Writes the one-rank context and clears the flags a launch is going to use.  A kernel, not a memset:
// the caller's stream may be under graph capture.
__global__ void __launch_bounds__(256) noalloc_prepare_kernel(long long* context, int* flags, int nflags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (int)(kScratchContextBytes / sizeof(long long))) context[i] = (i == 1) ? 1 : 0;  // [rank 0, world 1, base 0, ...]
  if (i < nflags) flags[i] = 0;
}

// ------------------------------------------------------------------------------------------------
// Context tensors whose contents the host has told the library (iris_hip_register_context)
// ------------------------------------------------------------------------------------------------
struct KnownContext {
  const int64_t* device_ptr;
  int rank, world;
  long long bases[kMaxCachedSlots];
};
std::vector<KnownContext> g_contexts;
std::mutex g_contexts_mutex;

// Fill p.hb_arg from the registry when the launch names a registered context tensor with the same
// rank and world size (anything else falls back to loading the bases on the device).
void heap_bases_from_registry(FusedParams& p, const int64_t* context_tensor) {
  p.hb_in_args = 0;
  if (!context_tensor || p.world > kMaxCachedSlots) return;
  std::lock_guard<std::mutex> lock(g_contexts_mutex);
  for (const KnownContext& k : g_contexts) {
    if (k.device_ptr != context_tensor) continue;
    if (k.rank != p.rank || k.world != p.world) return;
    for (int r = 0; r < kMaxCachedSlots; ++r) p.hb_arg[r] = k.bases[r];
    p.hb_in_args = 1;
    return;
  }
}

#ifdef IRIS_HIP_PHASE_STAMPS
unsigned long long* g_stamps = nullptr;  // diagnostic build: where the kernels record their phase stamps
long long g_stamp_rows = 0;              // ... and how many rows of 16 words the buffer holds
#endif

// Launches for the 32x32 kernel (decode_kernel.h): outputs of at most two 32x32 tiles per CU.  Such an
// output is a handful of 128x128 tiles on a handful of CUs, while 32x32 tiles with K split over the waves
// of a workgroup keep the whole chip busy; beyond two tiles per CU the 64x64 tiled kernel is ahead.
bool decode_sized(const FusedParams& p, int cu_count, int in_dtype) {
  if ((long long)cdiv(p.M, 32) * cdiv(p.N, 32) > 2ll * cu_count) return false;
  // ... and whose operands that kernel's 32-bit offsets reach (a tall A with long or padded rows does not
  // qualify: 16384 x 32 outputs of K = 65536 bf16 have 2 GiB of A).
  const long long a_rows = p.gather == GATHER_M ? p.M_local : p.M;
  return decode_offsets_fit(a_rows, p.s_am, p.K_local, in_dtype == IRIS_HIP_FP8_E4M3 ? 1 : 2, p.M + p.row_offset, p.s_cm, p.N);
}
// ... and whose A that kernel can fetch: not gathered, gathered by rows in whole 32-row tiles per slot, or
// gathered along K with every wave's 256 bytes of K inside one slot.
bool decode_gather_ok(const FusedParams& p, int in_dtype) {
  const int es = in_dtype == IRIS_HIP_FP8_E4M3 ? 1 : 2;
  if (p.gather == GATHER_M) return p.M_local % 32 == 0;
  if (p.gather == GATHER_K) return ((long long)p.K_local * es) % 256 == 0;
  return true;
}

// Whether the slot sum reads the peers' tiles past the caches' keep policy.  Up to 32 MiB of them are read through the
// caches: the slots of such a launch, its neighbours' and their outputs fit the 256 MB last-level cache, and lines that two
// tiles share are fetched once.  What does not fit would only push the rest
// out of it, dirty lines first.  Eight ranks, us, past the caches -> through them, with two workspaces in turn (and with six): fp16 two-shot
// 896x2880x512 (5 MB read) 18.9 -> 17.3 (20.2 -> 18.8), bf16 900x2896x512 23.5 -> 19.8 (23.6 -> 20.1), reduce-scatter
// 4096x4096x1376 (29 MB) 66.8 -> 57.9 (70.0 -> 69.9), float32 two-shot 2048x2880x1024 of four ranks (18 MB) 107.7 -> 103.6;
// one-shot 1024x2880x1376 (41 MB) 29.9 -> 28.6 (30.0 -> 32.3), 4096x4096x1376 (235 MB) 84.9 -> 95.5.  (All with peers' slots that nobody
// rewrites between the calls, as one process that plays every rank leaves them; tiles that come over the links have not been measured.)
// Rows that are no whole lines go by the same line: read through the caches at every size they are 11 % faster to 5 % slower.
bool peers_past_caches(const FusedParams& p, int out_dtype) {
  const long long all = (long long)p.M * p.N * elem_size(out_dtype) * (p.world - 1);
  const long long read = p.epi == EPI_ONE_SHOT || p.all_owners ? all : all / p.world;
  return epi_has_flags(p.epi) && read > (32ll << 20);
}

// Whether every row of C and aux starts and ends with a 128-byte line.
bool rows_of_whole_lines(const FusedParams& p, int out_dtype) {
  const int es = elem_size(out_dtype);
  return p.s_cn == 1 && ((p.s_cm * es) | ((long long)p.N * es)) % 128 == 0 && (((uintptr_t)p.aux | (uintptr_t)p.C) & 127) == 0;
}

// ------------------------------------------------------------------------------------------------
// 16- and 8-bit operands whose rows start anywhere, on the direct-to-LDS kernel (pack_kernel.h)
// ------------------------------------------------------------------------------------------------
ScratchAllocator g_scratch_allocator;

// The sizes that choose among the tiled kernels (run_fused, plan_packing): enough 256x256 tiles; at most two 64x64 tiles per CU; more
// 128x128 tiles than CUs.
bool fills_big_tiles(const FusedParams& p, int cu) { return (long long)cdiv(p.M, 256) * cdiv(p.N, 256) * 100 >= (long long)cu * 53; }
bool fits_64x64_tiles(const FusedParams& p, int cu) { return (long long)cdiv(p.M, 64) * cdiv(p.N, 64) <= 2ll * cu; }
bool needs_two_128x128_tiles(const FusedParams& p, int cu) { return (long long)cdiv(p.M, 128) * cdiv(p.N, 128) > cu; }

struct PackPlan {
  FusedParams p;      // the launch on the packed operands
  PackParams pack;
  size_t bytes;       // of both packed operands
  int kind;
};

// What a launch that the MFMA kernel cannot take as it is would look like with A and B laid out anew where they have to be.
// False: it cannot be brought to that kernel this way.
bool plan_packing(const FusedParams& p, int in_dtype, int out_dtype, int cu, PackPlan& plan) {
  if (in_dtype == IRIS_HIP_FP32 || out_dtype != (in_dtype == IRIS_HIP_FP16 ? IRIS_HIP_FP16 : IRIS_HIP_BF16)) return false;
  if (p.s_ak != 1 || (p.s_bn != 1 && p.s_bk != 1) || p.s_cn != 1) return false;
  const int es = elem_size(in_dtype), ce = 16 / es;
  const bool bkc = p.s_bn != 1;
  const int sources = p.gather == GATHER_K ? p.world : 1;
  auto whole = [&](long long n) { return (n + ce - 1) / ce * ce; };

  plan.kind = TILE_SMALL;
  if (fills_big_tiles(p, cu) && p.M > 64) plan.kind = TILE_BIG;
  else if (fits_64x64_tiles(p, cu)) plan.kind = TILE_SKINNY64;
  else if (needs_two_128x128_tiles(p, cu) && sources > 1) plan.kind = TILE_SMALL2;

  FusedParams& q = plan.p;
  q = p;
  memset(&plan.pack, 0, sizeof(plan.pack));
  plan.pack.heap_bases = p.heap_bases;
  plan.pack.rank = p.rank;
  const bool pack_a = !aligned16(p.A) || (p.s_am * es) % 16 || p.K_local % ce || (p.gather == GATHER_M && p.M_local % tile_rows(plan.kind));
  // (with several sources A's runs are padded one by one, and B's K has to follow)
  const bool pack_b = !aligned16(p.B) || ((bkc ? p.s_bn : p.s_bk) * es) % 16 || (bkc ? p.K_local : p.N) % ce || (sources > 1 && p.K_local % ce);
  const long long k_run = whole(p.K_local), k_all = sources * k_run;
  long long bytes_a = 0, bytes_b = 0;
  if (pack_a) {
    PackJob& j = plan.pack.job[0];
    j.src = p.A;
    j.src_row = p.s_am * es;
    j.rows = p.M;
    j.segments = sources;
    j.run = p.K_local;
    j.run_pieces = (int)(k_run / ce);
    j.slots_of_rows = p.gather == GATHER_M ? p.M_local : 0;
    j.slots_of_segments = p.gather == GATHER_K;
    bytes_a = (long long)p.M * k_all * es;
    q.s_am = k_all;
    q.gather = GATHER_NONE;
    q.M_local = p.M;
    q.K = q.K_local = sources > 1 ? (int)k_all : p.K;
  }
  if (pack_b) {
    PackJob& j = plan.pack.job[1];
    j.src = p.B;
    if (bkc) {
      j.src_row = p.s_bn * es;
      j.src_segment = (long long)p.K_local * es;
      j.rows = p.N;
      j.segments = sources;
      j.run = p.K_local;
      j.run_pieces = (int)(k_run / ce);
      q.s_bn = k_all;
      bytes_b = (long long)p.N * k_all * es;
    } else {
      const long long n_run = whole(p.N);
      j.src_row = p.s_bk * es;
      j.rows = sources > 1 ? (int)k_all : p.K;
      j.segments = 1;
      j.run = p.N;
      j.run_pieces = (int)(n_run / ce);
      if (sources > 1) {
        j.row_period = (int)k_run;
        j.row_run = p.K_local;
      }
      q.s_bk = n_run;
      bytes_b = j.rows * n_run * es;
    }
  }
  if (bytes_a >= (1ll << 31) || bytes_b >= (1ll << 31)) return false;  // (also what the kernel's tile offsets reach)
  const int bm = tile_rows(plan.kind), bn = tile_cols(plan.kind);
  const long long a_span = (long long)bm * q.s_am * es + (long long)q.K * es;
  const long long b_span = bkc ? (long long)bn * q.s_bn * es + (long long)q.K * es : (long long)q.K * q.s_bk * es + (long long)bn * es;
  if (a_span >= (1ll << 31) || b_span >= (1ll << 31)) return false;
  plan.pack.job[1].dst = (char*)((bytes_a + 255) / 256 * 256);  // offsets until the memory is there
  plan.bytes = (size_t)((bytes_a + 255) / 256 * 256 + bytes_b);
  if (plan.bytes > (1ull << 30)) return false;  // as much memory as a launch may ask for
  const int per_block = kPackThreads * kPackPieces;
  plan.pack.blocks[0] = (int)((bytes_a / 16 + per_block - 1) / per_block);
  plan.pack.blocks[1] = (int)((bytes_b / 16 + per_block - 1) / per_block);
  return true;
}

// Whether that is expected to take less time than the any-shape kernel, in us.  Both are modelled as a K loop, every CU as busy as the
// busiest one, at the rates (TFLOP/s) that 190 plain products showed (M 130 to 16000, N 300 to 8001, K 331 to 8001, bf16,
// two sets of operands in turn); packing moves its bytes at 5.2 TB/s and costs a launch.  What it gives and where it
// does not: 4000x2877x2501 125.4 -> 72.1 us, 2000x1501x8001 133.7 -> 84.3, 1000x701x8001 65.5 -> 44.8, e4m3 4000x4095x1371
// 55.5 -> 38.5; 4000x4095x331 25.6 -> 28.0, 500x4095x5001 54.0 -> 53.0, 16000x300x5001 127 -> 159, the last three left where they
// were.
//
// The model alone packed 2733 of 10000 launches of every operator (2, 4, 8 ranks and plain products, 16- and 8-bit, both layouts of
// B, M 1 to 12000, N 64 to 8192, K 200 to 9000, both ways timed in turn): 705 were slower for it, up to 1.9 times.  By tile, time
// packed : any-shape kernel, and how many were more than 3 % slower:
//   256x256               0.82, 55 of 758
//   128x128, one per CU   0.86, 66 of 472 from K = 2400 on; 0.96 at 2000 to 2500, 1.02 at 1600 to 2000, 1.15 at 800 to 1200
//   128x128, more tiles   1.04, two to a CU or one behind the other, but where the any-shape kernel has three nearly full rounds of
//                         64x128 tiles against two here and K is long: 0.93 (1999x2877x4003, bf16 93.6 -> 87.9 us, B transposed
//                         100.6 -> 97.9, e4m3 64.3 -> 58.6)
//   64x64, one per CU     0.83, 17 of 430; with more tiles 1.04, 154 of 297
//   instead of 32x32      1.03, 48 of 103 (e4m3 3x120x8685 18.7 -> 23.4 us); that tile also splits K over its waves, and the sums would not be
//                         those of a launch that gets no memory
// Operands gathered along K gain with every tile (0.54 to 0.82): the any-shape kernel pads the share of every slot to whole steps.
// Slot sums of other numbers of ranks than 2, 4 and 8 read the peers one behind the other, which one workgroup per CU does not
// hide (one-shot of three ranks, bf16 6000x2877x640 112 -> 138 us).
bool worth_packing(const FusedParams& p, int in_dtype, int out_dtype, int cu, const PackPlan& plan) {
  const bool fp8 = in_dtype == IRIS_HIP_FP8_E4M3;
  float any = 0.f;
  const int any_tile = choose_any_tile(p.M, p.N, cu, false, false, &any);
  if (any_tile == 4) return false;
  if (epi_has_flags(p.epi) && p.sum_peers && p.world != 1 && p.world != 2 && p.world != 4 && p.world != 8) return false;
  const float products = 2e-6f * cu * p.K;
  const float results = (float)p.M * p.N * elem_size(out_dtype) * 2e-7f;  // C, either way
  const int bm = tile_rows(plan.kind), bn = tile_cols(plan.kind);
  const long long tiles = (long long)cdiv(p.M, bm) * cdiv(p.N, bn);
  if ((p.gather != GATHER_K || p.world == 1) && plan.kind != TILE_BIG) {
    if (plan.kind == TILE_SMALL && p.K < (tiles > cu ? 4000 : 2400)) return false;
    const long long tiles_64x128 = (long long)cdiv(p.M, 64) * cdiv(p.N, 128);
    if (tiles > cu && !(plan.kind == TILE_SMALL && any_tile == 2 && tiles_64x128 * 3 > 8ll * cu && tiles_64x128 <= 3ll * cu)) return false;
  }
  const float rate = (plan.kind == TILE_BIG ? 1400.f : plan.kind == TILE_SMALL ? 1220.f : plan.kind == TILE_SMALL2 ? 964.f : tiles > cu ? 671.f : 560.f) * (fp8 ? 1.9f : 1.f);
  const float there = (float)bm * bn * ((tiles + cu - 1) / cu) / rate;
  const float packing = (plan.bytes ? 4.5f + plan.bytes * 2 / 5.2e6f : 0.f) + (plan.kind == TILE_SKINNY64 ? 4.f : 3.f);
  return packing + products * there + results < 0.92f * (4.f + products * any * (fp8 ? 0.7f : 1.f) + results);
}

// Launches p on packed operands, or, without memory for them, on the any-shape kernel.  Returns 0 or an error, or -1 with
// nothing done where the latter is to be launched as always.
int run_packed(const FusedParams& p, int in_dtype, int out_dtype, int device, int cu, hipStream_t s) {
  PackPlan plan;
  if (!plan_packing(p, in_dtype, out_dtype, cu, plan) || !worth_packing(p, in_dtype, out_dtype, cu, plan)) return -1;
  plan_tiles(plan.p, plan.kind, cu);
  void* memory = nullptr;
  if (plan.bytes) {
    memory = p.no_workspace_alloc ? nullptr : g_scratch_allocator.take(plan.bytes, s);
    if (!memory) {
      // Other ranks may have got theirs.  Where they could wait for tiles that this one never reaches, it takes the same tiles in the
      // same order (layout.h; replayed in tests/host_sim/layout_sim.cpp).
      if (publishes_alone(tile_launch(plan.p, plan.kind, cu), plan.p.group_m) && (p.epi != EPI_REDUCE_SCATTER || plan.p.interleave)) return -1;
      FusedParams q = p;
      q.group_m = plan.p.group_m;
      q.interleave = plan.p.interleave;
      return dispatch_generic(q, in_dtype, out_dtype, device, cu, s, plan.kind == TILE_BIG ? 0 : plan.kind == TILE_SKINNY64 ? 3 : 1);
    }
    PackParams& pack = plan.pack;
    pack.job[0].dst = (char*)memory;
    pack.job[1].dst = (char*)memory + (size_t)pack.job[1].dst;
    if (pack.blocks[0]) plan.p.A = pack.job[0].dst;
    if (pack.blocks[1]) plan.p.B = pack.job[1].dst;
    const dim3 grid(pack.blocks[0] + pack.blocks[1]);
    if (elem_size(in_dtype) == 2) hipLaunchKernelGGL((pack_kernel<2>), grid, dim3(kPackThreads), 0, s, pack);
    else hipLaunchKernelGGL((pack_kernel<1>), grid, dim3(kPackThreads), 0, s, pack);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      g_scratch_allocator.give_back(memory);
      return (int)e;
    }
  }
  const bool bkc = p.s_bn != 1;
  int rc = 0;
  switch (in_dtype) {
    case IRIS_HIP_BF16: rc = dispatch_mfma_rows<IN_BF16>(plan.p, plan.kind, bkc, device, s); break;
    case IRIS_HIP_FP16: rc = dispatch_mfma_rows<IN_F16>(plan.p, plan.kind, bkc, device, s); break;
    default: rc = dispatch_mfma_rows<IN_FP8>(plan.p, plan.kind, bkc, device, s);
  }
  g_scratch_allocator.give_back(memory);
  return rc;
}

// check_only: run every argument check and the kernel choice, launch nothing (0 = the launch would go out).
int run_fused(FusedParams p, int in_dtype, int out_dtype, int path, void* stream, bool check_only = false) {
  g_last_error[0] = 0;
#ifdef IRIS_HIP_PHASE_STAMPS
  p.stamps = g_stamps;
  p.stamp_rows = g_stamp_rows;
#endif
  if (p.M <= 0 || p.N <= 0 || p.K <= 0) return fail("M, N, K must be positive (got %d, %d, %d)", p.M, p.N, p.K);
  if (!p.A || !p.B || !p.C) return fail("A, B and C must not be NULL");
  if (p.world < 1 || p.rank < 0 || p.rank >= p.world) return fail("bad rank/world_size %d/%d", p.rank, p.world);
  if (epi_has_flags(p.epi)) {
    if (!p.aux || !p.locks) return fail("aux_buffer and locks must not be NULL");
    if (p.flag_bm <= 0 || p.flag_bn <= 0) return fail("block sizes must be positive");
  } else {
    p.flag_bm = 256;  // no flags on this path; any valid tile size
    p.flag_bn = 64;
  }
  // Every kernel translates addresses through the heap bases, also with one rank.
  if (!p.heap_bases) return fail("context_tensor must not be NULL");
  heap_bases_from_registry(p, (const int64_t*)p.heap_bases - 2);
  if (elem_size(in_dtype) == 0 || elem_size(out_dtype) == 0 || out_dtype == IRIS_HIP_FP8_E4M3)
    return fail("unsupported element types in=%d out=%d", in_dtype, out_dtype);

  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return (int)e;
  DeviceFacts* facts = nullptr;
  int rc = facts_for(device, &facts);
  if (rc) return rc;
  p.num_xcd = facts->xcc_count;
  p.whole_lines = rows_of_whole_lines(p, out_dtype);
  p.stream_peers = peers_past_caches(p, out_dtype);
  hipStream_t s = (hipStream_t)stream;

  // Tile choice (the tile list in fused_kernel.h has the measurements): the 256x256 tile from about half the
  // CUs busy (cross-over against the 128x128 tiles between 128 and 144 big tiles on 256 CUs) unless the output
  // has at most 64 rows; the latency-oriented 32x32 kernel (decode_kernel.h) for at most two such tiles per CU;
  // 64x64 tiles for at most two of those per CU; 64x128 tiles for at most 64 rows, and for at most two such
  // tiles per CU when K is short; else 128x128 - two workgroups per CU when there are more such tiles than CUs.
  const bool rows64_ok = !(p.gather == GATHER_M && p.M_local % 64);
  int kind = TILE_SMALL;
  if (fills_big_tiles(p, facts->cu_count) && !(p.M <= 64 && rows64_ok)) kind = TILE_BIG;
  else if (decode_sized(p, facts->cu_count, in_dtype) && decode_gather_ok(p, in_dtype) && p.world <= 8) kind = TILE_DECODE;
  else if (fits_64x64_tiles(p, facts->cu_count) && rows64_ok) kind = TILE_SKINNY64;
  else if (rows64_ok && (p.M <= 64 || ((long long)cdiv(p.M, 64) * cdiv(p.N, 128) <= 2ll * facts->cu_count &&
                                       (long long)p.K * elem_size(in_dtype) <= 2048)))
    kind = TILE_SKINNY;
  else if (needs_two_128x128_tiles(p, facts->cu_count)) kind = TILE_SMALL2;
  // IRIS_HIP_TILE = big | small | small2 | skinny | skinny64 overrides the choice among the tiled kernels (a tuning
  // aid; results do not depend on the tile shape beyond the order of the fp32 sums over K).
  static const int forced_tile = [] {
    const char* e = getenv("IRIS_HIP_TILE");
    if (!e) return -1;
    if (!strcmp(e, "big")) return (int)TILE_BIG;
    if (!strcmp(e, "small")) return (int)TILE_SMALL;
    if (!strcmp(e, "small2")) return (int)TILE_SMALL2;
    if (!strcmp(e, "skinny")) return (int)TILE_SKINNY;
    if (!strcmp(e, "skinny64")) return (int)TILE_SKINNY64;
    return -1;
  }();
  if (forced_tile >= 0 && kind != TILE_DECODE &&
      !mfma_ineligible(p, in_dtype, out_dtype, tile_rows(forced_tile), tile_cols(forced_tile)))
    kind = forced_tile;  // a tile the operands do not qualify for is not forced
  const char* why = mfma_ineligible(p, in_dtype, out_dtype, tile_rows(kind), tile_cols(kind));
  if (path == IRIS_HIP_PATH_MFMA && why) return fail("MFMA kernel not applicable: %s", why);
  if (path == IRIS_HIP_PATH_GENERIC || why) {
    if (!generic_supported(in_dtype, out_dtype)) return fail("unsupported element types in=%d out=%d", in_dtype, out_dtype);
    if (check_only) return 0;
    if (path == IRIS_HIP_PATH_AUTO) {
      rc = run_packed(p, in_dtype, out_dtype, device, facts->cu_count, s);
      if (rc >= 0) return rc;
    }
    return dispatch_generic(p, in_dtype, out_dtype, device, facts->cu_count, s);
  }
  if (check_only) return 0;

  const bool bkc = (p.s_bn != 1);
  switch (in_dtype) {
    case IRIS_HIP_BF16: rc = dispatch_mfma_in<IN_BF16>(p, kind, bkc, device, facts->cu_count, s); break;
    case IRIS_HIP_FP16: rc = dispatch_mfma_in<IN_F16>(p, kind, bkc, device, facts->cu_count, s); break;
    case IRIS_HIP_FP8_E4M3: rc = dispatch_mfma_in<IN_FP8>(p, kind, bkc, device, facts->cu_count, s); break;
    default: rc = fail("unsupported input type %d", in_dtype);
  }
  return rc;
}

bool fits_int(int64_t v) { return v > 0 && v < (1ll << 31); }

// iris_hip_matmul_all_reduce; check_only stops in front of the launch (see run_fused).
int matmul_all_reduce_impl(const void* A, const void* B, void* C, void* aux_buffer, int32_t* locks,
                               int64_t M, int64_t N, int64_t K,
                               int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                               int64_t stride_cm, int64_t stride_cn,
                               const int64_t* context_tensor, int32_t cur_rank, int32_t world_size,
                               int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                               int32_t variant, int32_t in_dtype, int32_t out_dtype, float scale,
                               int32_t acc_mode, int64_t spin_limit, int32_t* status, int32_t path,
                               void* stream, bool check_only, bool no_alloc = false) {
  (void)block_size_k;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K)) return fail("M, N, K must be in [1, 2^31)");
  if (variant != IRIS_HIP_VARIANT_ATOMIC && variant != IRIS_HIP_VARIANT_ONE_SHOT && variant != IRIS_HIP_VARIANT_TWO_SHOT)
    return fail("variant %d is not atomic (0), one_shot (2) or two_shot (3)", variant);
  FusedParams p;
  memset(&p, 0, sizeof(p));
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C; p.aux = (char*)aux_buffer; p.locks = locks;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.K_local = (int)K; p.gather = GATHER_NONE;
  p.s_am = stride_am; p.s_ak = stride_ak; p.s_bk = stride_bk; p.s_bn = stride_bn;
  p.s_cm = stride_cm; p.s_cn = stride_cn;
  p.heap_bases = context_tensor ? (const long long*)(context_tensor + 2) : nullptr;
  p.rank = cur_rank; p.world = world_size;
  p.flag_bm = block_size_m; p.flag_bn = block_size_n;
  p.epi = variant == IRIS_HIP_VARIANT_ATOMIC ? EPI_ATOMIC : variant == IRIS_HIP_VARIANT_ONE_SHOT ? EPI_ONE_SHOT : EPI_TWO_SHOT;
  p.acc_mode = acc_mode & ~IRIS_HIP_CLEAR_C; p.clear_c = (acc_mode & IRIS_HIP_CLEAR_C) != 0; p.all_owners = 0; p.sum_peers = 1;
  p.scale = scale; p.spin_limit = spin_limit; p.status = status;
  p.no_workspace_alloc = no_alloc ? 1 : 0;
  return run_fused(p, in_dtype, out_dtype, path, stream, check_only);
}

}  // namespace

namespace iris_host {

int fail(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_last_error, sizeof(g_last_error), fmt, ap);
  va_end(ap);
  return (int)hipErrorInvalidValue;
}

void clear_last_error() { g_last_error[0] = 0; }

void set_last_kernel(const char* name) { snprintf(g_last_kernel, sizeof(g_last_kernel), "%s", name); }

namespace {
struct SplitTileWorkspace {
  int device;
  hipStream_t stream;
  char* partials;
  int* flags;
  int nwg;
  long long slot_bytes;
  unsigned epoch;
};
constexpr int kMaxSplitWorkspacesPerDevice = 8;
std::vector<SplitTileWorkspace> g_split_workspaces;
std::mutex g_split_mutex;
}  // namespace

namespace {
std::atomic<int> g_split_mode{[] { const char* e = getenv("IRIS_HIP_STREAMK"); return e ? atoi(e) : -1; }()};
}
int split_tile_mode() { return g_split_mode.load(std::memory_order_relaxed); }
void set_split_tile_mode(int mode) { g_split_mode.store(mode < 0 ? -1 : (mode > 2 ? 2 : mode), std::memory_order_relaxed); }

int split_tile_workspace(int device, hipStream_t stream, int nwg, long long slot_bytes, char** partials, int** flags, int* epoch) {
  // Never under stream capture: the flag value of a launch is a kernel argument, a replayed launch would
  // meet the flags of its previous replay already at that value and read partial sums before they are
  // written.  (And nothing may be allocated or cleared on a capturing stream.)
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return 1;
  }
  std::lock_guard<std::mutex> lock(g_split_mutex);
  int on_device = 0;
  for (SplitTileWorkspace& w : g_split_workspaces) {
    if (w.device != device) continue;
    ++on_device;
    if (w.stream != stream || w.nwg < nwg || w.slot_bytes < slot_bytes) continue;
    w.epoch = w.epoch % 0x7FFFFFFFu + 1;  // 1 .. 2^31 - 1: never the 0 the flags start with
    *partials = w.partials;
    *flags = w.flags;
    *epoch = (int)w.epoch;
    return 0;
  }
  if (on_device >= kMaxSplitWorkspacesPerDevice) return 1;
  // First split launch on this stream.
  SplitTileWorkspace w{device, stream, nullptr, nullptr, nwg, slot_bytes, 1u};
  if (hipMalloc((void**)&w.partials, (size_t)nwg * (size_t)slot_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  if (hipMalloc((void**)&w.flags, (size_t)nwg * sizeof(int)) != hipSuccess ||
      hipMemsetAsync(w.flags, 0, (size_t)nwg * sizeof(int), stream) != hipSuccess) {
    (void)hipGetLastError();
    (void)hipFree(w.partials);
    if (w.flags) (void)hipFree(w.flags);
    return 1;
  }
  g_split_workspaces.push_back(w);
  *partials = w.partials;
  *flags = w.flags;
  *epoch = 1;
  return 0;
}

int device_facts(int device, int* cu_count, int* xcc_count) {
  DeviceFacts* f = nullptr;
  const int rc = facts_for(device, &f);
  if (rc) return rc;
  *cu_count = f->cu_count;
  *xcc_count = f->xcc_count;
  return 0;
}

}  // namespace iris_host

extern "C" {

int iris_hip_matmul_all_reduce(const void* A, const void* B, void* C, void* aux_buffer, int32_t* locks,
                               int64_t M, int64_t N, int64_t K,
                               int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                               int64_t stride_cm, int64_t stride_cn,
                               const int64_t* context_tensor, int32_t cur_rank, int32_t world_size,
                               int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                               int32_t variant, int32_t in_dtype, int32_t out_dtype, float scale,
                               int32_t acc_mode, int64_t spin_limit, int32_t* status, int32_t path,
                               void* stream) {
  return matmul_all_reduce_impl(A, B, C, aux_buffer, locks, M, N, K, stride_am, stride_ak, stride_bk, stride_bn, stride_cm,
                                stride_cn, context_tensor, cur_rank, world_size, block_size_m, block_size_n, block_size_k,
                                variant, in_dtype, out_dtype, scale, acc_mode, spin_limit, status, path, stream, false);
}

int iris_hip_matmul_all_reduce_noalloc(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                                       int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                                       int64_t stride_cm, int64_t stride_cn,
                                       int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                                       int32_t variant, int32_t in_dtype, int32_t out_dtype, float scale,
                                       int32_t path, void* stream) {
  g_last_error[0] = 0;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K)) return fail("M, N, K must be in [1, 2^31)");
  if (variant != IRIS_HIP_VARIANT_ONE_SHOT && variant != IRIS_HIP_VARIANT_TWO_SHOT)
    return fail("variant %d is not one_shot (2) or two_shot (3)", variant);
  if (block_size_m <= 0 || block_size_n <= 0) return fail("block sizes must be positive");
  const int es = elem_size(out_dtype);
  if (es == 0) return fail("unsupported element types in=%d out=%d", in_dtype, out_dtype);
  if (stride_cm < 0 || stride_cn < 0) return fail("negative output strides are not supported");
  if (stride_cm >= (1ll << 40) || stride_cn >= (1ll << 40)) return fail("output strides beyond 2^40 elements are not supported");
  // aux is addressed with C's strides: the bytes it spans and the flags of the tile grid must fit.
  const long long aux_bytes = ((long long)(M - 1) * stride_cm + (long long)(N - 1) * stride_cn + 1) * es;
  const long long nflags = (long long)cdiv((int)M, block_size_m) * cdiv((int)N, block_size_n);
  if (aux_bytes > (long long)IRIS_HIP_NOALLOC_MAX_AUX_BYTES)
    return fail("output of %lld x %lld spans %lld bytes, beyond the %lld bytes of the library's workspace; "
                "use iris_hip_matmul_all_reduce with a caller-owned workspace",
                (long long)M, (long long)N, aux_bytes, (long long)IRIS_HIP_NOALLOC_MAX_AUX_BYTES);
  if (nflags > IRIS_HIP_NOALLOC_MAX_FLAGS)
    return fail("%lld tiles of %d x %d, beyond the %d flags of the library's workspace; use larger block sizes "
                "or iris_hip_matmul_all_reduce with a caller-owned workspace",
                nflags, block_size_m, block_size_n, IRIS_HIP_NOALLOC_MAX_FLAGS);
  unsigned char* base = nullptr;
  int rc = scratch_for_current_device(&base);
  if (rc) return rc;
  long long* context = (long long*)base;
  int32_t* locks = (int32_t*)(base + kScratchContextBytes);
  void* aux = base + kScratchAuxOffset;
  // Every check of the launch itself (types, path, strides) before the prepare kernel goes out: a rejected
  // call enqueues nothing and leaves the workspace alone.
  rc = matmul_all_reduce_impl(A, B, C, aux, locks, M, N, K, stride_am, stride_ak, stride_bk, stride_bn, stride_cm, stride_cn,
                              (const int64_t*)context, 0, 1, block_size_m, block_size_n, block_size_k, variant, in_dtype,
                              out_dtype, scale, IRIS_HIP_ACC_FP32, 0, nullptr, path, stream, true, true);
  if (rc) return rc;
  const int threads = 256;
  const int need = (int)nflags > (int)(kScratchContextBytes / sizeof(long long)) ? (int)nflags : (int)(kScratchContextBytes / sizeof(long long));
  hipLaunchKernelGGL(noalloc_prepare_kernel, dim3((need + threads - 1) / threads), dim3(threads), 0, (hipStream_t)stream,
                     context, locks, (int)nflags);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return (int)e;
  return matmul_all_reduce_impl(A, B, C, aux, locks, M, N, K, stride_am, stride_ak, stride_bk, stride_bn, stride_cm,
                                stride_cn, (const int64_t*)context, 0, 1, block_size_m, block_size_n, block_size_k,
                                variant, in_dtype, out_dtype, scale, IRIS_HIP_ACC_FP32, 0, nullptr, path, stream, false, true);
}

int iris_hip_matmul_reduce_scatter(const void* A, const void* B, void* C, void* aux_buffer, int32_t* locks,
                                   int64_t M, int64_t N, int64_t K,
                                   int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                                   int64_t stride_cm, int64_t stride_cn,
                                   const int64_t* context_tensor, int32_t cur_rank, int32_t world_size,
                                   int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                                   int32_t all_owners, int32_t sum_peers,
                                   int32_t in_dtype, int32_t out_dtype, float scale, int32_t acc_mode,
                                   int64_t spin_limit, int32_t* status, int32_t path, void* stream) {
  (void)block_size_k;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K)) return fail("M, N, K must be in [1, 2^31)");
  FusedParams p;
  memset(&p, 0, sizeof(p));
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C; p.aux = (char*)aux_buffer; p.locks = locks;
  p.M = (int)M; p.N = (int)N; p.K = (int)K; p.K_local = (int)K; p.gather = GATHER_NONE;
  p.s_am = stride_am; p.s_ak = stride_ak; p.s_bk = stride_bk; p.s_bn = stride_bn;
  p.s_cm = stride_cm; p.s_cn = stride_cn;
  p.heap_bases = context_tensor ? (const long long*)(context_tensor + 2) : nullptr;
  p.rank = cur_rank; p.world = world_size;
  p.flag_bm = block_size_m; p.flag_bn = block_size_n;
  p.epi = EPI_REDUCE_SCATTER;
  p.acc_mode = acc_mode & ~IRIS_HIP_CLEAR_C; p.clear_c = (acc_mode & IRIS_HIP_CLEAR_C) != 0; p.all_owners = all_owners ? 1 : 0; p.sum_peers = sum_peers ? 1 : 0;
  p.scale = scale; p.spin_limit = spin_limit; p.status = status;
  return run_fused(p, in_dtype, out_dtype, path, stream);
}

int iris_hip_all_gather_matmul(const void* A_sharded, const void* B, void* C, const void* bias,
                               int64_t M, int64_t N, int64_t K, int64_t K_local,
                               int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                               int64_t stride_cm, int64_t stride_cn, int64_t stride_bias,
                               const int64_t* context_tensor, int32_t cur_rank, int32_t world_size,
                               int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                               int32_t gather_dim, int32_t in_dtype, int32_t out_dtype, int32_t bias_dtype,
                               float scale, int32_t path, void* stream) {
  (void)block_size_m; (void)block_size_n; (void)block_size_k;
  if (!fits_int(M) || !fits_int(N) || !fits_int(K) || !fits_int(K_local))
    return fail("M, N, K, K_local must be in [1, 2^31)");
  FusedParams p;
  memset(&p, 0, sizeof(p));
  p.A = (const char*)A_sharded; p.B = (const char*)B; p.C = (char*)C; p.bias = (const char*)bias;
  p.M = (int)M; p.N = (int)N; p.K = (int)K;
  if (gather_dim == IRIS_HIP_GATHER_K) {
    if (K != (int64_t)world_size * K_local)
      return fail("K (%lld) must equal world_size (%d) * K_local (%lld)", (long long)K, world_size, (long long)K_local);
    p.gather = GATHER_K; p.K_local = (int)K_local; p.M_local = (int)M;
  } else if (gather_dim == IRIS_HIP_GATHER_M) {
    if (K_local != K) return fail("gather along M needs K_local == K");
    if (M % world_size) return fail("gather along M needs M divisible by world_size");
    p.gather = GATHER_M; p.K_local = (int)K; p.M_local = (int)(M / world_size);
  } else {
    return fail("gather_dim %d is not 1 (K) or 2 (M)", gather_dim);
  }
  if (bias && elem_size(bias_dtype) < 2) return fail("unsupported bias type %d", bias_dtype);
  p.s_am = stride_am; p.s_ak = stride_ak; p.s_bk = stride_bk; p.s_bn = stride_bn;
  p.s_cm = stride_cm; p.s_cn = stride_cn; p.s_bias = stride_bias; p.bias_dtype = bias_dtype;
  p.heap_bases = context_tensor ? (const long long*)(context_tensor + 2) : nullptr;
  p.rank = cur_rank; p.world = world_size;
  p.epi = EPI_STORE; p.scale = scale;
  return run_fused(p, in_dtype, out_dtype, path, stream);
}

int iris_hip_matmul_all_gather(const void* A, const void* B, void* C_gathered, const void* bias,
                               int64_t M_local, int64_t M, int64_t N, int64_t K,
                               int64_t stride_am, int64_t stride_ak, int64_t stride_bk, int64_t stride_bn,
                               int64_t stride_cm_gathered, int64_t stride_cn_gathered, int64_t stride_bias,
                               const int64_t* context_tensor, int32_t cur_rank, int32_t world_size,
                               int32_t block_size_m, int32_t block_size_n, int32_t block_size_k,
                               int32_t in_dtype, int32_t out_dtype, int32_t bias_dtype, float scale,
                               int32_t path, void* stream) {
  (void)block_size_m; (void)block_size_n; (void)block_size_k;
  if (!fits_int(M_local) || !fits_int(M) || !fits_int(N) || !fits_int(K))
    return fail("M_local, M, N, K must be in [1, 2^31)");
  if (world_size < 1 || M != M_local * world_size)
    return fail("M (%lld) must equal M_local (%lld) * world_size (%d)", (long long)M, (long long)M_local, world_size);
  if (bias && elem_size(bias_dtype) < 2) return fail("unsupported bias type %d", bias_dtype);
  FusedParams p;
  memset(&p, 0, sizeof(p));
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C_gathered; p.bias = (const char*)bias;
  p.M = (int)M_local; p.N = (int)N; p.K = (int)K; p.K_local = (int)K; p.gather = GATHER_NONE;
  p.s_am = stride_am; p.s_ak = stride_ak; p.s_bk = stride_bk; p.s_bn = stride_bn;
  p.s_cm = stride_cm_gathered; p.s_cn = stride_cn_gathered; p.s_bias = stride_bias; p.bias_dtype = bias_dtype;
  p.heap_bases = context_tensor ? (const long long*)(context_tensor + 2) : nullptr;
  p.rank = cur_rank; p.world = world_size;
  p.row_offset = (int)(cur_rank * M_local);
  p.epi = EPI_ALL_GATHER; p.scale = scale;
  return run_fused(p, in_dtype, out_dtype, path, stream);
}

int iris_hip_register_context(const int64_t* context_tensor, const int64_t* host_copy, int32_t num_words) {
  g_last_error[0] = 0;
  if (!context_tensor || !host_copy) return fail("context_tensor and host_copy must not be NULL");
  if (num_words < 3) return fail("a context tensor has at least 3 words (rank, world size, one heap base)");
  const int64_t rank = host_copy[0], world = host_copy[1];
  if (world < 1 || rank < 0 || rank >= world || num_words < 2 + world)
    return fail("bad context contents: rank %lld, world size %lld, %d words", (long long)rank, (long long)world, num_words);
  KnownContext k;
  k.device_ptr = context_tensor;
  k.rank = (int)rank;
  k.world = (int)world;
  for (int r = 0; r < kMaxCachedSlots; ++r) k.bases[r] = r < world ? (long long)host_copy[2 + r] : 0ll;
  std::lock_guard<std::mutex> lock(g_contexts_mutex);
  for (KnownContext& e : g_contexts)
    if (e.device_ptr == context_tensor) {
      e = k;
      return 0;
    }
  g_contexts.push_back(k);
  return 0;
}

int iris_hip_unregister_context(const int64_t* context_tensor) {
  g_last_error[0] = 0;
  std::lock_guard<std::mutex> lock(g_contexts_mutex);
  for (size_t i = 0; i < g_contexts.size(); ++i)
    if (g_contexts[i].device_ptr == context_tensor) {
      g_contexts.erase(g_contexts.begin() + i);
      break;
    }
  return 0;
}

int iris_hip_query(int32_t device, int32_t* cu_count, int32_t* xcc_count, int32_t* lds_bytes_per_block) {
  g_last_error[0] = 0;
  DeviceFacts* f = nullptr;
  int rc = facts_for(device, &f);
  if (rc) return rc;
  if (cu_count) *cu_count = f->cu_count;
  if (xcc_count) *xcc_count = f->xcc_count;
  if (lds_bytes_per_block) *lds_bytes_per_block = f->lds_per_block;
  // Set-up call of the host layer: also look up the no-allocation entry point's workspace address
  // when `device` is the current one, so that its first call has nothing left to resolve.
  int current = -1;
  if (hipGetDevice(&current) == hipSuccess && current == device) {
    unsigned char* unused = nullptr;
    rc = scratch_for_current_device(&unused);
    if (rc) return rc;
  }
  return 0;
}

#ifdef IRIS_HIP_PHASE_STAMPS
// Diagnostic build only: device buffer of `rows` rows of 16 64-bit words, or NULL.  A launch writes row
// it * (number of workgroups) + (workgroup) for the first eight tiles `it` of every workgroup; rows beyond
// the buffer are not written.
void iris_hip_debug_set_stamps(void* device_buffer, long long rows) {
  g_stamps = (unsigned long long*)device_buffer;
  g_stamp_rows = device_buffer ? rows : 0;
}
#endif

void iris_hip_set_split_tiles(int32_t mode) { iris_host::set_split_tile_mode(mode); }

const char* iris_hip_last_error(void) { return g_last_error; }
const char* iris_hip_last_kernel(void) { return g_last_kernel; }
void iris_hip_set_scratch_allocator(iris_hip_allocate_fn allocate, iris_hip_release_fn release) {
  g_scratch_allocator.release.store(release, std::memory_order_release);
  g_scratch_allocator.allocate.store(release ? allocate : nullptr, std::memory_order_release);
}

int iris_hip_stream_capturing(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return status != hipStreamCaptureStatusNone;
}

int iris_hip_abi_version(void) { return 7; }

}  // extern "C"
