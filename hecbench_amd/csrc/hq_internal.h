// Internal helpers shared by the libhq translation units (not part of the ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hq.h"

// internal flag bit of the split-K kernels: formal release/acquire fences in the arrival protocol
#define HQ_FLAG_STRICT_FENCES 0x80000000u

#define HQ_HIP_TRY(expr)                      \
  do {                                        \
    hipError_t hq_e_ = (expr);                \
    if (hq_e_ != hipSuccess) return (int)hq_e_; \
  } while (0)

typedef uint32_t hq_u2v __attribute__((ext_vector_type(2)));
typedef uint32_t hq_u4v __attribute__((ext_vector_type(4)));

// The launch status of a kernel enqueued with <<<>>> (packers, clearing kernels) as an hq return code.
static inline int hq_launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? HQ_OK : (int)e;
}

// ---- launches ------------------------------------------------------------------------------------------------------
// A call that is short on the device costs what its launch costs on the host, and there the runtime handles a kernel's arguments
// one by one: thirteen of them 3.75 us a launch, two to four 2.65 (an empty kernel, launches back to back; the <<<>>> path's
// pushed configuration and the separate look at the last error are 0.15 of it).  So a kernel takes its arguments packed into
// a few vectors, which the wave finds in scalar registers as it would find scalars (the first 14 dwords; the Makefile's
// preload option), and reads them with HqReader in the order in which hq_launch() was given them.
#define HQ_ARGS8 hq_u4v hq_a0, hq_u4v hq_a1
#define HQ_ARGS12 HQ_ARGS8, hq_u4v hq_a2
#define HQ_ARGS16 HQ_ARGS12, hq_u2v hq_a3, hq_u2v hq_a4
#define HQ_ARGS24 HQ_ARGS16, hq_u4v hq_a5, hq_u4v hq_a6
#define HQ_PASS8 hq_a0, hq_a1
#define HQ_PASS12 HQ_PASS8, hq_a2
#define HQ_PASS16 HQ_PASS12, hq_a3, hq_a4
#define HQ_PASS24 HQ_PASS16, hq_a5, hq_a6
#define HQ_ARGS28 HQ_ARGS24, hq_u4v hq_a7
#define HQ_PASS28 HQ_PASS24, hq_a7
struct HqReader {
  uint32_t d[28];
  int at = 0;
  template <typename... V>
  __device__ __forceinline__ explicit HqReader(V... v) {
    int n = 0;
    (put(v, n), ...);
  }
  __device__ __forceinline__ void put(hq_u2v v, int& n) { d[n++] = v.x; d[n++] = v.y; }
  __device__ __forceinline__ void put(hq_u4v v, int& n) { d[n++] = v.x; d[n++] = v.y; d[n++] = v.z; d[n++] = v.w; }
  __device__ __forceinline__ uint32_t word() { return d[at++]; }
  __device__ __forceinline__ uint64_t twice() {
    at += at & 1;
    const uint64_t lo = d[at];
    at += 2;
    return (uint64_t)d[at - 1] << 32 | lo;
  }
  // what a kernel's pointer argument points to is global memory: so the compiler would know, and is told
  template <typename T>
  __device__ __forceinline__ operator T*() { return (T*)(__attribute__((address_space(1))) T*)twice(); }
  __device__ __forceinline__ operator int() { return (int)word(); }
  __device__ __forceinline__ operator uint32_t() { return word(); }
  __device__ __forceinline__ operator float() { return __builtin_bit_cast(float, word()); }
  __device__ __forceinline__ operator int64_t() { return (int64_t)twice(); }
};

template <typename... T>
constexpr size_t hq_packed_bytes() {
  size_t n = 0;
  ((n = (n + sizeof(T) - 1) / sizeof(T) * sizeof(T) + sizeof(T)), ...);
  return n;
}
template <typename... P, typename... T>
static inline int hq_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t smem, hipStream_t stream, T... args) {
  constexpr size_t room = (sizeof(P) + ...);
  static_assert(((sizeof(T) == 4 || sizeof(T) == 8) && ...), "what HqReader reads");
  static_assert(hq_packed_bytes<T...>() <= room, "the words that the kernel declares");
  alignas(16) unsigned char buf[room] = {};
  size_t n = 0;
  auto put = [&](const auto& x) {
    n = (n + sizeof(x) - 1) / sizeof(x) * sizeof(x);
    __builtin_memcpy(buf + n, &x, sizeof(x));
    n += sizeof(x);
  };
  (put(args), ...);
  void* params[sizeof...(P)];
  size_t at = 0, i = 0;
  ((params[i++] = buf + at, at += sizeof(P)), ...);
  const hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, params, smem, stream);
  if (e != hipSuccess) (void)hipGetLastError();  // it is this call's error and returned with it
  return e == hipSuccess ? HQ_OK : (int)e;
}
template <typename T> struct HqSame { typedef T type; };  // keeps the arguments out of the deduction
// A kernel that takes its arguments as they are: a structure, which it loads for itself; pointers whose __restrict__ the generated
// code turns to account (the 8-bit quantiser of 10^7 floats 10.9 us, 11.7 with packed arguments); or a kernel whose instructions
// the compiler orders better so (the dense column kernel, the 64-row product) and whose calls wait for the device anyway.
template <typename... P>
static inline int hq_launch_as_is(void (*kernel)(P...), dim3 grid, dim3 block, size_t smem, hipStream_t stream, typename HqSame<P>::type... args) {
  void* params[] = {const_cast<void*>(static_cast<const void*>(&args))...};
  const hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, params, smem, stream);
  if (e != hipSuccess) (void)hipGetLastError();
  return e == hipSuccess ? HQ_OK : (int)e;
}

struct HqDevice {
  int ordinal;
  int cus;         // compute units reported by hipGetDeviceProperties
  int lds_per_cu;  // bytes
  bool ok;         // gfx950
};

// Device facts for the current device (cached per ordinal).  Returns an hq code.
int hq_current_device(const HqDevice** out);

struct HqWorkspace {
  float* partial;      // split-K partial sums
  unsigned* counters;  // zero between calls: arrival counters (self-resetting), or exchange slots of two each (hq_meet)
  size_t partial_floats;
  size_t ncounters;
};

// Workspace of (current device, stream) holding at least the requested sizes, and counters for want_slots slots unless the stream is
// being captured or they cannot be had.
// Allocated on first use, grown geometrically on demand (reserve: to no more than the request), freed by hq_shutdown().
int hq_get_workspace(hipStream_t stream, size_t need_floats, size_t need_counters,
                     HqWorkspace* out, size_t want_slots = 0, bool reserve = false);
// A second one of the stream, for kernels that do without under capture: no graph uses it, so its calls are ordered with everything
// that does, whatever is replayed elsewhere.
int hq_get_eager_workspace(hipStream_t stream, size_t need_floats, size_t need_counters, HqWorkspace* out, bool reserve = false);
// Whether that would allocate while the stream is being captured, where an allocation is an error: a plan that can do
// without a workspace then does.
bool hq_workspace_out_of_reach(hipStream_t stream, size_t need_floats, size_t need_counters);
// Where the `nsplit` shares of a divided K meet, `floats` partial sums in all: in exchange slots (*arrivals null, *partial the slots,
// up to kHqMeetMost shares and no formal fences), or (nsplit 0: in any case) through partial sums and arrival counters.  The workspace has room for those
// either way, so a captured call finds what an eager one has left behind, and gives the same bits on both ways.
int hq_get_split(hipStream_t stream, size_t floats, size_t counters, int nsplit, float** partial, unsigned** arrivals);

// Caller-provided scratch of the GPTQ 3-bit paths (the entry point that allocates nothing passes its
// fixed device array here; a null pointer means "use the stream's workspace").
struct HqQ3Scratch {
  float* partial;          // split-K partial sums, also the batched GEMM's re-ordered activations
  size_t partial_floats;
  float* rows;             // 256 floats: row sums and row scales of the batched GEMM
  unsigned* counters;      // split-K arrival counters (cleared by the call that uses them)
  size_t ncounters;
  float* sums;             // raw sums of the batched GEMM's K split
  size_t sums_floats;
  float* tiles;            // all that the tiled kernels take, in place of partial, rows and sums (it may overlap those)
  size_t tiles_floats;
};
int hq_q3_matvec_impl(const void* x, int x_dtype, const int32_t* qweight, const float* scales, const float* zeros,
                      float* y, int K, int N, int batch_M, unsigned flags, hipStream_t stream,
                      const HqQ3Scratch* fixed);
// Batched 3-bit GEMM: the pre-pass (activations [M][K] -> operand-slot order of Mpad rows and Gpad k-groups, row sums and
// 1 / row scale; the product's arrival counters cleared), and the tiled kernels for many rows.
int hq_q3_gemm_prep_launch(const void* A, void* Ap, float* rowsum, float* rowinv, int M, int K, int Mpad, int Gpad,
                           unsigned* counters, size_t ncounters, hipStream_t stream);
bool hq_q3_tiles_serve(int N, int M);
// (cut_off: and the columns that the tiles leave to the one-launch kernel, which does without where there is no room)
int hq_q3_tiles_need(int cus, int K, int N, int M, bool cut_off, size_t* floats, size_t* counters);
void hq_q3_tiles_bound(int cus, int max_K, size_t* floats, size_t* counters);
int hq_q3_tiles_launch(const void* x, const int32_t* qweight, const float* scales, const float* zeros, float* y, int K, int N,
                       int M, unsigned flags, hipStream_t stream, const HqQ3Scratch* fixed);
float hq_q3_tiles_us(int cus, int K, int N, int M);  // estimate of a call, pre-pass included
// The same product in one launch (small and medium problems), always able to do without scratch.  Making the plan tries up to 32
// forms and shares (0.25 us), so whoever chooses this kernel makes it once, after everything that can be decided without it, and
// hands it to the launch.
struct HqQ3DirectPlan {
  int kind, tm, tn, ks, nmt, ntiles, T, nshare, L;
  float us;  // estimate of a call
  size_t partial_floats, counters;
};
bool hq_q3_direct_can(int K, int N);  // whether the kernel can take the matrix at all
bool hq_q3_direct_forced();           // a test's override
HqQ3DirectPlan hq_q3_direct_plan(int cus, int K, int N, int M, bool undivided);
// Columns col0 (a multiple of 256) to N; the plan is one of N - col0 columns.
int hq_q3_direct_launch(HqQ3DirectPlan plan, int cus, const void* x, const int32_t* qweight, const float* scales, const float* zeros,
                        float* y, int K, int N, int M, int col0, unsigned flags, hipStream_t stream, const HqQ3Scratch* fixed);
// The kernel of a batch where scratch is no question (so that a test can say what it runs).
enum HqQ3Kernel { HQ_Q3_KERNEL_BLOCK, HQ_Q3_KERNEL_DIRECT, HQ_Q3_KERNEL_ROWS64, HQ_Q3_KERNEL_TILES };
int hq_q3_batch_kernel(int cus, int K, int N, int M);
int hq_q3_gemm_kernel_of(int cus, int K, int N, int M);  // of those that hq_q3_gemm_launch chooses from
// Resolves the current device's copy of the fixed scratch array (once per device).
int hq_noalloc_setup(void);

// Launch-shape overrides for tests and sweeps (hq_set_tunable, or the environment variable of the
// same name, which is read once per process).  hq_tune returns dflt while a knob is unset; it costs
// one relaxed atomic load.
enum HqTunable {
  HQ_TUNE_Q3_WAVES, HQ_TUNE_Q3_STEPS, HQ_TUNE_Q3_KSPLIT, HQ_TUNE_Q3_TILE, HQ_TUNE_Q3_SMALL_BATCH, HQ_TUNE_Q3_ROW_BLOCKS, HQ_TUNE_LUT_PATH, HQ_TUNE_LUT_KSPLIT,
  HQ_TUNE_NF4_PIPE, HQ_TUNE_AQLM_ROWS, HQ_TUNE_Q8_WGS, HQ_TUNE_Q8_FAST, HQ_TUNE_GEMV_LDS, HQ_TUNE_GEMV_SPLIT, HQ_TUNE_SPLITK_FENCES, HQ_TUNE_Q3_TILES, HQ_TUNE_LUT_FINE, HQ_TUNE_COUNT
};
int hq_tune(HqTunable id, int dflt);

// ---- the lanes of a wave together ----------------------------------------------------------------------------------------
// On the data path's own lane exchanges (DPP) inside each row of 16 lanes, then the four rows' results as scalars: no LDS.  As a
// butterfly of shuffles, which go through the LDS crossbar, 0.2 us more where it is exposed (the AQLM matvec's waves end with one:
// 1311 x 9536, three code books, 10.75 / 10.45 us; the batched product's pre-pass has two: 32 x 4096 x 11008 13.55 / 13.3).
template <int CTRL>
__device__ __forceinline__ float hq_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float hq_lane(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
template <typename OP>
__device__ __forceinline__ float hq_quad(float v, OP op) {
  v = op(v, hq_dpp<0xB1>(v));     // quad_perm [1,0,3,2]
  return op(v, hq_dpp<0x4E>(v));  // quad_perm [2,3,0,1]
}
template <typename OP>
__device__ __forceinline__ float hq_row(float v, OP op) {
  v = hq_quad(v, op);
  v = op(v, hq_dpp<0x141>(v));     // row_half_mirror
  return op(v, hq_dpp<0x140>(v));  // row_mirror
}
template <typename OP>
__device__ __forceinline__ float hq_wave(float v, OP op) {
  v = hq_row(v, op);
  return op(op(hq_lane(v, 0), hq_lane(v, 16)), op(hq_lane(v, 32), hq_lane(v, 48)));
}
struct HqAdd {
  __device__ __forceinline__ float operator()(float x, float y) const { return x + y; }
};
struct HqMax {
  __device__ __forceinline__ float operator()(float x, float y) const { return fmaxf(x, y); }
};
struct HqMin {
  __device__ __forceinline__ float operator()(float x, float y) const { return fminf(x, y); }
};
__device__ __forceinline__ float hq_wave_sum(float v) { return hq_wave(v, HqAdd()); }
__device__ __forceinline__ float hq_wave_max(float v) { return hq_wave(v, HqMax()); }

// Sum of the nsplit partial sums p[s * stride] of a K split, added in split order, up to eight in hq_meet's tree (the result does
// not depend on which workgroup arrived last, nor on which way the sums met).  The loads are device-scope atomic loads, which bypass the non-coherent
// cache levels; eight of them are in flight at a time - one after the other each costs a trip to memory, and
// the last workgroup of a tile is the last thing a kernel does.
__device__ __forceinline__ float hq_sum_partials(const float* p, size_t stride, int nsplit) {
  float sum = 0.f;
  if (nsplit <= 8) {  // in the tree of hq_meet
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = __hip_atomic_load(p + (size_t)min(j, nsplit - 1) * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int j = 2; j < 8; ++j) v[j] = j < nsplit ? v[j] : 0.f;
    return 0.f + (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
  }
  for (int s0 = 0; s0 < nsplit; s0 += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int s = s0 + j < nsplit ? s0 + j : nsplit - 1;
      v[j] = __hip_atomic_load(p + (size_t)s * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += s0 + j < nsplit ? v[j] : 0.f;
  }
  return sum;
}

// A few shares of K meet without a count: two and two in a slot of their column, {1, a sum} in one 64-bit exchange at the memory
// side.  Whoever finds the slot empty is done; whoever finds the other's sum goes on with both, to the next pair, and the one that
// goes through all holds the total.  Where the shares arrive together that is one trip to memory for two of them and two for four,
// in place of three (the partial sums' acknowledgement, the count, and the sums back).  Nobody waits for anybody, and the sums are
// added in the same tree whoever comes first: (0 + 1) + (2 + 3).  A slot is empty again when its second visitor has gone.
// slots: this column's, `stride` apart, nsplit - 1 of them.  True in the lanes that hold the total.
__device__ __forceinline__ bool hq_meet(unsigned long long* slots, size_t stride, int share, int nsplit, float& v) {
  for (int n = nsplit, first = 0; n > 1; first += n >> 1, n = (n + 1) >> 1, share >>= 1) {
    if ((share ^ 1) >= n) continue;  // the last of an odd number goes on by itself
    unsigned long long* slot = slots + (size_t)(first + (share >> 1)) * stride;
    const unsigned long long other =
        __hip_atomic_exchange(slot, 1ull << 32 | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!(other >> 32)) return false;
    v += __uint_as_float((uint32_t)other);
    __hip_atomic_store(slot, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  return true;
}
// Up to eight shares, three trips at most.  3-bit matvec, count / exchange, us: two shares 8192 x 640 5.1 / 4.2, 8192 x 28672 18.1 / 17.2;
// three 11008 x 4096 6.45 / 6.2; five 20480 x 4096 9.4 / 9.1; eight 32768 x 2048 7.9 / 7.5; ten 39136 x 364 7.0 / 7.3 (four trips: not
// taken).  Four rows, two shares, 4224 x 2200 6.9 / 6.05.  LUT-GEMM: two shares 8192 x 8192 8.15 / 7.35, three 11008 x 4096 7.8 / 7.1,
// six 6016 x 2265 (two planes) 5.8 / 5.0, eight 7552 x 2166 (groups of 64) 6.9 / 6.2.
constexpr int kHqMeetMost = 8;
constexpr size_t kHqMostSlots = (size_t)4 << 20;  // 32 MB
// The slots of `floats` partial sums in nsplit shares; 0: they do not meet by exchange.
inline size_t hq_split_slots(size_t floats, int nsplit) {
  const size_t n = nsplit > 1 && nsplit <= kHqMeetMost ? floats / nsplit * (nsplit - 1) : 0;
  return n <= kHqMostSlots ? n : 0;
}

// Packed rows that start at any multiple of four or one column (N not a multiple of 32 words): the 128-byte lines at the edges of
// a column tile belong to its neighbour too.
__host__ __device__ __forceinline__ bool hq_tiles_share_lines(const void* w, int N) { return ((N & 31) | ((int)(uintptr_t)w & 127)) != 0; }
// Column tile (or block of rows) of workgroup x of a row of ntiles workgroups.  Workgroup x runs on XCD x mod 8, so tile x would have its neighbours
// on two other XCDs, and both would fetch the lines between them from memory.  Where there are such lines an XCD takes consecutive
// tiles and finds them in its L2; where there are none the plain order stays, which spreads an XCD's reads over more of the memory.
// (ntiles from the arguments, not from gridDim: that is a load of its own ahead of every address, 0.3 us.)
__device__ __forceinline__ int hq_column_tile(int x, int ntiles, bool share_lines) {
  const int xcd = x & 7;
  return share_lines ? xcd * (ntiles >> 3) + min(xcd, ntiles & 7) + (x >> 3) : x;
}

// Raw sums of a share of K, write-through to the memory side, and back past the caches of this XCD.
typedef float hq_f4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void hq_store_share(hq_f4v* p, hq_f4v v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ hq_f4v hq_load_share(const hq_f4v* p) {  // hq_wait_shares() before the value is used
  hq_f4v v;
  asm volatile("global_load_dwordx4 %0, %1, off sc1" : "=&v"(v) : "v"(p) : "memory");
  return v;
}
template <int N>
__device__ __forceinline__ void hq_wait_shares(hq_f4v (&v)[N]) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));  // no use moves in front of the wait
}

// Streaming stores: write-through (sc1) and nontemporal (nt), i.e. the data is on its way to memory at once
// and is not kept in the L2.  For a 33.5 MB write stream on MI355X: 5.80 us against 6.46 us with nt alone
// and 7.04 us with plain stores.  The compiler cannot see that the assembly is a store, so the wait states it
// would put between a store of more than 64 bits and the next write to the data registers are part of the
// assembly.
__device__ __forceinline__ void hq_store_stream(hq_u4v* p, hq_u4v v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void hq_store_stream(hq_u2v* p, hq_u2v v) {
  asm volatile("global_store_dwordx2 %0, %1, off sc1 nt" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void hq_store_stream(uint32_t* p, uint32_t v) {
  asm volatile("global_store_dword %0, %1, off sc1 nt" ::"v"(p), "v"(v) : "memory");
}
