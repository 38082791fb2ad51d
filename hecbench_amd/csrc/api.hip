// Library-wide state of libhq: device facts, per-stream workspaces, error text.
#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "hq_internal.h"

namespace {
std::mutex g_mu;
std::map<int, HqDevice> g_devices;
constexpr int kListedDevices = 64;
std::atomic<const HqDevice*> g_known[kListedDevices];  // entries of g_devices that are gfx950 parts
std::map<std::pair<int, hipStream_t>, HqWorkspace> g_workspaces;
std::map<std::pair<int, hipStream_t>, HqWorkspace> g_eager;  // of hq_get_eager_workspace
// Counters that a workspace begins with.  With exchange slots for every batch (8192 rows of partial sums) and up to 75,000 columns they
// grow no later than the partial sums: an allocation is an error while any other stream is being captured.
constexpr size_t kLeastCounters = (size_t)1 << 20;
std::vector<std::pair<int, void*>> g_retired;  // outgrown buffers, freed by hq_shutdown()
}  // namespace

// ---- launch-shape overrides ------------------------------------------------------------------
// Every knob is an int that is "unset" by default.  The environment variable of the same name is
// read ONCE (first use), hq_set_tunable() changes a knob at run time; a launch path reads a knob
// with one relaxed atomic load, never the environment.
namespace {
const char* const kTunableNames[HQ_TUNE_COUNT] = {
    "HQ_Q3_WAVES", "HQ_Q3_STEPS", "HQ_Q3_KSPLIT", "HQ_Q3_TILE", "HQ_Q3_SMALL_BATCH", "HQ_Q3_ROW_BLOCKS", "HQ_LUT_PATH", "HQ_LUT_KSPLIT", "HQ_NF4_PIPE",
    "HQ_AQLM_ROWS", "HQ_Q8_WGS", "HQ_Q8_FAST", "HQ_GEMV_LDS", "HQ_GEMV_SPLIT", "HQ_SPLITK_FENCES", "HQ_Q3_TILES", "HQ_LUT_FINE"};
constexpr int kUnset = INT_MIN;
std::atomic<int> g_tunables[HQ_TUNE_COUNT];
std::once_flag g_tunables_once;

void seed_tunables_from_env() {
  for (int i = 0; i < HQ_TUNE_COUNT; ++i) {
    int v = kUnset;
    const char* e = std::getenv(kTunableNames[i]);
    if (e && *e) {
      char* end = nullptr;
      const long r = std::strtol(e, &end, 10);
      if (end && *end == '\0') v = (int)r;
    }
    g_tunables[i].store(v, std::memory_order_relaxed);
  }
}
}  // namespace

int hq_tune(HqTunable id, int dflt) {
  std::call_once(g_tunables_once, seed_tunables_from_env);
  const int v = g_tunables[id].load(std::memory_order_relaxed);
  return v == kUnset ? dflt : v;
}

extern "C" int hq_set_tunable(const char* name, int value, int clear) {
  if (!name) return HQ_ERR_NULL_POINTER;
  std::call_once(g_tunables_once, seed_tunables_from_env);
  for (int i = 0; i < HQ_TUNE_COUNT; ++i)
    if (std::strcmp(name, kTunableNames[i]) == 0) {
      g_tunables[i].store(clear ? kUnset : value, std::memory_order_relaxed);
      return HQ_OK;
    }
  return HQ_ERR_BAD_ENUM;
}

int hq_current_device(const HqDevice** out) {
  int dev = 0;
  HQ_HIP_TRY(hipGetDevice(&dev));
  // every call passes here: a device seen before costs one load, no lock (map nodes stay where they are)
  const bool listed = dev >= 0 && dev < kListedDevices;
  if (listed) {
    if (const HqDevice* known = g_known[dev].load(std::memory_order_acquire)) {
      *out = known;
      return HQ_OK;
    }
  }
  std::lock_guard<std::mutex> lk(g_mu);
  auto it = g_devices.find(dev);
  if (it == g_devices.end()) {
    hipDeviceProp_t p;
    HQ_HIP_TRY(hipGetDeviceProperties(&p, dev));
    HqDevice d;
    d.ordinal = dev;
    d.cus = p.multiProcessorCount;
    d.lds_per_cu = (int)p.maxSharedMemoryPerMultiProcessor;
    d.ok = std::strncmp(p.gcnArchName, "gfx950", 6) == 0 && p.warpSize == 64;
    it = g_devices.emplace(dev, d).first;
  }
  if (!it->second.ok) return HQ_ERR_UNSUPPORTED_DEVICE;
  *out = &it->second;
  if (listed) g_known[dev].store(&it->second, std::memory_order_release);
  return HQ_OK;
}

namespace {
// Device memory whose first `zero` bytes are zero when this returns: nothing of it is left to a caller's stream, so a graph that was captured on one stream and
// is replayed on another finds it zero whatever its own stream has still to do.  Cleared on a stream of the library's own: the
// default stream may not be touched while another is being captured.
std::map<int, hipStream_t> g_fill;  // per device
hipError_t alloc_zeroed(int dev, void** p, size_t bytes, size_t zero) {
  hipStream_t& fill = g_fill[dev];
  hipError_t e = fill ? hipSuccess : hipStreamCreateWithFlags(&fill, hipStreamNonBlocking);
  if (e != hipSuccess) {
    fill = nullptr;
    return e;
  }
  e = hipMalloc(p, bytes);
  if (e != hipSuccess) return e;
  e = hipMemsetAsync(*p, 0, zero, fill);
  if (e == hipSuccess) e = hipStreamSynchronize(fill);
  if (e != hipSuccess) (void)hipFree(*p);
  return e;
}
// Around the allocations of a call on a stream that is not being captured: they do not make a capture invalid that another stream is
// in the middle of.  (On a stream that is, an allocation stays the error that it is.)
struct BesideCaptures {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  bool exchanged = false;
  explicit BesideCaptures(hipStream_t stream) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone)
      exchanged = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    else
      (void)hipGetLastError();
  }
  ~BesideCaptures() {
    if (exchanged) (void)hipThreadExchangeStreamCaptureMode(&mode);
  }
};
}  // namespace

int hq_get_workspace(hipStream_t stream, size_t need_floats, size_t need_counters, HqWorkspace* out, size_t want_slots,
                     bool reserve) {
  int dev = 0;
  HQ_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_mu);
  HqWorkspace& ws = g_workspaces[std::make_pair(dev, stream)];
  if (ws.partial_floats < need_floats) {
    // grow geometrically: a stream that sees larger and larger problems allocates O(log) times; a reservation names the largest
    size_t n = ws.partial_floats ? ws.partial_floats * 2 : (size_t)1 << 20;
    while (n < need_floats) n *= 2;
    if (reserve) n = need_floats;
    float* p = nullptr;
    const BesideCaptures beside(stream);
    HQ_HIP_TRY(hipMalloc((void**)&p, n * sizeof(float)));
    // kernels in flight may still read the previous buffer: it is kept until hq_shutdown()
    if (ws.partial) g_retired.push_back(std::make_pair(dev, (void*)ws.partial));
    ws.partial = p;
    ws.partial_floats = n;
  }
  size_t want = std::max(need_counters, 2 * want_slots);
  if (want > need_counters && ws.ncounters < want) {  // slots can be done without: none of them while capturing
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
      (void)hipGetLastError();
      want = need_counters;
    }
  }
  if (ws.ncounters < want) {
    size_t n = ws.ncounters ? ws.ncounters * 2 : kLeastCounters;
    while (n < want) n *= 2;
    if (reserve) n = want > (size_t)1 << 14 ? want : (size_t)1 << 14;
    unsigned* c = nullptr;
    const BesideCaptures beside(stream);
    const hipError_t e = alloc_zeroed(dev, (void**)&c, n * sizeof(unsigned), n * sizeof(unsigned));
    if (e == hipSuccess) {
      if (ws.counters) g_retired.push_back(std::make_pair(dev, (void*)ws.counters));
      ws.counters = c;
      ws.ncounters = n;
    } else {
      (void)hipGetLastError();
      if (ws.ncounters < need_counters) return (int)e;
    }
  }
  *out = ws;
  return HQ_OK;
}

int hq_get_eager_workspace(hipStream_t stream, size_t need_floats, size_t need_counters, HqWorkspace* out, bool reserve) {
  int dev = 0;
  HQ_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_mu);
  HqWorkspace& ws = g_eager[std::make_pair(dev, stream)];
  if (ws.partial_floats < need_floats || ws.ncounters < need_counters) {
    size_t n = ws.partial_floats ? ws.partial_floats * 2 : (size_t)1 << 18;
    while (n < need_floats) n *= 2;
    if (reserve) n = std::max(need_floats, ws.partial_floats);
    const size_t c = std::max(need_counters, ws.ncounters);
    // one buffer, the counters in front; not cleared on the stream, which may be in the middle of a capture where one allows
    // allocations: a reservation's memset would wait for a replay
    unsigned* p = nullptr;
    const BesideCaptures beside(stream);
    const hipError_t e = alloc_zeroed(dev, (void**)&p, (c + n) * sizeof(unsigned), c * sizeof(unsigned));
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return (int)e;
    }
    if (ws.counters) g_retired.push_back(std::make_pair(dev, (void*)ws.counters));
    ws = HqWorkspace{reinterpret_cast<float*>(p + c), p, n, c};
  }
  *out = ws;
  return HQ_OK;
}

int hq_get_split(hipStream_t stream, size_t floats, size_t counters, int nsplit, float** partial, unsigned** arrivals) {
  const size_t slots = hq_tune(HQ_TUNE_SPLITK_FENCES, 0) ? 0 : hq_split_slots(floats, nsplit);
  HqWorkspace ws;
  const int rc = hq_get_workspace(stream, floats, counters, &ws, slots);
  if (rc != HQ_OK) return rc;
  const bool meet = slots > 0 && ws.ncounters >= 2 * slots;
  *partial = meet ? reinterpret_cast<float*>(ws.counters) : ws.partial;
  *arrivals = meet ? nullptr : ws.counters;
  return HQ_OK;
}

bool hq_workspace_out_of_reach(hipStream_t stream, size_t need_floats, size_t need_counters) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_workspaces.find(std::make_pair(dev, stream));
    if (it != g_workspaces.end() && it->second.partial_floats >= need_floats && it->second.ncounters >= need_counters) return false;
  }
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(stream, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone;
}

// Upper bound of what any hq_q3_matvec call with K <= max_K, N <= max_N (any batch) and any hq_lut_gemv call
// of those sizes takes from its stream's workspace on a device of `cus` compute units, with the default launch
// policy.  Host arithmetic only.  (tests/test_workspace_cpu.py checks it against the per-call need over a
// sweep of shapes.)
static void reserve_bound(int cus, int max_K, int max_N, size_t* floats, size_t* counters) {
  // batched GEMM: re-ordered activations of 64 rows (128 bytes per input feature, K padded to 1024), the row
  // sums and scales, and - whenever some N <= max_N leaves compute units without a 128-column tile and K has
  // two or more ranges of four steps, i.e. always but for very short K - the raw sums of its K split, at most
  // 256 blocks of 64 x 128
  const size_t kpad = ((size_t)max_K + 1023) / 1024 * 1024;
  const size_t gemm_floats = kpad * 32 + 128 + (kpad >= 2048 ? (size_t)256 * 64 * 128 : 0);
  // split-K matvecs: a partial row of 64 floats per column tile and split - one split per 4096 elements of K
  // (a shorter K than max_K splits no further); narrow tiles (16 or 32 columns) only while tiles x splits stay
  // within the compute units.  The LUT kernels: two workgroups per compute unit, 128 floats each.
  const size_t tiles = ((size_t)max_N + 63) / 64;
  const size_t rounds = ((size_t)max_K + 4095) / 4096;
  const size_t full_split = tiles * rounds;
  const size_t per_cu = tiles + 2 * (size_t)cus;
  size_t split_floats = (full_split > per_cu ? full_split : per_cu) * 64 * 2;
  // and a row of 64 per tile and 1024 elements of K where those cut K finest
  const size_t finest = tiles * (((size_t)max_K + 1023) / 1024) * 64;
  if (finest > split_floats) split_floats = finest;
  // batches 2 ... 64 on the matvec-like kernel: one partial row per tile, range of K and activation row, at most
  // 8192 of them whatever the shape
  if ((size_t)8192 * 64 > split_floats) split_floats = (size_t)8192 * 64;
  *floats = gemm_floats > split_floats ? gemm_floats : split_floats;
  // many rows: the tiled kernels
  size_t tile_floats = 0, tile_counters = 0;
  hq_q3_tiles_bound(cus, max_K, &tile_floats, &tile_counters);
  if (tile_floats > *floats) *floats = tile_floats;
  // arrival counters: one per column tile, narrow tiles four per 64 columns, row blocks sixteen per tile
  *counters = tiles > 1 ? tiles * 16 : 16;
  if (tile_counters > *counters) *counters = tile_counters;
  // and the slots in which up to eight shares of K meet, two counters each: a row of 64 per column tile and share but one, of 1024
  // elements of K at least (the LUT kernels; narrow tiles of the matvec stay within the compute units) or of 4096 and for every
  // row of a batch, where partial sums take 8192 rows at most
  auto shares = [&](size_t k) { return std::min<size_t>(((size_t)max_K + k - 1) / k, kHqMeetMost); };
  size_t slots = 0;
  if (max_K > 1024) slots = tiles * (shares(1024) - 1) * 64;
  if (max_K > 4096) slots = std::max({slots, (size_t)cus * 64, std::min<size_t>(tiles * (shares(4096) - 1) * 64, 8192) * 64});
  *counters = std::max(*counters, 2 * std::min(slots, kHqMostSlots));
}
// The same of an eager hq_aqlm_matvec call of max_N rows, from memory of its own: eight sums a row, rows padded to whole groups (an
// eighth of the compute units), a counter for each group.
static void reserve_bound_eager(int cus, int max_N, size_t* floats, size_t* counters) {
  *counters = (size_t)cus / 8;
  *floats = 8 * (std::min<size_t>(max_N, 1 << 20) + *counters);
}

extern "C" int hq_reserve_need(int compute_units, int max_K, int max_N, int64_t* floats, int64_t* counters) {
  if (!floats || !counters) return HQ_ERR_NULL_POINTER;
  if (max_K < 0 || max_N < 0 || compute_units <= 0) return HQ_ERR_BAD_SHAPE;
  size_t f = 0, c = 0;
  reserve_bound(compute_units, max_K, max_N, &f, &c);
  size_t ef = 0, ec = 0;
  reserve_bound_eager(compute_units, max_N, &ef, &ec);
  *floats = (int64_t)(f + ef);
  *counters = (int64_t)(c + ec);
  return HQ_OK;
}

extern "C" int hq_reserve_workspace(void* stream, int max_K, int max_N) {
  if (max_K < 0 || max_N < 0) return HQ_ERR_BAD_SHAPE;
  const HqDevice* d = nullptr;
  int rc = hq_current_device(&d);
  if (rc != HQ_OK) return rc;
  size_t floats = 0, counters = 0;
  reserve_bound(d->cus, max_K, max_N, &floats, &counters);
  HqWorkspace ws;
  rc = hq_get_workspace((hipStream_t)stream, floats, counters, &ws, 0, true);
  if (rc != HQ_OK) return rc;
  reserve_bound_eager(d->cus, max_N, &floats, &counters);
  return hq_get_eager_workspace((hipStream_t)stream, floats, counters, &ws, true);
}

extern "C" int hq_shutdown(void) {
  HQ_HIP_TRY(hipDeviceSynchronize());
  std::lock_guard<std::mutex> lk(g_mu);
  int cur = 0;
  HQ_HIP_TRY(hipGetDevice(&cur));
  int rc = HQ_OK;
  auto release = [&](int dev, void* p) {
    if (!p) return;
    hipError_t e = hipSetDevice(dev);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipFree(p);
    if (e != hipSuccess && rc == HQ_OK) rc = (int)e;
  };
  for (auto& kv : g_workspaces) {
    release(kv.first.first, kv.second.partial);
    release(kv.first.first, kv.second.counters);
  }
  for (auto& kv : g_fill) {
    hipError_t e = kv.second ? hipSetDevice(kv.first) : hipSuccess;
    if (e == hipSuccess && kv.second) e = hipStreamDestroy(kv.second);
    if (e != hipSuccess && rc == HQ_OK) rc = (int)e;
  }
  g_fill.clear();
  for (auto& kv : g_eager) release(kv.first.first, kv.second.counters);
  for (auto& r : g_retired) release(r.first, r.second);
  g_workspaces.clear();
  g_eager.clear();
  g_retired.clear();
  (void)hipSetDevice(cur);
  return rc;
}

extern "C" int hq_abi_version(void) { return 1; }

extern "C" const char* hq_strerror(int code) {
  switch (code) {
    case HQ_OK: return "ok";
    case HQ_ERR_NULL_POINTER: return "hq: null pointer argument";
    case HQ_ERR_BAD_SHAPE: return "hq: shape argument out of range or not a multiple of the required tile";
    case HQ_ERR_BAD_ENUM: return "hq: unknown dtype / table / flag value";
    case HQ_ERR_MISALIGNED: return "hq: pointer not aligned as required";
    case HQ_ERR_UNSUPPORTED_DEVICE: return "hq: current device is not a gfx950 (MI355X) GPU";
    case HQ_ERR_TOO_LARGE: return "hq: problem exceeds the library's limits";
    default: break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "hq: unknown error code";
}

extern "C" int hq_init(void) {
  const HqDevice* d = nullptr;
  int rc = hq_current_device(&d);
  if (rc != HQ_OK) return rc;
  HqWorkspace ws;
  rc = hq_get_workspace(nullptr, 1, 1, &ws);
  if (rc != HQ_OK) return rc;
  return hq_noalloc_setup();  // this device's address of the fixed scratch of hq_q3_matvec_noalloc
}

extern "C" int hq_device_info(int* compute_units, int* wavefront_size, int* lds_bytes_per_cu,
                              int* memory_clock_khz, int* memory_bus_bits, char* name,
                              int name_len) {
  int dev = 0;
  HQ_HIP_TRY(hipGetDevice(&dev));
  hipDeviceProp_t p;
  HQ_HIP_TRY(hipGetDeviceProperties(&p, dev));
  if (compute_units) *compute_units = p.multiProcessorCount;
  if (wavefront_size) *wavefront_size = p.warpSize;
  if (lds_bytes_per_cu) *lds_bytes_per_cu = (int)p.maxSharedMemoryPerMultiProcessor;
  if (memory_clock_khz) *memory_clock_khz = p.memoryClockRate;
  if (memory_bus_bits) *memory_bus_bits = p.memoryBusWidth;
  if (name && name_len > 0) {
    std::snprintf(name, (size_t)name_len, "%s (%s)", p.name, p.gcnArchName);
  }
  return HQ_OK;
}
