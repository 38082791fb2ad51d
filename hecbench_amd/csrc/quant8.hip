// bitsandbytes dynamic-map 8-bit quantisation for gfx950.
//
// Replaces dQuantize<0> / kQuantize<256,256> (src/quantBnB-hip/main.cu:13-130 in
// the HeCBench tree): a 7-step binary search over the sorted 256-entry code
// table followed by a midpoint comparison against the neighbour on the side of x
// (ties keep the pivot).  Bit-exact with the reference for every input.
// A lane converts four consecutive floats (one 128-bit load) into one packed 32-bit store.  A sorted
// table (the normal case, checked in the kernel) is served, in large calls, by a bucket table of thresholds built in LDS
// by every workgroup: one LDS read and about ten vector instructions per element instead of nine reads
// and over forty; any other table, and every table in small calls, by the descent itself, read from LDS in level order.
#include "hq_internal.h"

namespace {

typedef float f4v __attribute__((ext_vector_type(4)));

// The reference search (pivot 127, steps 64..1) walks a perfect binary tree over the table
// entries 0..254 whose leaves are the even indices.  Two facts make it cheap:
//  * stored level by level (node j of level k at (1 << (k-1)) - 1 + j, holding entry
//    ((2j+1) << (8-k)) - 1), the nodes one level touches are contiguous in LDS, so lanes on
//    different nodes hit different banks instead of a few banks 2^(8-k) entries apart;
//  * the bounds the reference tracks on the way down are, at the leaf p, always the
//    neighbours p+1 (the nearest ancestor above; entry 255 when p = 254) and p-1
//    (the nearest ancestor below; none when p = 0), so they need not be tracked: the leaf's two midpoints
//    lie next to each other.
// lds: [0..254] level order, [256] minus infinity, [257 + i] midpoint of entries i and i + 1.
// j4: four times the node's number in its level, the byte offset of its entry.
__device__ __forceinline__ float level_entry(const float* lds, int k, uint32_t j4) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(lds + (1u << k) - 1) + j4);
}
__device__ __forceinline__ uint32_t next_node(uint32_t j4, float x, float val) { return (j4 << 1) | (x > val ? 4u : 0u); }
// The leaf's decision, by selects: with branches on the side of x the lanes of a wave took all of them in turn.
__device__ __forceinline__ uint32_t leaf_code(const float* lds, uint32_t j4, float val, float x) {
  const float2 mid = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(lds + 256) + 2 * j4);
  const bool up = x > val;
  // ties keep the pivot (strict comparisons, src/quantBnB-hip/main.cu:47-65)
  return (j4 >> 1) + ((up & (x > mid.y)) ? 1u : 0u) - ((!up & (x < mid.x)) ? 1u : 0u);
}
__device__ __forceinline__ uint32_t quantize_one(const float* lds, float x) {
  uint32_t j4 = 0;
  float val = lds[0];
#pragma unroll
  for (int k = 1; k < 8; ++k) {
    j4 = next_node(j4, x, val);
    val = level_entry(lds, k, j4);
  }
  return leaf_code(lds, j4, val, x);
}

// ---- fast path for a sorted table ---------------------------------------------------------------
// With the table in increasing order the reference's result is a step function of x: it is the number
// of thresholds T_i = (c_i + c_i+1) / 2, i = 0..254, that x has passed, where an even i is passed by
// x > T_i and an odd i by x >= T_i (ties keep the pivot, and pivots are the even entries).  That holds
// whenever c_i < T_i < c_i+1; a gap where rounding or equal entries break it is "degenerate".
// Inputs are binned by a monotone key (the exponent and six mantissa bits of |x| + M / 4096: 64 buckets per
// binade down to M / 4096, linear below, one overflow bucket beyond the largest magnitude M; the
// sign picks one of two slots).  A bucket's entry holds the number of thresholds in lower buckets and
// the one threshold inside it (an odd i as the float just below T_i, so that every test is x > t;
// +inf if there is none), so a lookup is one 8-byte LDS read, one compare and one add.  Buckets with
// two or more thresholds, or touching a degenerate gap, carry a NaN pattern instead of a count: one
// unordered compare of that word with x finds them and the NaN inputs, and those lanes take the tree
// descent instead.

constexpr int kKeyShift = 17;       // six mantissa bits
constexpr int kMaxBuckets = 13 * 64 + 66;  // per sign: 12 binades from off to M, the linear one, a partial top, overflow
constexpr uint32_t kSlow = 0x7fc00000u;

constexpr int kThreads = 1024;  // one table for sixteen waves, two workgroups per compute unit
constexpr int kDescentThreads = 512;  // of a workgroup that only descends

struct FastTables {
  uint2 entry[2 * kMaxBuckets];  // slot 2 * idx (x >= +0) or 2 * idx + 1 (sign bit set): {threshold, count}
  uint32_t pos[256 + 2];         // place of every threshold's bucket in value order, non-decreasing; then beyond all
  float tval[256];               // the thresholds as "x > t" tests
};

// The key: |x| scaled so that M / 4096 becomes 2, plus 2, cut at `top` (the first value of the overflow bucket, where a NaN
// lands too).  Between 2 and 2^17 the exponent's low four bits count up from zero, so the bucket number is ten bits of it.
struct Key {
  float scale, top;
};
__device__ __forceinline__ uint32_t bucket_of(float y) { return (__float_as_uint(y) >> kKeyShift) & 1023u; }
__device__ __forceinline__ uint32_t bucket_slot(float x, const Key& key) {
  const float y = fminf(fmaf(fabsf(x), key.scale, 2.f), key.top);
  return __builtin_amdgcn_alignbit(bucket_of(y), __float_as_uint(x), 31);
}
// buckets in the order of the values they hold: negative overflow first, positive overflow last
__device__ __forceinline__ uint32_t slot_order(uint32_t slot, uint32_t cnt) {
  const uint32_t idx = slot >> 1;
  return (slot & 1u) ? cnt - idx : cnt + 1 + idx;
}
__device__ __forceinline__ uint32_t order_slot(uint32_t pos, uint32_t cnt) {
  return pos <= cnt ? 2 * (cnt - pos) + 1 : 2 * (pos - cnt - 1);
}

// a, b: table entries t and t + 1 of thread t (t < 255).  All threads.  The places of the thresholds' buckets are sorted, so
// a bucket finds the number of thresholds before it by bisection, and with it the one inside it, if any: eight dependent
// LDS reads and three barriers, and one table serves 1024 threads.  (Before: counting into the buckets and a scan over
// them, six barriers, in each of five workgroups of 256 threads per compute unit.)
__device__ __forceinline__ void build_fast_tables(FastTables& ft, float a, float b, const Key& key, uint32_t cnt) {
  const int t = threadIdx.x;
  const uint32_t nb = 2 * cnt + 2;  // buckets, both signs and overflows
  bool degenerate = false;
  if (t < 255) {
    float T = (b + a) * 0.5f;
    degenerate = !(a < T && T < b);
    float tv;
    if (t & 1) {  // x >= T: as x > the float just below T; a zero T must let -0 pass, so it goes to the negative side
      if (T == 0.f) T = -0.f;
      const uint32_t u = __float_as_uint(T);
      tv = T == 0.f ? __uint_as_float(0x80000001u) : __uint_as_float(T > 0.f ? u - 1 : u + 1);
    } else {      // x > T: a zero T must not let +0 pass from a higher bucket, so it goes to the positive side
      T = T + 0.f;
      tv = T;
    }
    ft.pos[t] = slot_order(bucket_slot(T, key), cnt);
    ft.tval[t] = tv;
  } else if (t < 258) {
    ft.pos[t] = 0xffffffffu;
  }
  __syncthreads();
  constexpr uint32_t kPer = (2 * kMaxBuckets + kThreads - 1) / kThreads;  // buckets per thread
  uint32_t i[kPer];  // thresholds before bucket t + k * kThreads: fewer than 256
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) i[k] = 0;
#pragma unroll
  for (uint32_t step = 128; step > 0; step >>= 1)
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) i[k] += ft.pos[i[k] + step - 1] < t + k * kThreads ? step : 0u;
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t p = t + k * kThreads;
    if (p < nb) {
      const bool one = ft.pos[i[k]] == p, two = ft.pos[i[k] + 1] == p;
      uint2 e;
      e.x = one ? __float_as_uint(ft.tval[i[k]]) : 0x7f800000u;  // +inf: x > t never holds
      e.y = two ? kSlow : i[k];
      ft.entry[order_slot(p, cnt)] = e;
    }
  }
  if (!__syncthreads_or(degenerate)) return;
  if (degenerate) {  // every input between and on the two entries is in one of their buckets
    ft.entry[bucket_slot(a, key)].y = kSlow;
    ft.entry[bucket_slot(b, key)].y = kSlow;
    if (a == 0.f || b == 0.f) ft.entry[0].y = ft.entry[1].y = kSlow;  // both zeros' buckets
  }
  __syncthreads();
}

constexpr int kAhead = 2;  // 16-byte loads of a thread and step: 64 KB of a step per compute unit, what it holds in flight

// What bounds it: HBM (5 bytes per element) behind the fixed cost of the tables, and close behind the lookups, ten vector
// operations and one random 8-byte LDS read per element.  A thread takes every gridDim.x * 1024-th quad; its first loads
// are in flight while the tables are built, and a step's go out together while the step before is converted (one by one
// as registers come free: 118 against 109 us at 2^27; four per thread: 118).
// us per call, before -> now: 10^7 11.8 -> 10.9, 2^24 16.8 -> 16.5, 2^27 109.7 -> 108.6 (6.2 TB/s).
// FAST: the bucket table, if the code table is sorted; otherwise every call descends.
template <bool FAST, int THREADS>
__global__ __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(8, 8))) void quantize8_kernel(
    const float* __restrict__ code, const float* __restrict__ A, uint8_t* __restrict__ out, int64_t n, int vec_ok) {
  __shared__ __align__(16) float s_code[512];
  const int t = threadIdx.x;
  const int64_t nquads = vec_ok ? n / 4 : 0;
  const int64_t stride = (int64_t)gridDim.x * THREADS;
  const int64_t t0 = (int64_t)blockIdx.x * THREADS + t;
  f4v v[kAhead];
  auto load = [&](int64_t i) { return __builtin_nontemporal_load(reinterpret_cast<const f4v*>(A) + (i < nquads ? i : nquads - 1)); };
  // the table first: a compute unit returns its loads in the order they were issued
  const float ct = code[min(t, 255)], cn = code[min(t + 1, 255)];
  const float M = FAST ? fmaxf(fabsf(code[0]), fabsf(code[255])) : 0.f;
  const int level = 32 - __builtin_clz((unsigned)min(t, 254) + 1);  // 1..8
  const float ordered = code[((2 * (min(t, 254) + 1 - (1 << (level - 1))) + 1) << (8 - level)) - 1];
  __builtin_amdgcn_sched_barrier(0);
  if (nquads > 0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) v[k] = load(t0 + k * stride);
  }
  __builtin_amdgcn_sched_barrier(0);
  if (t < 256) {
    s_code[t] = ordered;  // level-order slot t: entry ((2j+1) << (8-k)) - 1
    s_code[t < 255 ? 257 + t : 256] = t < 255 ? (cn + ct) * 0.5f : -__builtin_inff();
  }
  bool fast = false;
  if constexpr (FAST) {
    __shared__ __align__(16) FastTables ft;
    // the fast path wants a sorted table of finite, moderate values (midpoints cannot overflow) with a
    // usable magnitude
    Key key;
    key.scale = 8192.f / M;
    const float y_top = fmaf(M, key.scale, 2.f);
    const uint32_t cnt = bucket_of(y_top) + 1;  // index of the overflow bucket
    key.top = __uint_as_float((__float_as_uint(y_top) & ~((1u << kKeyShift) - 1)) + (1u << kKeyShift));
    fast = __syncthreads_and((ct <= cn) && fabsf(ct) <= 1e30f) && M >= 1e-30f &&
                      cnt < (uint32_t)kMaxBuckets;
    if (fast) {
      build_fast_tables(ft, ct, cn, key, cnt);
      const int64_t wave0 = t0 - (t & 63);  // the wave's first quad
      for (int64_t step = 0; wave0 + step < nquads; step += kAhead * stride) {
        // the next step's loads go out together, clamped instead of under a branch
        f4v vn[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) vn[k] = load(t0 + step + (kAhead + k) * stride);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
          const int64_t i = t0 + step + k * stride;
          if (wave0 + step + k * stride >= nquads) break;  // wave-uniform
          const float x[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
          uint32_t q[4];
          uint64_t slow = 0;
          uint2 en[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) en[e] = ft.entry[bucket_slot(x[e], key)];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            q[e] = en[e].y + (x[e] > __uint_as_float(en[e].x) ? 1u : 0u);
            // unordered: a flagged bucket or a NaN input
            slow |= __builtin_amdgcn_fcmpf(__uint_as_float(en[e].y), x[e], 8);  // FCMP_UNO
          }
          if (slow) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (q[e] > 255u || x[e] != x[e]) q[e] = quantize_one(s_code, x[e]);
          }
          if (i < nquads)
            __builtin_nontemporal_store(q[0] | (q[1] << 8) | (q[2] << 16) | (q[3] << 24), reinterpret_cast<uint32_t*>(out) + i);
        }
#pragma unroll
        for (int k = 0; k < kAhead; ++k) v[k] = vn[k];
      }
    }
  } else {
    __syncthreads();
  }
  if (!fast) {
    // The descent for a quad's four elements at a time, level by level: four independent LDS reads are in flight per level
    // instead of one dependent chain per element, the next step's loads run under them.  Vector instructions bound it,
    // three per level, and close behind the LDS reads.  Unsorted table, us per call, five workgroups of 256 threads with
    // eight elements in lockstep / 1024 threads, four elements and a branch on the leaf's side / this: 2^22 elements
    // 8.8 / 10.9 / 8.6, 10^7 16.9 / 18.9 / 14.8, 2^24 25.4 / 26.8 / 20.8, 2^27 275 / 214 / 152 (eight elements spill here:
    // 10^7 20.2).
    const int64_t wave0 = t0 - (t & 63);
    for (int64_t step = 0; wave0 + step < nquads; step += kAhead * stride) {
      f4v vn[kAhead];
      if (wave0 + step + kAhead * stride < nquads) {  // wave-uniform
#pragma unroll
        for (int k = 0; k < kAhead; ++k) vn[k] = load(t0 + step + (kAhead + k) * stride);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int64_t i = t0 + step + k * stride;
        if (wave0 + step + k * stride >= nquads) break;  // wave-uniform
        const float x[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        uint32_t j4[4], q[4];
        float val[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { j4[e] = 0; val[e] = s_code[0]; }
#pragma unroll
        for (int l = 1; l < 8; ++l) {
#pragma unroll
          for (int e = 0; e < 4; ++e) j4[e] = next_node(j4[e], x[e], val[e]);
#pragma unroll
          for (int e = 0; e < 4; ++e) val[e] = level_entry(s_code, l, j4[e]);
          __builtin_amdgcn_sched_barrier(0);  // the compiler would descend one element after the other to save registers
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = leaf_code(s_code, j4[e], val[e], x[e]);
        if (i < nquads)
          __builtin_nontemporal_store(q[0] | (q[1] << 8) | (q[2] << 16) | (q[3] << 24), reinterpret_cast<uint32_t*>(out) + i);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) v[k] = vn[k];
    }
  }
  for (int64_t e = nquads * 4 + t0; e < n; e += stride) out[e] = (uint8_t)quantize_one(s_code, A[e]);
}

}  // namespace

extern "C" int hq_quantize_dynamic8(const float* code, const float* A, uint8_t* out, int64_t n,
                                    void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (n < 0) return HQ_ERR_BAD_SHAPE;
  if (n == 0) return HQ_OK;
  if (!code || !A || !out) return HQ_ERR_NULL_POINTER;
  if (((uintptr_t)code & 3) || ((uintptr_t)A & 3)) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  const int vec_ok = !((uintptr_t)A & 15) && !((uintptr_t)out & 3);
  // Building the bucket table takes a workgroup as long as descending for some 24 elements a thread: up to 5 M elements every call
  // descends, in smaller workgroups, whatever the table (us, bucket table / descent: 2^14 elements 4.9 / 4.2, 2^18 5.75 / 4.2,
  // 2^20 5.9 / 4.6, 2^21 6.8 / 5.5, 2^22 8.2 / 7.25, 2^23 11.1 / 11.9; workgroups of 256, 512, 1024 threads: 2^20 5.0, 4.6, 4.6; 2^22
  // 7.4, 7.25, 7.8).  HQ_Q8_FAST: 1 the bucket table, 0 the descent, unset: this rule.
  constexpr int64_t kDescend = (int64_t)5 << 20;
  const int mode = hq_tune(HQ_TUNE_Q8_FAST, -1);
  const bool fast = mode < 0 ? n > kDescend : mode != 0;
  const int threads = fast ? kThreads : kDescentThreads;
  int64_t blocks = (n / 4 + threads - 1) / threads;
  // workgroups per CU (bucket table, us with one / two: 10^7 12.8 / 11.5, 2^25 31.1 / 31.0, 2^27 108.6 / 118.2): two fill the CU's queue
  // between the ends, where latency or the order of the stream counts more; the descent as many as fit
  const int per_cu = fast ? (n > kDescend && n < ((int64_t)1 << 26) ? 2 : 1) : 2048 / kDescentThreads;
  const int64_t cap = (int64_t)dev->cus * hq_tune(HQ_TUNE_Q8_WGS, per_cu);
  if (blocks > cap) blocks = cap;
  if (blocks < 1) blocks = 1;
  if (!fast)
    return hq_launch_as_is(quantize8_kernel<false, kDescentThreads>, dim3((unsigned)blocks), dim3(threads), 0, stream, code, A, out, n,
                           vec_ok);
  return hq_launch_as_is(quantize8_kernel<true, kThreads>, dim3((unsigned)blocks), dim3(threads), 0, stream, code, A, out, n, vec_ok);
}
