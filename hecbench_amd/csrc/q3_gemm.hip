// Batched GPTQ 3-bit GEMM for gfx950 (fp16 activations, fp32 output):
//
//   out[m][n] = sum_k A[m][k] * (s[n]*q[k][n] - z[n])
//             = s[n] * sum_k A[m][k]*q[k][n]  -  z[n] * sum_k A[m][k]
//
// The reference benchmark has only the batch-1 matvec
// (src/quant3MatMul-hip/kernels.h in the HeCBench tree); this is the same
// arithmetic applied to up to 64 activation rows per pass on the matrix cores.  It serves 33 to 64 rows of 9e7 weights and more that
// leave it column tiles for half the compute units or have a K of 16384, and stands in where a captured call finds room for 64 rows' activations only; fewer rows and smaller matrices go through
// q3_direct.hip, more rows through q3_prefill.hip, whose pre-pass is the one here.
//
// As in the matvec, the packed codes are never converted: an AND turns a 32-bit
// window of the packed string into two subnormal-fp16 MFMA operands
// (q3_recipe.h).  The factor 2^pos of each operand slot is folded into the
// activations by a small pre-pass that also reorders them into operand-slot order
// ([k-group][mfma j][row][8 halves]), scales every row by a power of two so that
// the fold stays inside the fp16 normal range, and computes the row sums for the
// zero term.
// The main kernel streams the weights once: a workgroup (4 waves, one per SIMD) owns 128
// output columns and all of K and walks K in steps of 8 k-groups; each wave owns two
// k-groups of a step, loads their activation slices (from L2) and packed rows (from
// HBM) straight into registers three steps ahead, and multiplies 2 k-groups x 128
// columns x 64 rows per step with 32x32x16 fp16 MFMAs (fp32 accumulate).  There is
// no LDS traffic and no barrier in the loop.  The four waves' accumulators are
// summed through LDS at the end and scale/zero are applied once per output.
#include <mutex>

#include "hq_internal.h"
#include "q3_recipe.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;       // one per SIMD, up to 512 registers each
constexpr int kStepGroups = 8;  // k-groups a workgroup consumes per step (two per wave)
constexpr int kDeep = 3;        // steps of operands in flight ahead of the one being multiplied
constexpr int kBufs = kDeep + 1;
constexpr int kChunk = kStepGroups * kBufs;  // the pre-pass pads K to a multiple of this many k-groups
constexpr int kTileN = 128;     // output columns per workgroup
constexpr int kRowBlocks = 2, kRows = 32 * kRowBlocks;  // activation rows of a pass over the weights
constexpr int kMaxSplitGroups = 256;  // workgroups of a K-split launch (tiles times splits)
constexpr int kFixedMaxK = 16384;     // longest K of a batched call in the fixed scratch

// ---- pre-pass: activations -> operand-slot order, scaled by P[m] * 2^-pos; row sums ------------
// Ap[((g*4 + j)*Mpad + m)*8 + e] = A[m][32g + k] * P[m] * 2^-pos(k) with slot(k) = 8j + e; rows >= M and
// groups >= G hold zeros.  One block per row: it finds the row's largest magnitude and sum, picks the
// power of two P[m] that puts the largest magnitude in [2^14, 2^15), and re-orders its row.  The 2^-pos
// of an operand slot (pos <= 7) then leaves every entry within 2^21 of its row's largest an fp16 normal
// number, i.e. exactly the input's mantissa; the main kernel's epilogue divides by P[m] again.  (Without
// P[m] the slot factor alone pushed activations below 2^-7 into the fp16 subnormals.)
// It also clears the arrival counters of the product behind it: they come back to zero by themselves, but a call that was cut
// short leaves some behind, with which no later call would finish those tiles.
// Every second pair of k-groups enters negated.  The matrix instruction cuts its sum towards minus infinity, a little for
// every sixteen products: with all sums of one sign that was an offset of the whole result, 95 % of its error and growing
// with K.  The kernels keep the negated pairs in accumulators of their own (odd waves, odd parts of K) and subtract those at
// the end, so that the cuts of the two halves cancel.  Error of the result against 64 bits (2-norm): 300 rows, K=4096, N=4100
// 9.1e-6 -> 1.8e-6; 128 rows, K=8192, N=2048 1.28e-5 -> 1.8e-6; 295 rows, K=1376, N=11252 5.5e-6 -> 1.8e-6; same time.
__global__ __launch_bounds__(256) void q3_gemm_prep(const _Float16* __restrict__ A, _Float16* __restrict__ Ap,
                                                   float* __restrict__ rowsum, float* __restrict__ rowinv,
                                                   int M, int K, int Mpad, int Gpad, unsigned* __restrict__ counters,
                                                   int ncounters) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int G = K >> 5;
  // Eight consecutive rows share the 128-byte lines of Ap; workgroups b, b + 8, b + 16, ... run on the same
  // XCD, so the rows of a line go to workgroups of one XCD and its L2 writes whole lines back instead of
  // eight XCDs writing an eighth of every line each.
  // (a multiple of 64 workgroups whatever Mpad; those beyond Mpad have nothing to do).
  const int m = ((int)blockIdx.x & ~63) + (blockIdx.x & 7) * 8 + ((blockIdx.x >> 3) & 7);
  if (m >= Mpad) return;
  __shared__ float s_sum[4], s_max[4];
  float sum = 0.f, amax = 0.f;
  if (m < M) {
    const u4v* src = reinterpret_cast<const u4v*>(A + (size_t)m * K);
    const int n16 = K >> 3;
    for (int i0 = 0; i0 < n16; i0 += 4 * 256) {
      u4v raw[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * 256 + (int)threadIdx.x;
        raw[u] = src[min(i, n16 - 1)];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * 256 + (int)threadIdx.x;
        const _Float16* in = reinterpret_cast<const _Float16*>(&raw[u]);
        float s8 = 0.f, m8 = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          s8 += (float)in[e];
          m8 = fmaxf(m8, fabsf((float)in[e]));
        }
        sum += i < n16 ? s8 : 0.f;
        amax = i < n16 ? fmaxf(amax, m8) : amax;
      }
    }
  }
  sum = hq_wave_sum(sum);
  amax = hq_wave_max(amax);
  if (lane == 0) { s_sum[wv] = sum; s_max[wv] = amax; }
  __syncthreads();
  amax = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
  // P = 2^(14 - floor(log2 amax)); an all-zero or non-finite row keeps P = 1 (fp16 magnitudes span 2^-24 .. 2^16)
  const int ex = (int)((__float_as_uint(amax) >> 23) & 255u) - 127;
  const int pe = (amax > 0.f && ex < 128) ? 14 - ex : 0;
  if (threadIdx.x == 0) {
    rowsum[m] = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
    rowinv[m] = __uint_as_float((uint32_t)(127 - pe) << 23);
  }
  // second pass over the row (it is in the caches now): thread = k-group
  for (int g = threadIdx.x; g < Gpad; g += 256) {
    _Float16 out[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) out[i] = (_Float16)0.f;
    if (m < M && g < G) {
      const u4v* src = reinterpret_cast<const u4v*>(A + (size_t)m * K + 32 * g);
      u4v raw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) raw[i] = src[i];
      const _Float16* in = reinterpret_cast<const _Float16*>(raw);
#pragma unroll
      for (int k = 0; k < 32; ++k)
        out[hq_q3::slot_of(k)] =
            (_Float16)((float)in[k] * __uint_as_float((uint32_t)(127 + pe - hq_q3::pos_of(k)) << 23 | (uint32_t)(g & 2) << 30));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u4v* dst = reinterpret_cast<u4v*>(Ap + ((size_t)(g * 4 + j) * Mpad + m) * 8);
      *dst = *reinterpret_cast<const u4v*>(out + 8 * j);
    }
  }
  for (int i = m * 256 + (int)threadIdx.x; i < ncounters; i += Mpad * 256) counters[i] = 0u;
}

// Sixteen two-field registers of one column's k-group (see q3_recipe.h).
__device__ __forceinline__ void unpack16(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t (&a)[16]) {
  using namespace hq_q3;
  const uint32_t win[7] = {w0,
                           __builtin_amdgcn_alignbit(w1, w0, 4),
                           __builtin_amdgcn_alignbit(w1, w0, 10),
                           w1,
                           __builtin_amdgcn_alignbit(w2, w1, 9),
                           w2,
                           w2 >> 7};
#pragma unroll
  for (int r = 0; r < 16; ++r) a[r] = win[kRecipe[r].window] & mask_of(r);
}

struct GemmArgs {
  const uint32_t* w;
  const u4v* Ap;        // [Gpad][4][Mpad] 16-byte operand chunks
  const float* rowsum;  // [Mpad]
  const float* rowinv;  // [Mpad] 1 / P[m]
  const float* scales;
  const float* zeros;
  float* out;           // [M][N]
  float* partial;       // K split: [tile][split][Mpad][128] raw sums of a workgroup
  unsigned* counters;   // and the workgroups of each tile that have left theirs; null: q3_gemm_reduce adds them
  int M, K, N, Gpad;
  int nsplit, spp;      // workgroups per column tile, steps per workgroup (a multiple of kBufs)
  unsigned flags;
};

// ---- main kernel -----------------------------------------------------------------------------------
// One wave per SIMD with up to 512 registers (the accumulators of 64 rows x 128 columns take 128 of them,
// in the accumulation registers), kDeep steps of operands in flight.  The buffers rotate by unrolling,
// never by copying: a register move out of a buffer whose load is still in flight would wait for it.
// (Two waves per SIMD with one step in flight measured 38.4 us at M=64, K=8192, N=28672 against 36.2; the
// depth itself, 2 to 5 steps, changes little: what a workgroup moves through its CU's L1 - all of the
// re-ordered activations, 1 MB, next to 0.4 MB of weights - bounds the loop, not the latency.)
// SHARED: column tiles share 128-byte lines (hq_column_tile; a kernel of its own, so that nothing stands in front of the other's
// first loads).
template <bool SHARED>
__global__ __launch_bounds__(kWaves * 64) void q3_gemm_kernel(const uint32_t* w_, const u4v* Ap_, int M_, int K_, int N_,
                                                             int Gpad_, int nsplit_, int spp_, unsigned flags_,
                                                             const float* scales_, const float* zeros_,
                                                             const float* rowsum_, const float* rowinv_, float* out_,
                                                             float* partial_, unsigned* counters_) {
  // leading scalars, not the struct: the first 14 dwords of the arguments arrive preloaded in scalar registers
  GemmArgs a;
  a.w = w_; a.Ap = Ap_; a.rowsum = rowsum_; a.rowinv = rowinv_; a.scales = scales_; a.zeros = zeros_; a.out = out_;
  a.partial = partial_; a.counters = counters_; a.M = M_; a.K = K_; a.N = N_; a.Gpad = Gpad_; a.nsplit = nsplit_; a.spp = spp_; a.flags = flags_;
  constexpr int MB = kRowBlocks, Mpad = kRows;
  extern __shared__ u4v lds[];  // used by the final reduction only
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int nl = lane & 31, kb = lane >> 5;
  const int G = a.K >> 5;
  // K split: workgroup (tile, split) takes steps t_begin .. t_begin + nsteps - 1 (both multiples of kBufs:
  // Gpad is a multiple of 32 k-groups) and the last of the tile to arrive, or q3_gemm_reduce, adds them up
  const int t_begin = blockIdx.y * a.spp;
  const int nsteps = min(a.spp, a.Gpad / kStepGroups - t_begin);
  const int tile = SHARED ? hq_column_tile(blockIdx.x, (a.N + kTileN - 1) / kTileN, true) : (int)blockIdx.x;
  const int col0 = tile * kTileN;
  const int col = min(col0 + 4 * nl, a.N - 4);
  const size_t row_stride = (size_t)a.N;
  const int n_out = col0 + 4 * nl;
  f4v sc = {0.f, 0.f, 0.f, 0.f}, zr = {0.f, 0.f, 0.f, 0.f};
  if (n_out < a.N) {
    sc = *reinterpret_cast<const f4v*>(a.scales + n_out);
    zr = *reinterpret_cast<const f4v*>(a.zeros + n_out);
  }
  // final reduction: a wave finishes rows 8*wv .. 8*wv+7 of every 32-row block, half wave kb four of them
  float rs[MB][4], ri[MB][4];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      rs[mb][j] = a.rowsum[mb * 32 + 8 * wv + 4 * kb + j];
      ri[mb][j] = a.rowinv[mb * 32 + 8 * wv + 4 * kb + j] * 16777216.f;  // 2^24: the unit of the code operands
    }

  f16v acc[MB][4];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mb][q][i] = 0.f;

  const u4v* ap_lane = a.Ap + (size_t)((2 * wv + kb) * 4) * Mpad + nl;
  auto load_step = [&](int tl, u4v (&A)[4][MB], uint32_t (&wr)[3][4]) {
    const int t = t_begin + tl;
    const int g = min(t * kStepGroups + 2 * wv + kb, G - 1);  // padded groups: any valid weights, zero activations
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const u4v v = __builtin_nontemporal_load(
          reinterpret_cast<const u4v*>(a.w + (size_t)(3 * g + j) * row_stride + col));
      wr[j][0] = v.x; wr[j][1] = v.y; wr[j][2] = v.z; wr[j][3] = v.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) A[j][mb] = ap_lane[(size_t)t * (kStepGroups * 4 * Mpad) + j * Mpad + mb * 32];
  };
  auto compute = [&](const u4v (&A)[4][MB], const uint32_t (&wr)[3][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t f[16];
      unpack16(wr[0][q], wr[1][q], wr[2][q], f);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u4v bv = {f[4 * j], f[4 * j + 1], f[4 * j + 2], f[4 * j + 3]};
        const h8 B = __builtin_bit_cast(h8, bv);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          acc[mb][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, A[j][mb]), B, acc[mb][q], 0, 0, 0);
      }
    }
  };

  u4v Ab[kBufs][4][MB];
  uint32_t wb[kBufs][3][4];
#pragma unroll
  for (int b = 0; b < kDeep; ++b) load_step(min(b, nsteps - 1), Ab[b], wb[b]);
  for (int t0 = 0; t0 < nsteps; t0 += kBufs) {
#pragma unroll
    for (int b = 0; b < kBufs; ++b) {
      // step t0 + b is multiplied from buffer b while step t0 + b + kDeep goes into the buffer freed one
      // step ago (the last trips re-read the last step instead of branching)
      load_step(min(t0 + b + kDeep, nsteps - 1), Ab[(b + kDeep) % kBufs], wb[(b + kDeep) % kBufs]);
      __builtin_amdgcn_sched_barrier(0);
      compute(Ab[b], wb[b]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __syncthreads();

  float* red = reinterpret_cast<float*>(lds);
  constexpr int REGION = 32 * kTileN;
  auto share = [&](int split, int m) {  // this lane's raw sums of row m
    return reinterpret_cast<f4v*>(a.partial + (((size_t)tile * a.nsplit + split) * Mpad + m) * kTileN) + nl;
  };
  auto finish = [&](f4v v, int mb, int j) {
    const int m = mb * 32 + 8 * wv + 4 * kb + j;
    if (m >= a.M || n_out >= a.N) return;
    f4v o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = sc[e] * (v[e] * ri[mb][j]) - zr[e] * rs[mb][j];
    f4v* dst = reinterpret_cast<f4v*>(a.out + (size_t)m * a.N + n_out);
    if (a.flags & HQ_FLAG_ACCUMULATE) { const f4v old = *dst; o += old; }
    *dst = o;
  };
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    if (mb) __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int r = (i >> 2) * 8 + kb * 4 + (i & 3);
      const f4v v = {acc[mb][0][i], acc[mb][1][i], acc[mb][2][i], acc[mb][3][i]};
      *reinterpret_cast<f4v*>(red + (size_t)wv * REGION + r * kTileN + 4 * nl) = v;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int r = 8 * wv + 4 * kb + j;
      const int m = mb * 32 + r;
      f4v v = *reinterpret_cast<const f4v*>(red + r * kTileN + 4 * nl);
#pragma unroll
      for (int w = 1; w < kWaves; ++w) {  // odd waves' k-groups are the negated ones (see the pre-pass)
        const f4v part = *reinterpret_cast<const f4v*>(red + (size_t)w * REGION + r * kTileN + 4 * nl);
        v = w & 1 ? v - part : v + part;
      }
      if (a.nsplit > 1) {
        hq_store_share(share(blockIdx.y, m), v);
      } else {
        finish(v, mb, j);
      }
    }
  }
  if (a.nsplit == 1 || !a.counters) return;
  // Every wave waits for the acknowledgement of its write-through stores, the workgroup counts itself at the memory side,
  // and the last of the tile adds the raw sums in split order, four splits' loads in flight.  (As a kernel of its own this took
  // 3.4 to 5.1 us and a launch: 64 rows, K=4096, N=11008, which the one-launch kernel has taken over since, 19.9 -> 18.5 us; with eight
  // splits of 64 rows, 256 KB for one workgroup, the kernel of its own stays ahead, 24.4 against 25.4 at K=16384, N=4096.)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();  // also: nobody reads the waves' sums in LDS any more
  unsigned* flag = reinterpret_cast<unsigned*>(lds);
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(&a.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = old == (unsigned)(a.nsplit - 1);
    if (old == (unsigned)(a.nsplit - 1))  // ready for the next call
      __hip_atomic_store(&a.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!*flag) return;
  constexpr int F = 4 * MB, AT_ONCE = 4;
  f4v sum[F];
#pragma unroll
  for (int i = 0; i < F; ++i) sum[i] = f4v{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.nsplit; s0 += AT_ONCE) {
    f4v x[AT_ONCE * F];
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k)
#pragma unroll
      for (int i = 0; i < F; ++i)
        x[k * F + i] = hq_load_share(share(min(s0 + k, a.nsplit - 1), (i >> 2) * 32 + 8 * wv + 4 * kb + (i & 3)));
    hq_wait_shares(x);
#pragma unroll
    for (int k = 0; k < AT_ONCE; ++k)
      if (s0 + k < a.nsplit) {
#pragma unroll
        for (int i = 0; i < F; ++i) sum[i] += x[k * F + i];
      }
  }
#pragma unroll
  for (int i = 0; i < F; ++i) finish(sum[i], i >> 2, i & 3);
}

// K split: sums the workgroups' raw sums of a tile in split order and applies scale, zero and the row's power
// of two.  A thread owns four adjacent columns of one row.
__global__ __launch_bounds__(256) void q3_gemm_reduce(GemmArgs a) {
  constexpr int Mpad = kRows;
  const int tile = blockIdx.x;
  const int nl = threadIdx.x & 31;
  const int n_out = tile * kTileN + 4 * nl;
  if (n_out >= a.N) return;
  const f4v sc = *reinterpret_cast<const f4v*>(a.scales + n_out);
  const f4v zr = *reinterpret_cast<const f4v*>(a.zeros + n_out);
  for (int m = blockIdx.y * 8 + (threadIdx.x >> 5); m < a.M; m += gridDim.y * 8) {
    const float* p = a.partial + (((size_t)tile * a.nsplit) * Mpad + m) * kTileN + 4 * nl;
    f4v v = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < a.nsplit; s0 += 8) {  // eight loads in flight, added in split order
      f4v t[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int s = s0 + j < a.nsplit ? s0 + j : a.nsplit - 1;
        t[j] = __builtin_nontemporal_load(reinterpret_cast<const f4v*>(p + (size_t)s * Mpad * kTileN));
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < a.nsplit) v += t[j];
    }
    const float ri = a.rowinv[m] * 16777216.f, rs = a.rowsum[m];
    f4v o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = sc[e] * (v[e] * ri) - zr[e] * rs;
    f4v* dst = reinterpret_cast<f4v*>(a.out + (size_t)m * a.N + n_out);
    if (a.flags & HQ_FLAG_ACCUMULATE) { const f4v old = *dst; o += old; }
    *dst = o;
  }
}

template <bool SHARED>
int launch_gemm_t(const GemmArgs& a, int ntiles, hipStream_t stream) {
  const size_t smem = (size_t)kWaves * 32 * kTileN * 4;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&q3_gemm_kernel<SHARED>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  if (attr != hipSuccess) return (int)attr;
  hipLaunchKernelGGL(q3_gemm_kernel<SHARED>, dim3(ntiles, a.nsplit), dim3(kWaves * 64), smem, stream, a.w, a.Ap, a.M, a.K,
                     a.N, a.Gpad, a.nsplit, a.spp, a.flags, a.scales, a.zeros, a.rowsum, a.rowinv, a.out, a.partial,
                     a.counters);
  return hq_launch_status();
}
int launch_gemm(const GemmArgs& a, hipStream_t stream) {
  const int ntiles = (a.N + kTileN - 1) / kTileN;
  const int rc = hq_tiles_share_lines(a.w, a.N) ? launch_gemm_t<true>(a, ntiles, stream) : launch_gemm_t<false>(a, ntiles, stream);
  if (rc != HQ_OK || a.nsplit == 1 || a.counters) return rc;
  hipLaunchKernelGGL(q3_gemm_reduce, dim3(ntiles, (a.M + 7) / 8 < 8 ? (a.M + 7) / 8 : 8), dim3(256), 0, stream, a);
  return hq_launch_status();
}

}  // namespace

// Launch plan of the batched GEMM (host arithmetic only; the launch, the workspace reservation and the size
// query share it).  K split: column tiles alone leave most CUs idle when N is small (N = 4096: 32 tiles), so K
// is cut into as many ranges as give every CU a workgroup (at most kMaxSplitGroups of them, which is what the
// fixed scratch of the entry point that allocates nothing holds), each range a multiple of kBufs steps; the
// workgroups leave raw sums in the workspace and the last one, or a second kernel, adds them in split order (deterministic).
namespace {
struct GemmPlan {
  int Gpad, nsplit, spp;
  size_t ap_halves, partial_floats, counters;
};
GemmPlan gemm_plan(int cus, int K, int N) {
  GemmPlan p;
  const int G = K / 32;
  p.Gpad = (G + kChunk - 1) / kChunk * kChunk;
  p.ap_halves = (size_t)p.Gpad * 4 * kRows * 8;
  const int ntiles = (N + kTileN - 1) / kTileN;
  const int nsteps = p.Gpad / kStepGroups;
  p.nsplit = (cus < kMaxSplitGroups ? cus : kMaxSplitGroups) / ntiles;
  if (p.nsplit > nsteps / kBufs) p.nsplit = nsteps / kBufs;
  if (p.nsplit < 1) p.nsplit = 1;
  p.spp = (nsteps + p.nsplit - 1) / p.nsplit;
  p.spp = (p.spp + kBufs - 1) / kBufs * kBufs;
  p.nsplit = (nsteps + p.spp - 1) / p.spp;
  p.partial_floats = p.nsplit > 1 ? (size_t)ntiles * p.nsplit * kRows * kTileN : 0;
  p.counters = p.nsplit > 1 ? (size_t)ntiles : 1;
  return p;
}
}  // namespace

int hq_q3_gemm_prep_launch(const void* A, void* Ap, float* rowsum, float* rowinv, int M, int K, int Mpad, int Gpad,
                           unsigned* counters, size_t ncounters, hipStream_t stream) {
  hipLaunchKernelGGL(q3_gemm_prep, dim3((Mpad + 63) / 64 * 64), dim3(256), 0, stream, reinterpret_cast<const _Float16*>(A),
                     reinterpret_cast<_Float16*>(Ap), rowsum, rowinv, M, K, Mpad, Gpad, counters, (int)ncounters);
  return hq_launch_status();
}

namespace {
// Which batches take the one-launch kernel (q3_direct.hip).  Up to 32 rows every one; up to 64, which are two of its row tiles, as
// long as reading the weights twice costs less than the pre-pass (9e7 weights: 63 rows, K=5984, N=13008 23.1 -> 19.8 us, but 57
// rows, K=4896, N=21956 25.5 -> 30.0), and, where the 64-row kernel has too few column tiles and cuts K, than its shares as well
// (64 rows, K=6016, N=16380 23.4 -> 19.9; 37, K=12032, N=8176 24.8 -> 21.9; 58, K=13824, N=11568 36.1 -> 34.3; 45, K=12864, N=8612 30.3 ->
// 26.2).  A K of 16384 and more stays with that kernel: 2.5e8 weights and more are as fast there (64 rows, K=32768, N=8192 45.7 / 46.4,
// K=49152, N=12288 94.7 / 106; 40, K=16384, N=8192 28.4 / 28.0), few columns are not (48, K=24576, N=4096 28.8 / 24.7).  Beyond 64 rows by the
// two estimates (over 270 timed problems of 97 and more rows the choice
// costs 0.3 % on average against the better of the two, 15 % at most).  65 to 96 rows of a narrow matrix (N <= 4096) always, where
// the 64-row kernel reads the weights twice: 78 rows, K=6880, N=584 19.5 -> 8.6.
// The plan is made only where it is looked at: by the estimates, or by the launch of a batch that the kernel serves.
bool direct_serves(int cus, int K, int N, int M, HqQ3DirectPlan* plan) {
  if (!hq_q3_direct_can(K, N)) return false;
  const bool forced = hq_q3_direct_forced();
  if (!forced && hq_tune(HQ_TUNE_Q3_TILES, -1) >= 0) return false;  // tests: the other kernels
  const bool cut = 2 * ((N + kTileN - 1) / kTileN) <= cus && K < 16384;  // the 64-row kernel would cut K
  if (!forced && M > 32 && M <= 64 && (int64_t)K * N >= (cut ? 250000000 : 90000000)) return false;
  *plan = hq_q3_direct_plan(cus, K, N, M, false);
  return forced || M <= 64 || !hq_q3_tiles_serve(N, M) || plan->us < hq_q3_tiles_us(cus, K, N, M);
}
}  // namespace

int hq_q3_gemm_kernel_of(int cus, int K, int N, int M) {
  HqQ3DirectPlan d;
  if (direct_serves(cus, K, N, M, &d)) return HQ_Q3_KERNEL_DIRECT;
  return hq_q3_tiles_serve(N, M) ? HQ_Q3_KERNEL_TILES : HQ_Q3_KERNEL_ROWS64;
}

// What the kernel of the plan takes, or the one that stands in for it where that is more.
int hq_q3_gemm_need(int cus, int K, int N, int M, size_t* floats, size_t* counters) {
  if (hq_q3_tiles_serve(N, M)) {
    hq_q3_tiles_need(cus, K, N, M, true, floats, counters);
  } else {
    const GemmPlan p = gemm_plan(cus, K, N);
    *floats = p.ap_halves / 2 + 2 * kRows + p.partial_floats;
    *counters = p.counters;
  }
  HqQ3DirectPlan d;
  if (direct_serves(cus, K, N, M, &d)) {
    if (d.partial_floats > *floats) *floats = d.partial_floats;
    if (d.counters > *counters) *counters = d.counters;
  }
  return HQ_OK;
}

int hq_q3_gemm_launch(const void* x, const int32_t* qweight, const float* scales, const float* zeros, float* y,
                      int K, int N, int M, unsigned flags, hipStream_t stream, const HqQ3Scratch* fixed) {
  if (((uintptr_t)x & 15) || (K & 7)) return HQ_ERR_MISALIGNED;
  if (((uintptr_t)scales & 15) || ((uintptr_t)zeros & 15) || ((uintptr_t)y & 15)) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  HqQ3DirectPlan direct;
  if (!(fixed && K > kFixedMaxK) && direct_serves(dev->cus, K, N, M, &direct))  // (a longer K is refused below)
    return hq_q3_direct_launch(direct, dev->cus, x, qweight, scales, zeros, y, K, N, M, 0, flags, stream, fixed);
  bool tiles = hq_q3_tiles_serve(N, M);
  if (tiles) {
    // 64 rows at a time need less: under capture without room for all rows' activations, and where the fixed array cannot hold
    // the tiles' plan (a device of more compute units than it was sized for; K beyond its limit, which is refused below)
    size_t floats, counters;
    hq_q3_tiles_need(dev->cus, K, N, M, false, &floats, &counters);
    tiles = fixed ? K <= kFixedMaxK && floats <= fixed->tiles_floats : !hq_workspace_out_of_reach(stream, floats, counters);
  }
  if (tiles) return hq_q3_tiles_launch(x, qweight, scales, zeros, y, K, N, M, flags, stream, fixed);
  const GemmPlan plan = gemm_plan(dev->cus, K, N);
  if (!fixed && hq_workspace_out_of_reach(stream, plan.ap_halves / 2 + 2 * kRows + plan.partial_floats, plan.counters) &&
      hq_q3_direct_can(K, N))  // under capture without room for these activations: none are needed there
    return hq_q3_direct_launch(hq_q3_direct_plan(dev->cus, K, N, M, false), dev->cus, x, qweight, scales, zeros, y, K, N, M, 0,
                               flags, stream, fixed);
  const int Gpad = plan.Gpad, nsplit = plan.nsplit, spp = plan.spp;
  const size_t ap_halves = plan.ap_halves, partial_floats = plan.partial_floats;
  _Float16* Ap;
  float *rowsum, *rowinv, *partial = nullptr;
  unsigned* counters;
  if (fixed) {
    if (ap_halves / 2 > fixed->partial_floats || partial_floats > fixed->sums_floats || plan.counters > fixed->ncounters) return HQ_ERR_TOO_LARGE;
    Ap = reinterpret_cast<_Float16*>(fixed->partial);
    rowsum = fixed->rows;
    rowinv = fixed->rows + kRows;
    partial = fixed->sums;
    counters = fixed->counters;
  } else {
    HqWorkspace ws;
    rc = hq_get_workspace(stream, ap_halves / 2 + 2 * kRows + partial_floats, plan.counters, &ws);
    if (rc != HQ_OK) return rc;
    Ap = reinterpret_cast<_Float16*>(ws.partial);
    rowsum = ws.partial + ap_halves / 2;
    rowinv = rowsum + kRows;
    partial = rowsum + 2 * kRows;
    counters = ws.counters;
  }
  // up to 64 rows per pass over the weights
  for (int m0 = 0; m0 < M; m0 += kRows) {
    const int Mb = M - m0 < kRows ? M - m0 : kRows;
    const _Float16* A = reinterpret_cast<const _Float16*>(x) + (size_t)m0 * K;
    rc = hq_q3_gemm_prep_launch(A, Ap, rowsum, rowinv, Mb, K, kRows, Gpad, counters, nsplit > 1 ? plan.counters : 0, stream);
    if (rc != HQ_OK) return rc;
    GemmArgs a;
    a.w = reinterpret_cast<const uint32_t*>(qweight);
    a.Ap = reinterpret_cast<const u4v*>(Ap);
    a.rowsum = rowsum;
    a.rowinv = rowinv;
    a.scales = scales;
    a.zeros = zeros;
    a.out = y + (size_t)m0 * N;
    a.M = Mb; a.K = K; a.N = N; a.Gpad = Gpad; a.flags = flags;
    a.partial = partial; a.counters = nsplit > 4 ? nullptr : counters; a.nsplit = nsplit; a.spp = spp;
    rc = launch_gemm(a, stream);
    if (rc != HQ_OK) return rc;
  }
  return HQ_OK;
}

// ---- the entry point that allocates nothing ----------------------------------------------------
// Its scratch (split-K partial sums and arrival counters of the matvec, re-ordered activations, row
// sums, row scales and K-split sums of the batched GEMM) lives in a fixed device array instead of the stream's
// workspace.  Every GPU holds its own copy of the array at its own address, resolved once per device.  It holds what the
// tiled kernels take at most (hq_q3_tiles_need, 256 compute units), so that every batch takes the kernels and the plan of
// hq_q3_matvec and returns its bits; the other paths use the front of it, within the limits they had before there were tiles.
namespace {
constexpr size_t kScratchRowBytes = 1024;                 // 256 floats
constexpr size_t kScratchCounterBytes = 64 * 1024 - kScratchRowBytes;
constexpr size_t kScratchPartialBytes = (size_t)2 << 20;  // 2 MiB: K <= 16384 batched, 8192 partial rows of 64 floats
constexpr size_t kScratchSumBytes = (size_t)kMaxSplitGroups * 64 * kTileN * sizeof(float);  // 8 MiB: the GEMM's K split
static_assert(kScratchPartialBytes == (size_t)kFixedMaxK * 64 * sizeof(_Float16), "64 rows of the longest K");
// tiles: 36 MiB of re-ordered activations, sums and scales of 8192 rows, 256 shares of 128 x 256 sums
constexpr size_t kScratchTileBytes = ((size_t)36 << 20) + 2 * 8192 * sizeof(float) + (size_t)256 * 128 * 256 * sizeof(float);
static_assert(kScratchTileBytes >= kScratchPartialBytes + kScratchSumBytes, "the other paths use the tiles' space");
constexpr size_t kScratchBytes = kScratchRowBytes + kScratchCounterBytes + kScratchTileBytes;  // 68 MiB + 128 KiB
}  // namespace
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];  // device address of `scratch` on each device, null until resolved

int scratch_of_current_device(void** out) {
  int dev = 0;
  HQ_HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return HQ_ERR_UNSUPPORTED_DEVICE;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    HQ_HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return (int)hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return HQ_OK;
}
}  // namespace

int hq_noalloc_setup(void) {
  void* p = nullptr;
  return scratch_of_current_device(&p);
}

extern "C" int hq_q3_matvec_noalloc(const void* x, int x_dtype, const int32_t* qweight, const float* scales,
                                    const float* zeros, float* y, int K, int N, int batch_M, unsigned flags,
                                    void* stream) {
  void* base = nullptr;
  int rc = scratch_of_current_device(&base);
  if (rc != HQ_OK) return rc;
  unsigned char* b = static_cast<unsigned char*>(base);
  HqQ3Scratch s;
  s.rows = reinterpret_cast<float*>(b);
  s.counters = reinterpret_cast<unsigned*>(b + kScratchRowBytes);
  s.ncounters = kScratchCounterBytes / sizeof(unsigned);
  b += kScratchRowBytes + kScratchCounterBytes;
  s.partial = reinterpret_cast<float*>(b);
  s.partial_floats = kScratchPartialBytes / sizeof(float);
  s.sums = reinterpret_cast<float*>(b + kScratchPartialBytes);
  s.sums_floats = kScratchSumBytes / sizeof(float);
  s.tiles = reinterpret_cast<float*>(b);
  s.tiles_floats = kScratchTileBytes / sizeof(float);
  return hq_q3_matvec_impl(x, x_dtype, qweight, scales, zeros, y, K, N, batch_M, flags, (hipStream_t)stream, &s);
}
