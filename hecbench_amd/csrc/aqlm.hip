// AQLM 1x16 code-book matvec for gfx950 (fp16 in / fp16 out).
//
// Replaces Code1x16MatVec / code1x16_matvec (src/quantAQLM-hip/main.cu:29-139
// in the HeCBench tree).
//
//   y[m] = fp16_rn( scale[m] * sum_g dot8(codebook[cb(m)][u16(codes[m][g])], x[8g..8g+7]) )
//
// One wave owns ROWS consecutive output rows, or the four waves of a workgroup share them (SPLIT).  Lane l always works on the same
// 64 activations (codes 8l..8l+7 of a 512-code chunk), so the activations live
// in registers for every row of the wave.  A row chunk is
// one 128-bit code load per lane (1 KB contiguous per wave); each code gathers a
// 16-byte code-book entry (the 1 MB code book stays L2-resident) and feeds four
// fp16 dot2 instructions with fp32 accumulation.  Lanes are combined with a
// cross-lane butterfly, the scale is applied in fp32 and the result is rounded
// to fp16 once.
#include "hq_internal.h"

namespace {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

struct AqlmArgs {
  const u4v* codes;      // [M][K/64] as 16-byte units
  const u4v* codebooks;  // 16-byte entries
  const _Float16* scales;  // nullable
  const u4v* x;          // [K/8]
  _Float16* y;
  int M, K;
  int cb_sizes[4];
  int cb_stride;  // in 16-byte units
};

__device__ __forceinline__ h2v as_h2(uint32_t v) { return __builtin_bit_cast(h2v, v); }

__device__ __forceinline__ float dot8(u4v e, u4v xv, float acc) {
  // components are copied to scalars first: bit-casting a vector element in place
  // makes the compiler read element 0 for every component
  const uint32_t e0 = e.x, e1 = e.y, e2 = e.z, e3 = e.w;
  const uint32_t x0 = xv.x, x1 = xv.y, x2 = xv.z, x3 = xv.w;
  acc = __builtin_amdgcn_fdot2(as_h2(e0), as_h2(x0), acc, false);
  acc = __builtin_amdgcn_fdot2(as_h2(e1), as_h2(x1), acc, false);
  acc = __builtin_amdgcn_fdot2(as_h2(e2), as_h2(x2), acc, false);
  acc = __builtin_amdgcn_fdot2(as_h2(e3), as_h2(x3), acc, false);
  return acc;
}

// Where the activations come from: a wave's 64 activations per lane lie 128 bytes apart, so loaded straight into registers
// (XLDS false) every load takes an address per lane, 512 of them in front of the wave's first codes.  XLDS: the workgroup
// copies x into LDS in whole lines, behind the loads of the first codes, piece i of unit u at [i][u] (the pieces an odd
// number of units apart: neither the copy's stores nor the reads meet in a bank); the next chunk's codes are loaded under
// a chunk's gathers.  4096 x 4096 12.5 -> 12.1 us, 2123 x 6272 13.8 -> 11.7, 16234 x 10496 96.7 -> 90.7 (235 G gathers/s of the
// 257-262 that the L2 takes), 28672 x 4096 with three code books 68.2 -> 62.6.
constexpr int kMaxLdsK = 24576;  // 48 KB
__host__ __device__ constexpr int aqlm_x_stride(int units) { return (units + 7) / 8 * 8 + 1; }

template <int ROWS, bool XLDS, bool SPLIT>
__global__ __launch_bounds__(256) void aqlm_matvec_kernel(HQ_ARGS24) {
  // the first 14 dwords of the arguments arrive preloaded in scalar registers: all but scales and y
  HqReader r(HQ_PASS24);
  AqlmArgs a;
  a.codes = r; a.codebooks = r; a.x = r; a.M = r; a.K = r; a.cb_stride = r;
  for (int i = 0; i < 4; ++i) a.cb_sizes[i] = r;
  a.scales = r; a.y = r;
  const int lane = threadIdx.x & 63;
  // An XCD takes consecutive row blocks: it gathers from one or two of the code books instead of all (each has 1 MB, its L2 4), and the
  // workgroups whose results share a 128-byte line of y are on one XCD, whose L2 writes the line back whole.  (Dealt out in runs of
  // eight instead, three code books: 1119 x 2496 6.9 / 5.85 us, 864 x 7360 8.4 / 7.7, 1311 x 9536 11.9 / 10.8, 7513 x 4160 20.4 / 19.9;
  // one: 778 x 4160 5.5 / 5.3, 4096 x 4096 no difference.)
  constexpr int kPerBlock = SPLIT ? ROWS : 4 * ROWS;
  // (The number of workgroups as the host has it: gridDim is a load of its own, ahead of every address.  4096 x 4096 11.3 / 11.1 us,
  // 864 x 7360 three code books 8.1 / 7.8, 512 x 1024 4.3 / 3.55.)
  const int blk = hq_column_tile(blockIdx.x, (a.M + kPerBlock - 1) / kPerBlock, true);
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row0 = (SPLIT ? blk : blk * 4 + wv) * ROWS;
  const int chunk0 = SPLIT ? wv * 64 : 0, step = SPLIT ? 256 : 64;  // units: this wave's first chunk, and to its next
  static_assert(XLDS || !SPLIT, "shared rows take their activations from LDS");
  if (!XLDS && row0 >= a.M) return;  // wave-uniform
  const int units_per_row = a.K >> 6;         // 16-byte code units (8 codes) per row; K % 64 == 0
  extern __shared__ u4v xl[];
  const int xstride = aqlm_x_stride(units_per_row);
  auto load_codes = [&](int u, u4v (&cw)[ROWS]) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const int m = min(row0 + r, a.M - 1);
      cw[r] = __builtin_nontemporal_load(a.codes + (size_t)m * units_per_row + min(u, units_per_row - 1));
    }
  };
  u4v cw[ROWS];
  load_codes(chunk0 + lane, cw);
  if (XLDS) {
    for (int t = threadIdx.x; t < units_per_row * 8; t += 256) xl[(t & 7) * xstride + (t >> 3)] = a.x[t];
    __syncthreads();
    if (!SPLIT && row0 >= a.M) return;
  }
  const u4v* cb[ROWS];
  float acc[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    const int m = min(row0 + r, a.M - 1);
    const u4v* p = a.codebooks;
    for (int j = 0; j < 4 && m >= a.cb_sizes[j]; ++j) p += a.cb_stride;
    cb[r] = p;
    acc[r] = 0.f;
  }
  for (int u0 = chunk0; u0 < units_per_row; u0 += step) {
    const int u = u0 + lane;
    u4v next[ROWS];
    if (u0 + step < units_per_row) load_codes(u + step, next);  // under this chunk's gathers
    if (u < units_per_row) {
      u4v xv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) xv[i] = XLDS ? xl[i * xstride + u] : a.x[(size_t)u * 8 + i];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        const uint32_t w[4] = {cw[r].x, cw[r].y, cw[r].z, cw[r].w};
        u4v e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t code = (w[i >> 1] >> (16 * (i & 1))) & 0xffffu;  // read as unsigned
          e[i] = cb[r][code];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[r] = dot8(e[i], xv[i], acc[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) cw[r] = next[r];
  }
  __shared__ float part[4][ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    float v = hq_wave_sum(acc[r]);
    if (SPLIT) {
      if (lane == 0) part[wv][r] = v;
    } else if (lane == 0 && row0 + r < a.M) {
      if (a.scales) v *= (float)a.scales[row0 + r];
      a.y[row0 + r] = (_Float16)v;
    }
  }
  if (SPLIT) {
    __syncthreads();
    const int row = row0 + (int)threadIdx.x;
    if (threadIdx.x < ROWS && row < a.M) {
      float v = (part[0][threadIdx.x] + part[1][threadIdx.x]) + (part[2][threadIdx.x] + part[3][threadIdx.x]);
      if (a.scales) v *= (float)a.scales[row];
      a.y[row] = (_Float16)v;
    }
  }
}

}  // namespace

extern "C" int hq_aqlm_matvec(const int16_t* codes, const void* codebooks, const void* scales,
                              const void* x, void* y, int M, int K, const int cb_a_sizes[4],
                              int cb_stride_int4, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!codes || !codebooks || !x || !y || !cb_a_sizes) return HQ_ERR_NULL_POINTER;
  if (M <= 0 || K <= 0 || (K & 63) || cb_stride_int4 < 0) return HQ_ERR_BAD_SHAPE;
  if (((uintptr_t)codes & 15) || ((uintptr_t)codebooks & 15) || ((uintptr_t)x & 15) ||
      ((uintptr_t)y & 1) || ((uintptr_t)scales & 1))
    return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;

  AqlmArgs a;
  a.codes = (const u4v*)codes; a.codebooks = (const u4v*)codebooks; a.scales = (const _Float16*)scales;
  a.x = (const u4v*)x; a.y = (_Float16*)y; a.M = M; a.K = K; a.cb_stride = cb_stride_int4;
  for (int j = 0; j < 4; ++j) a.cb_sizes[j] = cb_a_sizes[j];
  // Rows per wave, and whether the four waves of a workgroup share its rows, each with every fourth chunk of 512 codes (split).
  // What counts is gathers in flight and evenly over the compute units.  Measured (us, one / two / four rows per wave; one / two
  // split): 4096 x 4096 11.7 12.4 12.8; 13.3 12.9 - 9788 x 5440 31.3 30.9 33.1; 34.2 33.0 - 28672 x 4096 three code books 62.0 61.1
  // 62.9; 71.9 68.2 - 28672 x 16384 291 239 237; 271 248 - 1228 x 16192 25.1 23.2 39.6; 17.1 16.6 - 2472 x 11968 24.9 27.1 27.2;
  // 21.9 20.2 - 512 x 16384 12.3 17.3 28.7; 9.4 9.4 - 689 x 5184 6.8 9.1 15; 6.3 6.5.  HQ_AQLM_ROWS: 1, 2, 4; 11, 12 split
  // (rows that go through LDS only: sharing longer ones was never the choice).
  int rows = hq_tune(HQ_TUNE_AQLM_ROWS, 0);
  bool split = rows == 11 || rows == 12;
  if (split) rows -= 10;
  split = split && K <= kMaxLdsK;
  if (rows != 1 && rows != 2 && rows != 4) {
    const long waves_wanted = (long)dev->cus * 8;
    if (K > kMaxLdsK) rows = M >= 4 * waves_wanted ? 4 : (M >= 2 * waves_wanted ? 2 : 1);
    else if (K > 8192) rows = M >= 8 * waves_wanted ? 4 : 2;
    else rows = M >= 4 * waves_wanted ? 2 : 1;
    split = K <= kMaxLdsK && (K > 8192 ? M < 2 * waves_wanted : (K >= 4096 && M <= waves_wanted));
  }
  const int per_block = split ? rows : 4 * rows;
  const int blocks = (M + per_block - 1) / per_block;
  // one row per wave: four rows share what the workgroup copies, and beyond 8192 elements that takes as long as it saves
  const bool lds = K <= (rows > 1 || split ? kMaxLdsK : 8192);
  const size_t smem = lds ? (size_t)aqlm_x_stride(K >> 6) * 8 * 16 : 0;
#define HQ_AQLM_GO(R, L, S)                                                                                                \
  return hq_launch(aqlm_matvec_kernel<R, L, S>, dim3(blocks), dim3(256), smem, stream, a.codes, a.codebooks, a.x, a.M, a.K, \
                   a.cb_stride, a.cb_sizes[0], a.cb_sizes[1], a.cb_sizes[2], a.cb_sizes[3], a.scales, a.y)
#define HQ_AQLM_ROWS_GO(R) \
  { if (lds) HQ_AQLM_GO(R, true, false); else HQ_AQLM_GO(R, false, false); }
  if (rows == 4) HQ_AQLM_ROWS_GO(4)
  else if (rows == 2 && split) HQ_AQLM_GO(2, true, true);
  else if (rows == 2) HQ_AQLM_ROWS_GO(2)
  else if (split) HQ_AQLM_GO(1, true, true);
  else HQ_AQLM_ROWS_GO(1)
#undef HQ_AQLM_ROWS_GO
#undef HQ_AQLM_GO
}
