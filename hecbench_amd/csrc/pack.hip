// Device-side packers and the 4-bit blockwise quantiser: the inverses of the unpack /
// dequantise steps of the matvec kernels, so that the family round-trips on the GPU.
//
//   hq_q3_pack       codes uint8 [K][N]          -> int32 [3K/32][N]   (layout of
//                                                    src/quant3MatMul-hip/kernels.h:42-86)
//   hq_bcq_pack      signs int8 [K][nb][N]       -> uint32 [K/32][nb][N] (bit packing of
//                                                    src/lut-gemm-hip/main.cu:118-134)
//   hq_quantize_4bit fp32 / fp16 [n]             -> packed nibbles + fp32 absmax per block
//                                                    (inverse of hq_dequant_nf4; no counterpart
//                                                    in the HeCBench tree)
#include "hq_internal.h"

namespace {

__global__ __launch_bounds__(256) void q3_pack_kernel(const uint8_t* __restrict__ codes,
                                                     uint32_t* __restrict__ mat, int G, int N) {
  // thread -> (k-group g, column n); consecutive threads take consecutive columns
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)G * N) return;
  const int g = (int)(t / N), n = (int)(t % N);
  const uint8_t* src = codes + (size_t)(32 * g) * N + n;
  uint64_t lo = 0;   // bits 0..63 of the 96-bit string
  uint32_t hi = 0;   // bits 64..95
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint64_t q = src[(size_t)i * N] & 7u;
    const int bit = 3 * i;
    if (bit < 64) lo |= q << bit;
    if (bit > 61) hi |= (uint32_t)(bit >= 64 ? q << (bit - 64) : q >> (64 - bit));
  }
  uint32_t* dst = mat + (size_t)(3 * g) * N + n;
  dst[0] = (uint32_t)lo;
  dst[N] = (uint32_t)(lo >> 32);
  dst[2 * (size_t)N] = hi;
}

__global__ __launch_bounds__(256) void bcq_pack_kernel(const int8_t* __restrict__ signs,
                                                      uint32_t* __restrict__ bW, int KW, int NB, int N) {
  // thread -> (k-word, plane, column)
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per_word = (int64_t)NB * N;
  if (t >= (int64_t)KW * per_word) return;
  const int kw = (int)(t / per_word);
  const int64_t rest = t % per_word;  // = b*N + n
  const int8_t* src = signs + (size_t)(32 * kw) * per_word + rest;
  uint32_t w = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) w |= (src[(size_t)i * per_word] > 0 ? 1u : 0u) << i;
  bW[t] = w;
}

// bitsandbytes code books (same literals as the dequantiser)
__constant__ float c_q_nf4[16] = {
    -1.0f, -0.6961928009986877f, -0.5250730514526367f, -0.39491748809814453f,
    -0.28444138169288635f, -0.18477343022823334f, -0.09105003625154495f, 0.0f,
    0.07958029955625534f, 0.16093020141124725f, 0.24611230194568634f,
    0.33791524171829224f, 0.44070982933044434f, 0.5626170039176941f,
    0.7229568362236023f, 1.0f};

// Nearest NF4 code of a value normalised to [-1, 1]: the number of midpoints between
// adjacent table entries (fp32 (a+b)*0.5) that lie strictly below it, so a value exactly
// on a midpoint takes the lower code.
__device__ __forceinline__ uint32_t nearest_nf4(const float* mid, float v) {
  uint32_t c = 0;
#pragma unroll
  for (int step = 8; step > 0; step >>= 1) c += (v > mid[c + step - 1]) ? step : 0;  // mid[0..14]
  return c;
}

// FP4 (sign bit 3, magnitudes {0, 1/192, 2/3, 1, 1/3, 1/2, 1/6, 1/4}): nearest magnitude,
// ties to the smaller one; codes in increasing magnitude order are 0,1,6,7,4,5,2,3.
__device__ __forceinline__ uint32_t nearest_fp4(float v) {
  const float a = fabsf(v);
  const float mags[8] = {0.0f, 0.005208333333f, 0.16666667f, 0.25f, 0.33333333f, 0.5f, 0.66666667f, 1.0f};
  const uint32_t code_of[8] = {0, 1, 6, 7, 4, 5, 2, 3};
  uint32_t idx = 0;
#pragma unroll
  for (int i = 0; i < 7; ++i) idx += (a > (mags[i] + mags[i + 1]) * 0.5f) ? 1u : 0u;
  return code_of[idx] | (v < 0.f ? 8u : 0u);
}

// Any even blocksize, any alignment: one wave per block of `blocksize` elements, absmax by a cross-lane butterfly, then one
// packed byte (two codes) per lane and stride of 64.
template <typename T>
__global__ __launch_bounds__(256) void quantize4_kernel(const T* __restrict__ x, uint8_t* __restrict__ packed,
                                                       float* __restrict__ absmax, int64_t n, int blocksize,
                                                       int table) {
  __shared__ float mid[16];
  if (threadIdx.x < 15) mid[threadIdx.x] = (c_q_nf4[threadIdx.x] + c_q_nf4[threadIdx.x + 1]) * 0.5f;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int64_t block = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t e0 = block * blocksize;
  if (e0 >= n) return;  // wave-uniform
  const int64_t e1 = e0 + blocksize < n ? e0 + blocksize : n;
  float amax = 0.f;
  for (int64_t e = e0 + lane; e < e1; e += 64) amax = fmaxf(amax, fabsf((float)x[e]));
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) amax = fmaxf(amax, __shfl_xor(amax, m));
  if (lane == 0) absmax[block] = amax;
  const float inv = amax > 0.f ? 1.0f / amax : 0.f;
  // pairs of elements -> one byte, high nibble first; blocksize is even so pairs never straddle blocks
  for (int64_t p = e0 / 2 + lane; 2 * p < e1; p += 64) {
    const float v0 = (float)x[2 * p] * inv;
    const bool has1 = 2 * p + 1 < n;  // odd n: the last low nibble is padding and stays 0
    const float v1 = has1 ? (float)x[2 * p + 1] * inv : 0.f;
    const uint32_t c0 = table ? nearest_fp4(v0) : nearest_nf4(mid, v0);
    const uint32_t c1 = has1 ? (table ? nearest_fp4(v1) : nearest_nf4(mid, v1)) : 0u;
    packed[p] = (uint8_t)((c0 << 4) | c1);
  }
}

// ---- the 4-bit quantiser's main path ---------------------------------------------------------------------------------
// Power-of-two blocks of 8 to 4096 elements.  A lane owns units of eight consecutive elements (one or two 128-bit
// loads, one packed dword out), a wave owns UNITS of them 512 elements apart, so a block lies within one workgroup: blocks
// up to 512 elements are blocksize / 8 lanes of one unit, longer ones all lanes of blocksize / 512 units of one to four waves.  The
// input is read once and stays in registers between the maximum and the codes.
//
// What bounds it: HBM, if the code search stays under 14 lane operations per fp16 element (45 M elements in the 17 us
// their bytes take).  The search is one LDS read: 32 equal cells over the table's range are narrower than the distance
// of any two decision thresholds, so a cell holds at most one, and the code is the cell's base code plus one compare.
// The cell of a threshold is computed with the very operations that find the cell of a value, and both are monotone,
// so every value gets the code the thresholds define, whatever the rounding.  32 cells of 8 bytes are one entry per
// bank pair: no LDS conflicts beyond equal addresses, which broadcast.
// Measured, 4096 x 11008, blocksize 64, NF4: fp16 203 -> 18.9 us (6.1 TB/s), fp32 33.9 us (6.1 TB/s).  Before: a wave per block, one or two elements per lane, a four-step search in LDS per element.
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));

// Maximum over groups of `lanes` (1, 2, 4, ... 64; wave-uniform) adjacent lanes; every lane of a group gets it.
__device__ __forceinline__ float group_max(float v, int lanes) {
  if (lanes >= 2) v = fmaxf(v, hq_dpp<0xB1>(v));    // quad_perm [1,0,3,2]
  if (lanes >= 4) v = fmaxf(v, hq_dpp<0x4E>(v));    // quad_perm [2,3,0,1]
  if (lanes >= 8) v = fmaxf(v, hq_dpp<0x141>(v));   // row_half_mirror
  if (lanes >= 16) v = fmaxf(v, hq_dpp<0x140>(v));  // row_mirror
  if (lanes >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  if (lanes >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  }
  return v;
}

struct Cell {
  float threshold;  // +inf where the cell holds none
  uint32_t base;    // thresholds in lower cells
};
constexpr int kCells = 32;

// Byte offset of the cell of a normalised value.  NF4 values span [-1, 1], FP4 magnitudes [0, 1] (a quotient may exceed
// the ends by a rounding).  SAFE: v may be NaN or infinite (cell 0, as no threshold lies below a NaN; the last cell
// for +inf).  Otherwise adding 2^20 leaves the position in cells at bit 3 and up of the sum.
template <bool NF4, bool SAFE>
__device__ __forceinline__ uint32_t cell_of(float v) {
  const float scale = NF4 ? 15.5f : 31.f, mid = NF4 ? 16.f : 0.5f;
  if (SAFE) return (uint32_t)fminf(fmaxf(fmaf(v, scale, mid), 0.f), (float)(kCells - 1)) * 8u;
  return __float_as_uint(fmaf(v, scale, mid + 1048576.f - 0.5f)) & 0xf8u;
}

template <bool NF4, bool SAFE>
__device__ __forceinline__ void build_cells(Cell* cells) {
  const int t = threadIdx.x;
  if (t < kCells) {
    constexpr float fp4_mags[8] = {0.0f, 0.005208333333f, 0.16666667f, 0.25f, 0.33333333f, 0.5f, 0.66666667f, 1.0f};
    constexpr int n = NF4 ? 15 : 7;
    uint32_t below = 0;
    float mine = __builtin_inff();
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const float thr = NF4 ? (c_q_nf4[i] + c_q_nf4[i + 1]) * 0.5f : (fp4_mags[i] + fp4_mags[i + 1]) * 0.5f;
      const uint32_t c = cell_of<NF4, SAFE>(thr) >> 3;
      below += c < (uint32_t)t ? 1u : 0u;
      mine = c == (uint32_t)t ? thr : mine;
    }
    cells[t].threshold = mine;
    cells[t].base = below;
  }
}

template <typename T>
struct Unit8;  // eight elements of a lane
template <>
struct Unit8<_Float16> {
  u4v w;
  __device__ void load(const _Float16* p) { w = *reinterpret_cast<const u4v*>(p); }
  __device__ void load_part(const _Float16* p, int n) {
    _Float16 e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = i < n ? p[i] : (_Float16)0.f;
    w = *reinterpret_cast<const u4v*>(e);
  }
  __device__ float amax() const {
    h2v m = {(_Float16)0.f, (_Float16)0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(h2v, w[i] & 0x7fff7fffu));
    return fmaxf((float)m.x, (float)m.y);
  }
  __device__ float operator[](int i) const {
    const uint32_t pair = w[i >> 1];
    return (float)__builtin_bit_cast(h2v, pair)[i & 1];
  }
};
template <>
struct Unit8<float> {
  float v[8];
  __device__ void load(const float* p) {
    *reinterpret_cast<u4v*>(v) = *reinterpret_cast<const u4v*>(p);
    *reinterpret_cast<u4v*>(v + 4) = *reinterpret_cast<const u4v*>(p + 4);
  }
  __device__ void load_part(const float* p, int n) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = i < n ? p[i] : 0.f;
  }
  __device__ float amax() const {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[i]));
    return m;
  }
  __device__ float operator[](int i) const { return v[i]; }
};

// UNITS units per lane.  SPAN: the waves that share a block (blocksize = 512 * UNITS * SPAN), one, two or all four; 0: a block is
// `lanes` = blocksize / 8 lanes of a unit.
template <typename T, bool NF4, int UNITS, int SPAN>
__global__ __launch_bounds__(256) void quantize4_units_kernel(const T* __restrict__ x, uint8_t* __restrict__ packed,
                                                             float* __restrict__ absmax, int64_t n, int shift, int lanes) {
  // fp16: 1 / amax is finite and quotients are infinite or NaN only where an input is, which zeroes 1 / amax
  // (inf * 0: a NaN of the default pattern, and fp16 payloads end above the cell's bits: cell 0)
  constexpr bool SAFE = sizeof(T) == 4;
  __shared__ Cell cells[kCells];
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  const int64_t e0 = ((int64_t)blockIdx.x * 4 + wv) * (512 * UNITS) + lane * 8;
  Unit8<T> u[UNITS];
#pragma unroll
  for (int i = 0; i < UNITS; ++i) {
    const int64_t e = e0 + 512 * i;
    if (e + 8 <= n) u[i].load(x + e);
    else u[i].load_part(x + e, (int)(n - e > 0 ? n - e : 0));
  }
  build_cells<NF4, SAFE>(cells);
  if (SPAN <= 1) __syncthreads();
  float am[UNITS];
#pragma unroll
  for (int i = 0; i < UNITS; ++i) am[i] = u[i].amax();
  if (SPAN) {
#pragma unroll
    for (int i = 1; i < UNITS; ++i) am[0] = fmaxf(am[0], am[i]);
    am[0] = group_max(am[0], 64);
    if (SPAN > 1) {
      __shared__ float wave_max[4];
      if (lane == 0) wave_max[wv] = am[0];
      __syncthreads();
#pragma unroll
      for (int w = 1; w < SPAN; ++w) am[0] = fmaxf(am[0], wave_max[wv ^ w]);
    }
#pragma unroll
    for (int i = 1; i < UNITS; ++i) am[i] = am[0];
  } else {
#pragma unroll
    for (int i = 0; i < UNITS; ++i) am[i] = group_max(am[i], lanes);
  }
  const char* tab = reinterpret_cast<const char*>(cells);
#pragma unroll
  for (int i = 0; i < UNITS; ++i) {
    const int64_t e = e0 + 512 * i;
    if (e >= n) continue;
    if ((lane & (lanes - 1)) == 0 && (!SPAN || i == 0) && (SPAN <= 1 || wv % SPAN == 0)) absmax[e >> shift] = am[i];
    const float inv = am[i] > 0.f ? 1.0f / am[i] : 0.f;
    uint32_t word = 0, sign = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int at = (k ^ 1) * 4;  // high nibble of a byte first
      const float v = u[i][k] * inv;
      const float m = NF4 ? v : fabsf(v);
      const Cell c = *reinterpret_cast<const Cell*>(tab + cell_of<NF4, SAFE>(m));
      word |= (c.base + (m > c.threshold ? 1u : 0u)) << at;
      if (!NF4) sign |= (v < 0.f ? 8u : 0u) << at;
    }
    // FP4 codes in increasing magnitude order are 0,1,6,7,4,5,2,3: bit 2 flips where bit 1 is set
    if (!NF4) word = (word ^ ((word & 0x22222222u) << 1)) | sign;
    if (e + 8 <= n) {
      hq_store_stream(reinterpret_cast<uint32_t*>(packed) + (e >> 3), word);
    } else {
      const int left = (int)(n - e);
      for (int b = 0; 2 * b < left; ++b) {  // odd n: the last low nibble is padding and stays 0
        const uint32_t byte = (word >> (8 * b)) & 255u;
        packed[e / 2 + b] = (uint8_t)(2 * b + 1 < left ? byte : byte & 0xf0u);
      }
    }
  }
}

template <typename T, int UNITS, int SPAN>
int launch_quantize4_units(const T* x, uint8_t* packed, float* absmax, int64_t n, int blocksize, int table, hipStream_t stream) {
  const int64_t groups = (n + 2048 * UNITS - 1) / (2048 * UNITS);
  if (groups > 0x7fffffff) return HQ_ERR_TOO_LARGE;
  const int shift = __builtin_ctz((unsigned)blocksize);
  const int lanes = SPAN ? 64 : blocksize / 8;
  const auto kernel = table == HQ_TABLE_NF4 ? &quantize4_units_kernel<T, true, UNITS, SPAN> : &quantize4_units_kernel<T, false, UNITS, SPAN>;
  return hq_launch_as_is(kernel, dim3((unsigned)groups), dim3(256), 0, stream, x, packed, absmax, n, shift, lanes);
}

// Units per lane.  Blocks up to 512 elements: one, as the wave launcher is the better load scheduler (2^23 fp16 elements
// 5.2 / 5.5 / 6.5 us with 1 / 2 / 4; fp32 4096 x 11008 33.9 / 36.2 / 37.9), except for large fp16 inputs, where a
// workgroup's table and barrier weigh more (4096 x 11008: 20.2 / 18.9 / 19.6).  Longer blocks keep to one (fp32) or two (fp16, and
// fp32 blocks of 4096, which have no more than four waves) units and are shared by the waves of a workgroup, which exchange their
// maxima at the barrier that the cells need anyway (us with one wave per block, of 2, 4, 8 units a lane / this: blocksize 4096 of
// 5521 fp16 elements 5.4 / 2.9, 1 M 4.9 / 3.0, 8.4 M 6.9 / 5.7, 45 M 22.5 / 20.3, fp32 38.6 / 35.2; 2048 of 45 M fp16 21.9 / 20.35,
// fp32 37.4 / 33.4; 1024 fp32 35.2 / 33.7.  One unit of fp16: 2048 22.4, 1024 22.3 instead of 20.3).
template <typename T>
int quantize4_units(const T* x, uint8_t* packed, float* absmax, int64_t n, int blocksize, int table, hipStream_t stream) {
  constexpr bool kHalf = sizeof(T) == 2;
  constexpr int kUnits = kHalf ? 2 : 1;
  if (blocksize == 1024) return launch_quantize4_units<T, kUnits, 2 / kUnits>(x, packed, absmax, n, blocksize, table, stream);
  if (blocksize == 2048) return launch_quantize4_units<T, kUnits, 4 / kUnits>(x, packed, absmax, n, blocksize, table, stream);
  if (blocksize == 4096) return launch_quantize4_units<T, 2, 4>(x, packed, absmax, n, blocksize, table, stream);
  if (sizeof(T) == 2 && n >= (int64_t)1 << 24)
    return launch_quantize4_units<T, 2, 0>(x, packed, absmax, n, blocksize, table, stream);
  return launch_quantize4_units<T, 1, 0>(x, packed, absmax, n, blocksize, table, stream);
}

}  // namespace

extern "C" int hq_q3_pack(const uint8_t* codes, int32_t* qweight, int K, int N, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!codes || !qweight) return HQ_ERR_NULL_POINTER;
  if (K <= 0 || N <= 0 || (K & 31)) return HQ_ERR_BAD_SHAPE;
  if ((uintptr_t)qweight & 3) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  const int64_t total = (int64_t)(K / 32) * N;
  if ((total + 255) / 256 > 0x7fffffff) return HQ_ERR_TOO_LARGE;
  hipLaunchKernelGGL(q3_pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, codes,
                     reinterpret_cast<uint32_t*>(qweight), K / 32, N);
  return hq_launch_status();
}

extern "C" int hq_bcq_pack(const int8_t* signs, uint32_t* bW, int K, int N, int nbits, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (!signs || !bW) return HQ_ERR_NULL_POINTER;
  if (K <= 0 || N <= 0 || (K & 31) || nbits < 1 || nbits > 8) return HQ_ERR_BAD_SHAPE;
  if ((uintptr_t)bW & 3) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  const int64_t total = (int64_t)(K / 32) * nbits * N;
  if ((total + 255) / 256 > 0x7fffffff) return HQ_ERR_TOO_LARGE;
  hipLaunchKernelGGL(bcq_pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, signs, bW, K / 32,
                     nbits, N);
  return hq_launch_status();
}

extern "C" int hq_quantize_4bit(const void* x, int x_dtype, uint8_t* packed, float* absmax, int64_t n_elems,
                                int blocksize, int table, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  if (n_elems < 0 || blocksize <= 0 || (blocksize & 1)) return HQ_ERR_BAD_SHAPE;
  if (x_dtype != HQ_DTYPE_F32 && x_dtype != HQ_DTYPE_F16) return HQ_ERR_BAD_ENUM;
  if (table != HQ_TABLE_NF4 && table != HQ_TABLE_FP4) return HQ_ERR_BAD_ENUM;
  if (n_elems == 0) return HQ_OK;
  if (!x || !packed || !absmax) return HQ_ERR_NULL_POINTER;
  if (((uintptr_t)x & (x_dtype == HQ_DTYPE_F16 ? 1 : 3)) || ((uintptr_t)absmax & 3)) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  // Power-of-two blocks that a wave holds and pointers the wide loads and stores take; a wave per block otherwise.
  if (blocksize >= 8 && blocksize <= 4096 && (blocksize & (blocksize - 1)) == 0 && !((uintptr_t)x & 15) &&
      !((uintptr_t)packed & 3))
    return x_dtype == HQ_DTYPE_F16
               ? quantize4_units((const _Float16*)x, packed, absmax, n_elems, blocksize, table, stream)
               : quantize4_units((const float*)x, packed, absmax, n_elems, blocksize, table, stream);
  const int64_t nblocks = (n_elems + blocksize - 1) / blocksize;
  if ((nblocks + 3) / 4 > 0x7fffffff) return HQ_ERR_TOO_LARGE;
  const dim3 grid((unsigned)((nblocks + 3) / 4));
  if (x_dtype == HQ_DTYPE_F16)
    return hq_launch_as_is(quantize4_kernel<_Float16>, grid, dim3(256), 0, stream, (const _Float16*)x, packed, absmax, n_elems, blocksize, table);
  return hq_launch_as_is(quantize4_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, packed, absmax, n_elems, blocksize, table);
}
