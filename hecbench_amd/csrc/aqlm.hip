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
// to fp16 once.  Calls of millions of codes go another way (aqlm_sliced_kernel).
#include <type_traits>

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

// ---- many codes: the code book in slices --------------------------------------------------------------------------------
// The kernel above is bound by the L2, which answers one request per clock and channel: 240-250 G gathers/s whatever the rest.  An
// eighth of the code book fits a compute unit's LDS, so here the workgroups of eight compute units, each with its eighth, go over
// the same rows: every code is read by all eight (a cached 2 bytes instead of a request of 16) and answered by the one that holds its
// entry; for the others it points at an entry of zeros.  Their sums meet through memory.  What bounds it now are the vector
// instructions, 6.5 for a code in the loop and 7.7 in all, in each of the eight, and the LDS reads under them.
// The eight of a group of rows run on one XCD, whose L2 reads the group's codes from memory once.
// Gathers from L2 -> in slices, weights from memory: 8192 x 4096 19.8 -> 16.1 us, 18359 x 3840 37.7 -> 25.7, 28672 x 4096 with three code
// books 60.3 -> 36.5, 16234 x 10496 89.2 -> 48.5, 28672 x 15872 228 -> 111 (550 G codes/s without the 8 us in front and behind; the vector
// units 0.8 busy, an LDS read 4.7 cycles of which 0.7 are conflicts).  That is after a quarter of a second of such calls: the first sixty
// after idle take 125 to 148, at the clock that the power management begins with; the gathers, bound by the L2, 228 to 240 throughout.
constexpr int kSlices = 8, kEntries = 65536 / kSlices;
constexpr int kSlicedThreads = 1024, kSlicedWaves = kSlicedThreads / 64, kSlicedRows = 4;
constexpr size_t kSlicedBytes = (size_t)(kEntries + 1) * 16;  // a slice and the entry of zeros; behind it the activations
constexpr int kSlicedMaxLds = 160 * 1024;  // K up to 15872
constexpr size_t sliced_smem(int units) { return kSlicedBytes + (size_t)aqlm_x_stride(units) * 8 * 16 + kSlicedWaves * 4; }

// A half of a register, shifted, in one instruction (of an AND and a shift the compiler makes two here).
template <int HALF>
__device__ __forceinline__ uint32_t half_shifted(uint32_t v, uint32_t by) {
  uint32_t r;
  if (HALF) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(r) : "v"(by), "v"(v));
  else asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(r) : "v"(by), "v"(v));
  return r;
}

__global__ __launch_bounds__(kSlicedThreads) void aqlm_sliced_kernel(HQ_ARGS28) {
  HqReader rd(HQ_PASS28);
  AqlmArgs a;
  a.codes = rd; a.codebooks = rd; a.x = rd; a.M = rd; a.K = rd; a.cb_stride = rd;
  const int groups = rd, sub_bits = rd;  // groups of rows; 2^sub_bits rows side by side in a wave
  for (int i = 0; i < 4; ++i) a.cb_sizes[i] = rd;
  a.scales = rd; a.y = rd;
  float* const partial = rd;       // [group][slice][rows of a group]
  unsigned* const counters = rd;   // [group], zero between calls
  constexpr int R = kSlicedRows;
  extern __shared__ u4v lds[];
  u4v* const xl = lds + kEntries + 1;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup b runs on XCD b mod 8
  const int place = blockIdx.x >> 3, slice = place & (kSlices - 1);
  const int per_xcd = (groups + 7) >> 3, group = (int)(blockIdx.x & 7) * per_xcd + place / kSlices;
  if (group >= groups) return;
  const int g0 = (int)((int64_t)a.M * group / groups), g1 = (int)((int64_t)a.M * (group + 1) / groups);
  if (g0 == g1) return;  // fewer rows than groups: none here, and no row whose codes could be read ahead of the first trip
  const int group_rows = (a.M + groups - 1) / groups;
  float* const mine = partial + (size_t)(group * kSlices + slice) * group_rows;

  const int units = a.K >> 6;  // of eight codes, a row
  const int xstride = aqlm_x_stride(units);
  const int width = 64 >> sub_bits, ul = lane & (width - 1);
  const int nchunk = (units + width - 1) >> (6 - sub_bits);
  // the first code book's slice, on its way before anything else
  constexpr int kFill = kEntries / kSlicedThreads;
  u4v e0[kFill];
  auto book_of = [&](int row, int& end) {  // the code book of a row, and where its rows end
    const u4v* book = a.codebooks;
    int j = 0;
    for (; j < 4 && row >= a.cb_sizes[j]; ++j) book += a.cb_stride;
    end = j < 4 ? min(g1, a.cb_sizes[j]) : g1;
    return book;
  };
  auto fetch = [&](const u4v* book) {
#pragma unroll
    for (int i = 0; i < kFill; ++i) e0[i] = book[slice * kEntries + i * kSlicedThreads + tid];
  };
  int b1;
  fetch(book_of(g0, b1));
  int bad = 0;  // infinities or NaN among the activations: there a code of another slice must not be multiplied by zero
  for (int t = tid; t < units * 8; t += kSlicedThreads) {
    const u4v v = a.x[t];
#pragma unroll
    for (int i = 0; i < 4; ++i) bad |= (v[i] & 0x7c00u) == 0x7c00u || (v[i] & 0x7c000000u) == 0x7c000000u;
    xl[(t & 7) * xstride + (t >> 3)] = v;
  }
  uint32_t* const tail = reinterpret_cast<uint32_t*>(xl + 8 * xstride);
  bad = __ballot(bad) != 0;
  if (lane == 0) tail[wv] = bad;
  if (tid == 0) lds[kEntries] = u4v{0, 0, 0, 0};

  // Addresses in LDS are made of a code's bits alone: the dynamic LDS of a kernel without static LDS begins at 0.
  typedef __attribute__((address_space(3))) const u4v* lds_entry;
  const unsigned char* const group_codes = reinterpret_cast<const unsigned char*>(a.codes + (size_t)g0 * units);
  auto rows_of = [&](auto masked_c, int b0, int b1) {
    constexpr bool masked = decltype(masked_c)::value;
    const int batch = kSlicedWaves * (R << sub_bits), trips = (b1 - b0 + batch - 1) / batch;
    // the lane's place is worked out anew where rows change: kept through the loop it would cost registers that there are not
    auto row_of = [&](int t, int r, int lane) { return b0 + (((t * kSlicedWaves + wv) * R + r) << sub_bits) + (lane >> (6 - sub_bits)); };
    auto lane_again = [&]() {
      int again = tid;
      asm("" : "+v"(again));
      return again & 63;
    };
    uint32_t row_at[R];
    auto point = [&](int t) {
      const int lane = lane_again();
#pragma unroll
      for (int r = 0; r < R; ++r) row_at[r] = (uint32_t)(min(row_of(t, r, lane), b1 - 1) - g0) * (uint32_t)(units * 16);
    };
    auto load_codes = [&](int c, u4v (&cw)[R]) {
      const uint32_t at = (uint32_t)min(c * width + ul, units - 1) * 16u;
#pragma unroll
      for (int r = 0; r < R; ++r) cw[r] = *reinterpret_cast<const u4v*>(group_codes + (row_at[r] + at));
    };
    u4v cw[R], xv[8];
    point(0);
    load_codes(0, cw);
    uint32_t four = 4;
    asm("" : "+v"(four));
    const uint32_t mine2 = (uint32_t)slice * (kEntries * 0x10001u);
    for (int t = 0; t < trips; ++t) {
      if (b0 + (((t * kSlicedWaves + wv) * R) << sub_bits) >= b1) break;  // no rows left for this wave
      float acc[R];
#pragma unroll
      for (int r = 0; r < R; ++r) acc[r] = 0.f;
      for (int c = 0; c < nchunk; ++c) {
        u4v next[R];
        int cn = c + 1;
        if (cn == nchunk) {
          cn = 0;
          point(t + 1);  // (past the last trip: the last row again)
        }
        load_codes(cn, next);
        const int u = c * width + ul;
        if (nchunk > 1 || t == 0) {
#pragma unroll
          for (int i = 0; i < 8; ++i) xv[i] = xl[i * xstride + min(u, units - 1)];
        }
        uint32_t beyond = u < units ? 0u : 0xffffffffu;  // lanes past the row's end: no entry
        asm("" : "+v"(beyond));
        auto row = [&](int r) {
          typedef uint16_t us2 __attribute__((ext_vector_type(2)));
          const uint32_t w[4] = {cw[r].x, cw[r].y, cw[r].z, cw[r].w};
          u4v e[8];
          uint32_t at[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const us2 most = {(uint16_t)kEntries, (uint16_t)kEntries};
            const uint32_t two = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2, (w[i] ^ mine2) | beyond), most));
            at[2 * i] = half_shifted<0>(two, four);
            at[2 * i + 1] = half_shifted<1>(two, four);
          }
#pragma unroll
          for (int i = 0; i < 8; ++i) e[i] = *(lds_entry)at[i];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            u4v x = xv[i];
            if (masked) x &= at[i] < kEntries * 16 ? 0xffffffffu : 0u;
            acc[r] = dot8(e[i], x, acc[r]);
          }
        };
#pragma unroll
        for (int r = 0; r < R; ++r) row(r);
#pragma unroll
        for (int r = 0; r < R; ++r) cw[r] = next[r];
      }
      const int lane = lane_again();
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float v = hq_row(acc[r], HqAdd());
        if (sub_bits < 2) {
          const float lo = hq_lane(v, 0) + hq_lane(v, 16), hi = hq_lane(v, 32) + hq_lane(v, 48);
          v = sub_bits == 0 ? lo + hi : (lane < 32 ? lo : hi);
        }
        const int m = row_of(t, r, lane);
        if ((lane & (width - 1)) == 0 && m < b1) __hip_atomic_store(mine + (m - g0), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  };

  for (int b0 = g0;;) {  // the rows of one code book after the other's
#pragma unroll
    for (int i = 0; i < kFill; ++i) lds[i * kSlicedThreads + tid] = e0[i];
    __syncthreads();
    if (b0 == g0) bad = __builtin_amdgcn_readfirstlane(__ballot(tail[lane & (kSlicedWaves - 1)] != 0) != 0);
    if (bad) rows_of(std::true_type(), b0, b1);
    else rows_of(std::false_type(), b0, b1);
    if (b1 >= g1) break;
    b0 = b1;
    fetch(book_of(b0, b1));
    __syncthreads();  // every wave is done with the last book's slice
  }

  // ---- the slices meet: the last workgroup of a group to arrive adds them in order ----
  uint32_t* const last = tail;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(&counters[group], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = old == kSlices - 1;
    if (old == kSlices - 1) __hip_atomic_store(&counters[group], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!*last) return;
  for (int r = tid; r < g1 - g0; r += kSlicedThreads) {
    float v = hq_sum_partials(partial + (size_t)group * kSlices * group_rows + r, group_rows, kSlices);
    if (a.scales) v *= (float)a.scales[g0 + r];
    a.y[g0 + r] = (_Float16)v;
  }
}

// Which calls go in slices, and how many rows a wave has side by side (a row of K / 64 units takes whole runs of 64, 32 or 16 lanes).
// Both times are fits to 60 problems of 1.2 M to 57 M codes on MI355X (spread 6 %; over them the choice costs 0.9 % on average
// against the better of the two): the gathers' 2.4 us and 242 G codes/s; in slices 8.1 us for the first data, the slice's way into LDS and
// the meeting of the eight, 1.86 us for a trip of the sixteen waves over one run of lanes and 0.5 beside for its sums, the last
// trip for its share of waves and a fifth more, 0.6 where there are several code books.  The line lies at 3 to 4.5 M codes: 2001 x 10240
// and 4096 x 4096 stay (10.3 us against 11.7), 8192 x 4096 19.8 -> 16.1, 28672 x 1024 18.6 -> 16.6.
struct SlicedPlan {
  int groups, sub_bits;  // groups 0: not in slices
};
SlicedPlan sliced_plan(const HqDevice* dev, int M, int K, bool several_books) {
  SlicedPlan p = {0, 0};
  const int force = hq_tune(HQ_TUNE_AQLM_ROWS, 0), units = K >> 6, groups = dev->cus / kSlices;
  // offsets within a group are 32-bit; a workspace of at most 32 MB
  if (groups < 1 || sliced_smem(units) > kSlicedMaxLds || M > 1 << 20 || (int64_t)(M / groups + 1) * units >= 1 << 28) return p;
  if (force >= 20 && force <= 22) return SlicedPlan{groups, force - 20};
  if (force) return p;
  float best = 0.97f * (2.4f + (float)M * (float)units * 8.f / (242e3f / 256.f * dev->cus));
  if (best < 10.f) return p;
  for (int sub = 0; sub < 3; ++sub) {
    const int chunks = (units + (64 >> sub) - 1) >> (6 - sub);
    const float trips = (float)((M + groups - 1) / groups) / (kSlicedWaves * (kSlicedRows << sub));
    const float part = trips - (int)trips;
    const float us = 8.1f + ((int)trips + (part > 0.f ? 0.2f + 0.8f * part : 0.f)) * (1.86f * chunks + 0.5f) + (several_books ? 0.6f : 0.f);
    if (us < best) {
      best = us;
      p = SlicedPlan{groups, sub};
    }
  }
  return p;
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
  // Many codes: in slices.  That kernel takes memory of its stream.  A captured call, whose graph may be replayed beside calls on that
  // stream and beside other graphs captured there (nobody had to order calls of this operator), and one that finds no memory stay with the other one.
  // Nor does one on the per-thread stream take it: one handle for as many streams as there are threads.
  const SlicedPlan sliced = sliced_plan(dev, M, K, cb_a_sizes[0] < M);
  if (sliced.groups > 0 && stream != hipStreamPerThread) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    HqWorkspace ws;
    const size_t group_rows = (M + sliced.groups - 1) / sliced.groups;
    if (hipStreamIsCapturing(stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone &&
        hq_get_eager_workspace(stream, (size_t)sliced.groups * kSlices * group_rows, sliced.groups, &ws) == HQ_OK) {
      static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&aqlm_sliced_kernel),
                                                         hipFuncAttributeMaxDynamicSharedMemorySize, kSlicedMaxLds);
      if (attr != hipSuccess) return (int)attr;
      return hq_launch(aqlm_sliced_kernel, dim3((sliced.groups + 7) / 8 * 8 * kSlices), dim3(kSlicedThreads), sliced_smem(K >> 6), stream,
                       a.codes, a.codebooks, a.x, a.M, a.K, a.cb_stride, sliced.groups, sliced.sub_bits, a.cb_sizes[0], a.cb_sizes[1],
                       a.cb_sizes[2], a.cb_sizes[3], a.scales, a.y, ws.partial, ws.counters);
    }
    (void)hipGetLastError();
  }
  // Rows per wave, and whether the four waves of a workgroup share its rows, each with every fourth chunk of 512 codes (split).
  // What counts is gathers in flight and evenly over the compute units.  Measured (us, one / two / four rows per wave; one / two
  // split): 4096 x 4096 11.7 12.4 12.8; 13.3 12.9 - 9788 x 5440 31.3 30.9 33.1; 34.2 33.0 - 28672 x 4096 three code books 62.0 61.1
  // 62.9; 71.9 68.2 - 28672 x 16384 291 239 237; 271 248 - 1228 x 16192 25.1 23.2 39.6; 17.1 16.6 - 2472 x 11968 24.9 27.1 27.2;
  // 21.9 20.2 - 512 x 16384 12.3 17.3 28.7; 9.4 9.4 - 689 x 5184 6.8 9.1 15; 6.3 6.5.  HQ_AQLM_ROWS: 1, 2, 4; 11, 12 split; 20 to 22 in slices
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
