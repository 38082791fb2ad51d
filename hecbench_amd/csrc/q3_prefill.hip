// Batched GPTQ 3-bit GEMM for gfx950, many rows (a prompt's tokens): fp16 activations, fp32 output,
//
//   out[m][n] = s[n] * sum_k A[m][k]*q[k][n]  -  z[n] * sum_k A[m][k]
//
// The operands are those of q3_gemm.hip: codes stay subnormal fp16 numbers (an AND per two weights, q3_recipe.h), the
// pre-pass writes the activations in operand-slot order with a power of two per row and the row sums.
//
// What bounds it: the matrix cores, and those by the power limit (1.9-2.0 GHz while all of them run).  The 64-row kernel
// streams weights and activations from the L2 into registers for 64 rows at a time: 16 passes over the weights for 1021
// rows, at 0.83 PFLOP/s.  Here a tile of 128 x 256 or 64 x 256 / 128 results stays in the accumulators of eight waves while
// its operands go through LDS in stages (loads straight into LDS, three to five stages in flight, one barrier per step).
//   - A wave holds 128 (64) rows x 64 columns and its own part of every step of K: an unpacked weight serves all of
//     the tile's rows (with the tile's rows cut between waves every weight was unpacked twice, and with few rows the
//     loop was bound by instructions: 0.51 against 0.35 us per 64 elements of K at 64 rows), two waves share a SIMD, and
//     a barrier comes once per 128 or 256 elements.
//   - Operand reads run one to three quarters of a step ahead, the LDS loads of a stage go out one by one between the
//     matrix instructions, and unpacking fills the slots between those.
//   - Tiles that do not fill a round of the compute units are divided along K (tile_plan), or, where they are few, left to the
//     one-launch kernel (cut_plan).
// K=8192, N=28672, 1021 rows: 574 -> 363-390 us (1.22-1.32 PFLOP/s; the library's fp16 product of 8192^3 runs at 1.2 here);
// 512 rows, K=4096, N=11008: 153 -> 52-57; 128 rows, K=8192, N=28672: 75 -> 58.
#include <type_traits>

#include "hq_internal.h"
#include "q3_tile.h"

namespace {

using namespace hq_q3;

constexpr int kWaves = 8;      // two per SIMD
constexpr int kThreads = 64 * kWaves;

// A wave multiplies MB 32-row blocks by 64 columns over one of KS parts of every step of K; the eight waves are KS parts
// times 8 / KS column blocks of 64, and the parts' sums meet in LDS at the end of a tile.
template <int MB, int KS>
struct Shape {
  static constexpr int kTileM = 32 * MB;
  static constexpr int kCols = kWaves / KS;                // column blocks of a tile
  static constexpr int kTileN = 64 * kCols;
  static constexpr int kABytes = 8 * KS * kTileM * 16;     // 2 KS k-groups x four operands x rows x 16 bytes
  static constexpr int kWBytes = 6 * KS * kTileN * 4;      // packed rows
  static constexpr int kStageBytes = kABytes + kWBytes;
  static constexpr int kStages = kStageBytes <= 28 * 1024 ? 5 : 3;
  static constexpr int kAhead = MB == 4 ? 1 : 3;           // operand quarters of a step in registers ahead of their use
  static constexpr int kALoads = kABytes / 1024 / kWaves;  // LDS loads (1 KB) of one wave and stage
  static constexpr int kWLoads = (kWBytes / 1024 + kWaves - 1) / kWaves;
  static constexpr int kLoads = kALoads + kWLoads;
  static constexpr int kFinal = 4 * MB / KS;               // groups of eight rows x 64 columns that a wave finishes
  static constexpr int kSmem = kStages * kStageBytes + 16;
  static_assert(kWaves * (KS - 1) * kFinal * 2048 <= kStages * kStageBytes, "the parts of K meet in the stages' LDS");
};

struct TileArgs {
  const uint32_t* w;
  const unsigned char* Ap;  // [2 KS T k-groups][4][Mpad][16 bytes]
  const float* rowsum;      // [Mpad]
  const float* rowinv;      // [Mpad]
  const float* scales;
  const float* zeros;
  float* out;
  float* partial;           // [rest][nshare][tile]
  unsigned* counters;       // [divided tiles]
  int M, N, G, Mpad, nmt;   // rows, columns, k-groups, padded rows, row tiles
  int T;                    // steps per tile
  int rounds, rest;         // whole tiles per workgroup, and the tiles that are left
  int nshare, L;            // which are divided into nshare shares of L steps, one per workgroup
  unsigned flags;
};

template <int MB, int KS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void q3_tile_kernel(TileArgs a) {
  using S = Shape<MB, KS>;
  extern __shared__ unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wv % S::kCols, kp = wv / S::kCols;  // column block, part of K
  const int nl = lane & 31, kb = lane >> 5;
  const int nwg = gridDim.x;
  // workgroup b runs on XCD b mod 8: an XCD takes consecutive tiles (row tiles of one column tile first), which share
  // weights and activations in its L2
  const int xcd = blockIdx.x & 7;
  const int v = xcd * (nwg >> 3) + min(xcd, nwg & 7) + (int)(blockIdx.x >> 3);

  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  uint32_t acol[S::kALoads];
  constexpr int kOpBytes = S::kTileM * 16;                  // one operand of the tile's rows
  const int op0 = wv * S::kALoads * 1024 / kOpBytes;        // this wave's first
#pragma unroll
  for (int i = 0; i < S::kALoads; ++i) {
    const int o = i * 1024 + lane * 16;
    acol[i] = (o / kOpBytes) * (a.Mpad * 16) + o % kOpBytes;
  }
  const size_t ap_step = (size_t)8 * KS * a.Mpad * 16, w_step = (size_t)6 * KS * a.N * 4;
  const unsigned char* a_lane = lds + ((8 * kp + kb * 4) * S::kTileM + nl) * 16;
  const unsigned char* w_lane = lds + S::kABytes + ((6 * kp + 3 * kb) * S::kTileN + wn * 64 + 2 * nl) * 4;

  for (int round = 0; round <= a.rounds; ++round) {
    // ---- steps t0 .. t0 + len - 1 of a tile ----
    int tile, t0 = 0, len = a.T, share = 0;
    if (round < a.rounds) {
      tile = round * nwg + v;
    } else {
      const int rt = v / a.nshare;
      if (rt >= a.rest) break;
      share = v - rt * a.nshare;
      tile = a.rounds * nwg + rt;
      t0 = share * a.L;
      len = min(a.L, a.T - t0);
    }
    const int ct = __builtin_amdgcn_readfirstlane(tile / a.nmt), mt = tile - ct * a.nmt;

    // ---- loader: this wave's part of a stage ----
    // A load covers 1 KB of packed rows: one row of 256 columns or two of 128.  The waves left over load the last again.
    constexpr int kLanes = S::kTileN / 4, kRowsPerLoad = 64 / kLanes;
    const uint32_t wcol = (uint32_t)min(ct * S::kTileN + 4 * (lane % kLanes), a.N - 4) * 4;
    const unsigned char *ap, *wp[S::kWLoads];
    uint32_t wlane[S::kWLoads];
    auto point = [&](int t) {
      ap = a.Ap + ((size_t)(8 * KS * t + op0) * a.Mpad + mt * S::kTileM) * 16;
#pragma unroll
      for (int i = 0; i < S::kWLoads; ++i) {
        const int row0 = min((wv + kWaves * i) * kRowsPerLoad, 6 * KS - kRowsPerLoad);
        auto row_of = [&](int r) { return min(6 * KS * t + r, 3 * a.G - 1); };  // past the end: any weights, zero activations
        const int p0 = row_of(row0);
        wp[i] = reinterpret_cast<const unsigned char*>(a.w + (size_t)p0 * a.N);
        wlane[i] = wcol;
        if (kRowsPerLoad > 1 && lane >= kLanes) wlane[i] += (uint32_t)(row_of(row0 + 1) - p0) * (uint32_t)a.N * 4u;
      }
    };
    int ld_left = len;
    uint32_t stage_ld = lds0;
    auto ld_advance = [&]() {
      stage_ld += S::kStageBytes;
      if (stage_ld == lds0 + S::kStages * S::kStageBytes) stage_ld = lds0;
      if (--ld_left > 1) {
        ap += ap_step;
#pragma unroll
        for (int i = 0; i < S::kWLoads; ++i) wp[i] += w_step;
      } else {
        // the last step: its k-groups may reach past the last one (zero activations there).  Beyond it the last step
        // again, which is never read.
        point(t0 + len - 1);
      }
    };
    auto dma = [&](int l) {
      if (l < S::kWLoads) load_lds(stage_ld + S::kABytes + min(wv + kWaves * l, S::kWBytes / 1024 - 1) * 1024, wlane[l], wp[l]);
      else load_lds(stage_ld + (wv * S::kALoads + l - S::kWLoads) * 1024, acol[l - S::kWLoads], ap);
    };

    f16v acc[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mb][q][i] = 0.f;

    constexpr int P = S::kAhead;
    u4v A[P + 1][MB];  // ring: quarter j of a step in A[j % (P + 1)]
    u2v wr[3];
    auto read_a = [&](uint32_t stage, int j) {
      const unsigned char* p = a_lane + stage;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) A[j % (P + 1)][mb] = *reinterpret_cast<const u4v*>(p + (j * S::kTileM + mb * 32) * 16);
    };
    auto read_w = [&](uint32_t stage, u2v (&dst)[3]) {
      const unsigned char* p = w_lane + stage;
#pragma unroll
      for (int j = 0; j < 3; ++j) dst[j] = *reinterpret_cast<const u2v*>(p + j * (S::kTileN * 4));
    };

    point(t0);
#pragma unroll
    for (int i = 0; i < S::kStages - 1; ++i) {
      if (i) ld_advance();
#pragma unroll
      for (int l = 0; l < S::kLoads; ++l) dma(l);
    }
    wait_loads_and_meet<(S::kStages - 2) * S::kLoads>();
    uint32_t stage = 0;  // byte offset of the stage being multiplied
    read_w(0, wr);
#pragma unroll
    for (int j = 0; j < P; ++j) read_a(0, j);
    u4v B[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) B[0][q] = unpack_quarter<0>(wr[0][q], wr[1][q], wr[2][q]);
    for (int s = 0; s < len; ++s) {
      const uint32_t stage1 = stage + S::kStageBytes == S::kStages * S::kStageBytes ? 0 : stage + S::kStageBytes;
      u2v wnext[3];
      // Quarter j: the reads of quarter j + P and some of the loads of the stage that is free go out first (one by one:
      // all at once they queue up in front of the address unit and hold up what stands behind them), then the
      // multiplications of this quarter with the unpacking of the next between them.
      auto quarter = [&](auto jc) {
        constexpr int j = decltype(jc)::value;
        if (j == 1) {
          // the next step's operands are in LDS once every wave's share has arrived; with that every wave is past
          // the step before this one, whose stage takes new loads
          wait_loads_and_meet<(S::kStages - 3) * S::kLoads>();
          ld_advance();
          read_w(stage1, wnext);
        }
        if (j + P < 4) read_a(stage, j + P);
        else read_a(stage1, j + P - 4);
#pragma unroll
        for (int l = 0; l < S::kLoads; ++l)
          if (j > 0 && l % 3 == j - 1) dma(l);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int jn = (j + 1) & 3;
#pragma unroll
        for (int q = 0; q < 2; ++q)
          B[(j + 1) & 1][q] = j < 3 ? unpack_quarter<jn>(wr[0][q], wr[1][q], wr[2][q])
                                    : unpack_quarter<jn>(wnext[0][q], wnext[1][q], wnext[2][q]);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[mb][q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, A[j % (P + 1)][mb]),
                                                                __builtin_bit_cast(h8, B[j & 1][q]), acc[mb][q], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2 * MB; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // one matrix instruction
          __builtin_amdgcn_sched_group_barrier(0x002, 8 / MB, 0);  // some vector instructions
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      quarter(std::integral_constant<int, 0>());
      quarter(std::integral_constant<int, 1>());
      quarter(std::integral_constant<int, 2>());
      quarter(std::integral_constant<int, 3>());
#pragma unroll
      for (int j = 0; j < 3; ++j) wr[j] = wnext[j];
      stage = stage1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load in flight into LDS from here on,
    __syncthreads();                                  // and no wave reads the stages any more

    // ---- the parts of K meet: part p finishes groups of eight rows p * kFinal and up ----
    // Selects instead of branches on the part: register indices stay constant.
    constexpr int F = S::kFinal;
    auto group = [&](int p, int i, int q) {  // group i of part kp ^ p
      f4v x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        auto of = [&](int part) { return acc[(part * F + i) / 4][q][4 * ((part * F + i) % 4) + e]; };
        x[e] = kp & 1 ? of(p ^ 1) : of(p);
        if (KS == 4) {
          const float y = kp & 1 ? of(p ^ 3) : of(p ^ 2);
          x[e] = kp & 2 ? y : x[e];
        }
      }
      return x;
    };
    f4v* const meet = reinterpret_cast<f4v*>(lds) + lane;
    auto at = [&](int to, int from) { return meet + ((to * (KS - 1) + from) * S::kCols + wn) * (F * 2 * 64); };
#pragma unroll
    for (int p = 1; p < KS; ++p)
#pragma unroll
      for (int i = 0; i < F * 2; ++i) at(kp ^ p, p - 1)[i * 64] = group(p, i / 2, i % 2);
    __syncthreads();
    f4v fin[F][2];
#pragma unroll
    for (int i = 0; i < F * 2; ++i) {
      f4v x = group(0, i / 2, i % 2);
#pragma unroll
      for (int p = 1; p < KS; ++p) {
        const f4v other = at(kp, p - 1)[i * 64];
        x = p & 1 ? x - other : x + other;  // odd parts' k-groups are the negated ones (see the pre-pass)
      }
      fin[i / 2][i % 2] = x;  // negated itself where kp is odd
    }
    __syncthreads();  // before the next tile's loads

    bool finish = true;
    if (round == a.rounds && a.nshare > 1) {
      // A share of a divided tile: raw sums go out, every wave waits for their acknowledgement, the workgroup counts
      // itself at the memory side, and the last to arrive adds the shares in order of k.
      const int rt = tile - a.rounds * nwg;
      auto slot = [&](int c) {
        return reinterpret_cast<f4v*>(a.partial) + (size_t)(rt * a.nshare + c) * (S::kTileM * S::kTileN / 4) + tid;
      };
      f4v* dst = slot(share);
#pragma unroll
      for (int i = 0; i < F * 2; ++i) hq_store_share(dst + i * kThreads, fin[i / 2][i % 2]);
      unsigned* last = reinterpret_cast<unsigned*>(lds + S::kStages * S::kStageBytes);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(&a.counters[rt], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *last = old == (unsigned)(a.nshare - 1);
        if (old == (unsigned)(a.nshare - 1))  // ready for the next call
          __hip_atomic_store(&a.counters[rt], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __syncthreads();
      finish = *last != 0;
      if (finish) {
        // two shares: the other's on top of this one's registers (a sum of two is the same either way); more: all of
        // them from memory
        const bool two = a.nshare == 2;
        for (int c = two ? 1 - share : 0; c < (two ? 2 - share : a.nshare); ++c) {
          const f4v* src = slot(c);
          f4v x[F * 2];
#pragma unroll
          for (int i = 0; i < F * 2; ++i) x[i] = hq_load_share(src + i * kThreads);
          hq_wait_shares(x);
#pragma unroll
          for (int i = 0; i < F * 2; ++i) fin[i / 2][i % 2] = !two && c == 0 ? x[i] : fin[i / 2][i % 2] + x[i];
        }
      }
    }
    if (finish) {
      const int n = ct * S::kTileN + wn * 64 + 2 * nl;
      const int nc = min(n, a.N - 2);
      const f2v sc = *reinterpret_cast<const f2v*>(a.scales + nc), zr = *reinterpret_cast<const f2v*>(a.zeros + nc);
#pragma unroll
      for (int i = 0; i < F; ++i) {
        const int m0 = mt * S::kTileM + (kp * F + i) * 8 + 4 * kb;
        const f4v ri = *reinterpret_cast<const f4v*>(a.rowinv + m0), rs = *reinterpret_cast<const f4v*>(a.rowsum + m0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (m0 + e < a.M && n < a.N) {
            const float unit = ri[e] * (kp & 1 ? -16777216.f : 16777216.f);  // 2^24: the unit of the code operands
            f2v o = {sc.x * (fin[i][0][e] * unit) - zr.x * rs[e], sc.y * (fin[i][1][e] * unit) - zr.y * rs[e]};
            f2v* p = reinterpret_cast<f2v*>(a.out + (size_t)(m0 + e) * a.N + n);
            if (a.flags & HQ_FLAG_ACCUMULATE) o += *p;
            __builtin_nontemporal_store(o, p);
          }
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loop counts its own loads only
  }
}

// Host arithmetic of a launch (the launch, the workspace reservation and the size query share it).
struct TilePlan {
  int tm, tn, ks, nmt, T, nwg, rounds, rest, nshare, L, Mpad;
  int cut;  // columns from here on go through the one-launch kernel; N: none
  HqQ3DirectPlan direct;
  float us;
  size_t ap_floats, row_floats, partial_floats, counters;
};

// The three tiles and what they cost, measured on MI355X (us): a step (64 * ks elements of K; between a launch of few
// workgroups and a full device, whose clock the power limit lowers), and dividing a tile's K into c shares.  A tile costs
// 3 us beside its steps (first loads from HBM, the parts of K meeting, results).  The large tile multiplies most per
// load and unpacked weight: K=8192, N=28672, 1021 rows 367 us against 397 and 520 with the smaller ones; 512 rows, K=4096,
// N=11008 52 / 58 / 68.  Smaller problems want more workgroups: 128 rows, K=8192, N=28672 61 / 57 / 78; 98 rows, K=4512, N=8712
// 33 / 24 / 27; 397 rows, K=2720, N=9220 41 / 40 / 37.  (The smallest are the one-launch kernel's: q3_direct.hip.)
struct TileKind {
  int tm, tn, ks;
  float step_us, share_us, per_share_us;
};
constexpr TileKind kKinds[3] = {{128, 256, 2, 1.4f, 4.0f, 3.2f}, {64, 256, 2, 0.8f, 3.5f, 1.15f}, {64, 128, 4, 1.0f, 3.5f, 1.15f}};
constexpr int kMaxShares = 8;
constexpr int kMaxWorkgroups = 512;  // bounds the workspace on larger devices

// What T steps of a tile take in c shares.
float tile_us(const TileKind& kind, int T, int c) {
  return 3.f + (T + c - 1) / c * kind.step_us + (c > 1 ? kind.share_us + c * kind.per_share_us : 0.f);
}

TilePlan tile_plan_of(int cus, int K, int N, int M, const TileKind& kind, int want_shares) {
  TilePlan p;
  const int G = K / 32;
  p.cut = N;
  p.tm = kind.tm; p.tn = kind.tn; p.ks = kind.ks;
  p.T = (G + 2 * p.ks - 1) / (2 * p.ks);
  p.nmt = (M + p.tm - 1) / p.tm;
  p.Mpad = p.nmt * p.tm;
  p.nwg = cus < kMaxWorkgroups ? cus : kMaxWorkgroups;
  const int ntiles = p.nmt * ((N + p.tn - 1) / p.tn);
  // whole tiles in full rounds of one workgroup per compute unit; the tiles that are left are divided along K
  p.rounds = ntiles / p.nwg;
  p.rest = ntiles - p.rounds * p.nwg;
  p.nshare = 1;
  float best = 0.f;
  for (int c = 1; p.rest && c <= kMaxShares && c * p.rest <= p.nwg && c <= p.T; ++c) {
    const float t = tile_us(kind, p.T, c);
    if (c == 1 || (want_shares ? c <= want_shares : t < best)) { best = t; p.nshare = c; }
  }
  p.us = p.rounds * (3.f + p.T * kind.step_us) + best;
  p.L = (p.T + p.nshare - 1) / p.nshare;
  p.nshare = (p.T + p.L - 1) / p.L;
  if (p.rounds == 0) p.nwg = p.rest * p.nshare;
  p.ap_floats = (size_t)p.T * 2 * p.ks * 4 * p.Mpad * 4;
  p.row_floats = 2 * (size_t)p.Mpad;
  p.partial_floats = p.nshare > 1 ? (size_t)p.rest * p.nshare * p.tm * p.tn : 0;
  p.counters = p.rest;
  return p;
}

// The same with the column tiles beyond the last full round left to the one-launch kernel, in a launch of its own behind this one.
// Dividing a few tiles along K costs most of a round whatever their number (shares of 128 x 256 sums go out to memory and come back):
// 1024 rows, K=2048, 33 column tiles of 256, the 33rd divided 50.7 us, as 32 x 64 tiles of the one-launch kernel 44.2.  1271 rows, K=2048,
// N=26476 (four rounds and 16 tiles) 155 -> 143; 1902, K=1056, N=13184 85 -> 74; 1580, K=1504, N=25548 156 -> 146; 290, K=6272, N=14240 66 ->
// 60.6.  From two fifths of a round on nothing is gained (1975, K=1632, N=10760, 176 tiles: 92.0 / 99.4), and with the smallest tile never.
// Without such columns the plan as it is.
TilePlan cut_plan(int cus, int K, int N, int M, const TileKind& kind, bool forced) {
  const TilePlan whole = tile_plan_of(cus, K, N, M, kind, 0);
  const int cols = whole.rounds * whole.nwg / whole.nmt;
  if ((!forced && (5 * whole.rest > 2 * whole.nwg || kind.ks != 2)) || whole.rounds < 1 || cols < 1 || cols * kind.tn >= N ||
      !hq_q3_direct_can(K, N))
    return whole;
  TilePlan p = tile_plan_of(cus, K, cols * kind.tn, M, kind, 0);
  p.direct = hq_q3_direct_plan(cus, K, N - p.cut, M, false);
  p.us += p.direct.us;
  return p;
}

// The least of the estimates; columns are cut off where that is less by 7 us, which the second launch takes beside its own estimate (it
// begins when the last tile has gone out), or by 1 where the call is longer than 36 us and the tile the large one, whose rounds then take
// more than theirs.  452 drawn problems for which the estimates alone are for the cut: 1.037 times as fast in the geometric mean as without any
// (all of them cut 1.032), 14 more than 3 % slower than without (76; 263 rows, 2240 x 13548 27.1 / 33.2, 1848 rows, 288 x 9420 40.6 / 49.5).
TilePlan tile_plan(int cus, int K, int N, int M) {
  const int force = hq_tune(HQ_TUNE_Q3_TILES, -1);  // tests: kind + 10 * shares (3 to 6 the one-launch kernel's, 9 none in particular; 100 + kind: cut)
  if (force >= 100 && force < 103) return cut_plan(cus, K, N, M, kKinds[force - 100], true);
  if (force >= 0 && force % 10 < 3) return tile_plan_of(cus, K, N, M, kKinds[force % 10], force / 10);
  TilePlan whole = tile_plan_of(cus, K, N, M, kKinds[0], 0);
  for (int i = 1; i < 3; ++i) {
    const TilePlan p = tile_plan_of(cus, K, N, M, kKinds[i], 0);
    if (p.us < whole.us) whole = p;
  }
  TilePlan best = whole;
  for (int i = 0; i < 3; ++i) {
    const TilePlan p = cut_plan(cus, K, N, M, kKinds[i], false);
    if (p.cut < N && p.us < best.us && p.us < whole.us - (i == 0 && whole.us > 36.f ? 1.f : 7.f)) best = p;
  }
  // Beside the one-launch kernel's estimate of the whole call a cut costs 6 more, and no more than the plan that it was better than; in
  // long calls, where that estimate is too little as well, nothing.  231 drawn problems that the sum alone gives to the tiles with a
  // cut, the one-launch kernel's time / theirs: 1999 rows, 960 x 4492 32.0 / 39.4, 1179, 1216 x 7208 34.4 / 40.4, 576, 1280 x 14524 34.6 /
  // 39.8; 1654, 2144 x 5056 59.0 / 47.5, 324, 2432 x 23040 54.2 / 48.0, 1992, 768 x 16592 87.8 / 74.8.  Taken throughout: 1.015 times as fast
  // as without any cut, 71 more than 3 % slower; this choice 1.033 and 9.
  if (best.cut < N && best.us < 50.f) best.us = best.us + 6.f < whole.us ? best.us + 6.f : whole.us;
  return best;
}

// Rows of one pass over the weights: equal passes of as many rows as 32 MB of re-ordered activations hold, 1024 at least.
int rows_per_pass(int K, int M) {
  int most = (int)(((size_t)16 << 20) / (size_t)K) / 128 * 128;
  most = most < 1024 ? 1024 : (most > 8192 ? 8192 : most);
  const int passes = (M + most - 1) / most;
  return ((M + passes - 1) / passes + 127) / 128 * 128;
}

template <int MB, int KS>
int launch_tiles(const TileArgs& a, int nwg, hipStream_t stream) {
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&q3_tile_kernel<MB, KS>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, Shape<MB, KS>::kSmem);
  if (attr != hipSuccess) return (int)attr;
  return hq_launch_as_is(q3_tile_kernel<MB, KS>, dim3(nwg), dim3(kThreads), Shape<MB, KS>::kSmem, stream, a);
}

}  // namespace

// Batches the tiled kernels serve.  Up to 64 rows go through the 64-row kernel of q3_gemm.hip (64 rows, K=8192, N=28672: 36.8 us
// there, 40.2 here; 32 rows 26.5 and 35.4; 58 rows, K=6464, N=13924 28.7 and 25.9), 65 to 96 rows of a narrow matrix through the
// one-launch kernel of q3_direct.hip (70 rows, K=4096, N=4096 8.7 us there, 17.6 here).
bool hq_q3_tiles_serve(int N, int M) { return M > 96 || (M > 64 && N > 4096); }

// What such a call takes (us): the tiles as planned, and the pre-pass in front of them (3.2 us, more for a long K and for its bytes).
float hq_q3_tiles_us(int cus, int K, int N, int M) {
  return tile_plan(cus, K, N, M).us + 3.2f + 0.0002f * K + (float)M * (float)K * (4.f / 4.5e6f);
}

int hq_q3_tiles_need(int cus, int K, int N, int M, bool cut_off, size_t* floats, size_t* counters) {
  *floats = *counters = 0;
  const int rows = rows_per_pass(K, M);
  for (int m0 = M > rows ? (M - 1) / rows * rows - rows : 0; m0 < M; m0 += rows) {  // the full pass and the last one
    const TilePlan p = tile_plan(cus, K, N, M - m0 < rows ? M - m0 : rows);
    size_t f = p.ap_floats + p.row_floats + p.partial_floats, c = p.counters;
    if (cut_off && p.cut < N) {  // one after the other in the same place
      if (p.direct.partial_floats > f) f = p.direct.partial_floats;
      if (p.direct.counters > c) c = p.direct.counters;
    }
    if (f > *floats) *floats = f;
    if (c > *counters) *counters = c;
  }
  return HQ_OK;
}

// Upper bound of hq_q3_tiles_need over every K <= max_K, any N and any M.
void hq_q3_tiles_bound(int cus, int max_K, size_t* floats, size_t* counters) {
  const size_t wgs = cus < kMaxWorkgroups ? cus : kMaxWorkgroups;
  // re-ordered activations, K padded to whole steps: 8192 rows of a short K, 32 MB of rows of a longer one, 1024 rows at least
  const size_t kpad = ((size_t)max_K + 255) / 256 * 256;
  const size_t of_32mb = ((size_t)16 << 20) / 2 + (size_t)8192 * 256 / 2;
  size_t ap = (size_t)8192 * kpad / 2 < of_32mb ? (size_t)8192 * kpad / 2 : of_32mb;
  if (ap < (size_t)1024 * kpad / 2) ap = (size_t)1024 * kpad / 2;
  // shares of divided tiles: one per workgroup, of the largest tile that is ever divided (a K of few steps is not)
  size_t tile = 0;
  for (const TileKind& kind : kKinds) {
    const int T = (max_K / 32 + 2 * kind.ks - 1) / (2 * kind.ks);
    bool divided = false;
    for (int t = 2; t <= T && !divided; ++t)
      for (int c = 2; c <= kMaxShares && c <= t; ++c) divided = divided || tile_us(kind, t, c) < tile_us(kind, t, 1);
    if (divided && (size_t)kind.tm * kind.tn > tile) tile = (size_t)kind.tm * kind.tn;
  }
  *floats = ap + 2 * 8192 + wgs * tile;
  *counters = wgs;
}

int hq_q3_tiles_launch(const void* x, const int32_t* qweight, const float* scales, const float* zeros, float* y, int K, int N,
                       int M, unsigned flags, hipStream_t stream, const HqQ3Scratch* fixed) {
  const HqDevice* dev = nullptr;
  int rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  size_t floats, ncounters;
  hq_q3_tiles_need(dev->cus, K, N, M, false, &floats, &ncounters);
  float* ap;
  unsigned* counters;
  if (fixed) {
    if (floats > fixed->tiles_floats || ncounters > fixed->ncounters) return HQ_ERR_TOO_LARGE;
    ap = fixed->tiles;
    counters = fixed->counters;
  } else {
    HqWorkspace ws;
    rc = hq_get_workspace(stream, floats, ncounters, &ws);
    if (rc != HQ_OK) return rc;
    ap = ws.partial;
    counters = ws.counters;
  }
  const int rows = rows_per_pass(K, M);
  for (int m0 = 0; m0 < M; m0 += rows) {
    const int Mb = M - m0 < rows ? M - m0 : rows;
    const TilePlan p = tile_plan(dev->cus, K, N, Mb);
    float* rowsum = ap + p.ap_floats;
    rc = hq_q3_gemm_prep_launch(reinterpret_cast<const _Float16*>(x) + (size_t)m0 * K, ap, rowsum, rowsum + p.Mpad, Mb, K,
                                p.Mpad, 2 * p.ks * p.T, counters, p.nshare > 1 ? p.counters : 0, stream);
    if (rc != HQ_OK) return rc;
    TileArgs a;
    a.w = reinterpret_cast<const uint32_t*>(qweight);
    a.Ap = reinterpret_cast<const unsigned char*>(ap);
    a.rowsum = rowsum; a.rowinv = rowsum + p.Mpad; a.partial = rowsum + p.row_floats;
    a.counters = counters;
    a.scales = scales; a.zeros = zeros; a.out = y + (size_t)m0 * N;
    a.M = Mb; a.N = N; a.G = K / 32; a.Mpad = p.Mpad; a.nmt = p.nmt; a.T = p.T; a.rounds = p.rounds; a.rest = p.rest;
    a.nshare = p.nshare; a.L = p.L; a.flags = flags;
    rc = p.tm == 128 ? launch_tiles<4, 2>(a, p.nwg, stream)
                     : (p.tn == 256 ? launch_tiles<2, 2>(a, p.nwg, stream) : launch_tiles<2, 4>(a, p.nwg, stream));
    if (rc == HQ_OK && p.cut < N)
      rc = hq_q3_direct_launch(p.direct, dev->cus, reinterpret_cast<const _Float16*>(x) + (size_t)m0 * K, qweight, scales, zeros,
                               y + (size_t)m0 * N, K, N, Mb, p.cut, flags, stream, fixed);
    if (rc != HQ_OK) return rc;
  }
  return HQ_OK;
}
