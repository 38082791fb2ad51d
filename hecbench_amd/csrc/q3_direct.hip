// Batched GPTQ 3-bit product in one launch, without a pre-pass, for the small and medium problems between the few rows of
// q3_block.hip and the many of q3_prefill.hip (fp16 activations, fp32 output):
//
//   out[m][n] = s[n] * sum_k A[m][k]*q[k][n]  -  z[n] * sum_k A[m][k]
//
// What bounds such a problem is latency: launches, the first data, and how fast one compute unit can pull its operands (64 KB in
// flight, 50 GB/s where HBM is among their sources).  The pre-pass of the other kernels was 3 to 5 us of 12 to 25, and their
// tiles, dividing K eight ways among workgroups, spent as long on adding up the shares.  So here
//   - activations are read as they lie, straight into LDS, and put in order on the way from LDS into the operand registers
//     (one byte permutation per register); nothing is scaled: the codes themselves become fp16 numbers, by one AND/OR per word
//     and v_cvt_scalef32_pk32_f16_fp6, which makes 32 of them at once (64 cycles; 3-bit fields as subnormals in place, as the
//     other kernels have them, need the activations scaled, and a multiplication for each to be rid of that: 0.38 -> 0.33 us for
//     256 elements of K);
//   - a tile is small, 32 rows by 64 or 128 columns, and its K is divided among the WAVES of a workgroup, each of which streams
//     its own operands through a ring of its own in LDS without ever meeting the others before the end (with operands shared
//     between waves and a barrier per step 13.4 instead of 10.3 us at 341 rows, K=4416, N=644);
//   - the rows' sums for the zero term come out of the operand registers (v_dot2_f32_f16).
// Measured, before -> now: 70 x 4096 x 4096 17.6 -> 8.7 us; 341 x 4416 x 644 21.6 -> 10.4; 39 x 4160 x 3176 16.6 -> 9.0; 128 x 4096 x
// 4096 18.0 -> 9.3; 64 x 4096 x 11008 18.4 -> 12.0; 210 x 6976 x 4592 28.7 -> 20.2; 23 x 1952 x 12980 12.6 -> 6.9; 0.3 of each of these
// by arguments that arrive in registers instead of a structure that is loaded first.
// Codes that are normal numbers also lose less in the matrix instruction, which aligns the products of a sum by their
// exponents: error against 64 bits 2e-7 of the result (2-norm) instead of 1.8e-6.
#include <type_traits>

#include "hq_internal.h"
#include "q3_tile.h"

namespace {

using namespace hq_q3;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u6v __attribute__((ext_vector_type(6)));
typedef uint32_t u16v __attribute__((ext_vector_type(16)));
typedef _Float16 h32 __attribute__((ext_vector_type(32)));

// Read six bits at a time the 96-bit string of a k-group and column is sixteen fp6 (e2m3) numbers: bits 0 to 2 of field f are
// code 2f, with the three above cleared the number code / 8; three bits further on, code 2f + 1.  Word w of the string: bits
// `first` and up of its fields, n of them.
constexpr uint32_t field_bits(int w, int first, int n) {
  uint32_t m = 0;
  for (int b = 0; b < 32; ++b)
    if ((32 * w + b) % 6 >= first && (32 * w + b) % 6 < first + n) m |= 1u << b;
  return m;
}

// A wave multiplies 32 rows by CB times 32 columns over its own part of every step of K (64 elements of 64 KS); the KS waves of a
// workgroup share a tile of 32 x 32 CB results and meet once, at its end.  Nothing a wave loads is read by another: each streams
// its operands through two stages of LDS of its own, without a barrier.
template <int CB, int KS>
struct Form {
  static constexpr int kThreads = 64 * KS;
  static constexpr int kTileM = 32, kTileN = 32 * CB;
  static constexpr int kABytes = kTileM * 128, kWBytes = 6 * kTileN * 4;  // a wave's stage: 128 bytes of every row, six packed rows
  static constexpr int kALoads = kABytes / 1024;           // LDS loads of a stage: activations,
  static constexpr int kWLoads = (kWBytes + 1023) / 1024;  // and packed rows, the last load by half of the lanes if CB is 2
  static constexpr int kLoads = kALoads + kWLoads, kStageBytes = kABytes + kWBytes;
  static constexpr int kUnits = 4 * CB;                    // groups of eight rows, every CB-th column
  static constexpr int kFinal = kUnits / KS;               // of which a wave finishes so many
  static constexpr int kWaveBytes = 2 * kStageBytes, kRing = KS * kWaveBytes, kMeet = KS * kUnits * 1024;
  static constexpr int kBulk = kRing > kMeet ? kRing : kMeet;
  static constexpr int kSums = 2 * KS * kTileM;            // floats: parts of the row sums
  static constexpr int kSmem = kBulk + (kSums + kTileM) * 4 + 16;
  static_assert(KS % 2 == 0, "odd parts of K enter negated");
  static_assert(CB == 2 || CB == 4, "a lane's columns are one LDS read");
  static_assert(kUnits % KS == 0, "every wave finishes as many units");
  static_assert(kSmem <= 160 * 1024, "LDS");
};

struct DirectArgs {
  const uint32_t* w;
  const _Float16* x;
  const float* scales;
  const float* zeros;
  float* out;
  float* partial;      // [tile][nshare][kTileM * kTileN]
  unsigned* counters;  // [tile], zero between calls
  int M, N, K, nmt, T, nshare, L, nwg;  // row tiles; steps of K, shares of L steps each; workgroups
  int ct0;             // column tiles in front of the first
  unsigned flags;
};

template <int CB, int KS>
__global__ __launch_bounds__(64 * KS, 2) void q3_direct_kernel(HQ_ARGS24) {
  // the first 14 dwords of the arguments (all that the loads need) arrive preloaded in scalar registers
  HqReader r(HQ_PASS24);
  DirectArgs a;
  a.w = r; a.x = r; a.M = r; a.N = r; a.K = r; a.nmt = r; a.T = r; a.nshare = r; a.L = r; a.nwg = r; a.ct0 = r; a.flags = r; a.scales = r; a.zeros = r;
  a.out = r; a.partial = r; a.counters = r;
  using S = Form<CB, KS>;
  typedef uint32_t wv_t __attribute__((ext_vector_type(CB)));
  extern __shared__ unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int kp = __builtin_amdgcn_readfirstlane(tid >> 6);  // part of K
  const int nl = lane & 31, kb = lane >> 5;
  const int G = a.K >> 5;
  // workgroup b runs on XCD b mod 8: an XCD takes consecutive tiles (row tiles of one column tile first), which share
  // weights and activations in its L2
  const int xcd = blockIdx.x & 7;
  const int v = xcd * (a.nwg >> 3) + min(xcd, a.nwg & 7) + (int)(blockIdx.x >> 3);
  const int tile = v / a.nshare, share = v - tile * a.nshare;
  const int ct_here = __builtin_amdgcn_readfirstlane(tile / a.nmt), mt = __builtin_amdgcn_readfirstlane(tile - ct_here * a.nmt);
  const int ct = a.ct0 + ct_here;
  const int t0 = share * a.L, len = min(a.L, a.T - t0);

  // ---- loader ----
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds + kp * S::kWaveBytes;
  const unsigned char* const abase = reinterpret_cast<const unsigned char*>(a.x + (size_t)mt * S::kTileM * a.K);
  // Activations keep their order: 16-byte piece c of a row's 128 bytes stands in column c ^ (row / 2 mod 8): the sixteen lanes
  // of a 128-bit LDS read pass, which are sixteen rows, then meet sixteen different bank groups.
  // Offsets of a step's pieces from its first.  In the last step of K a wave may have one k-group or none: it loads the last
  // k-group in place of those that are not there (and takes its codes as zero).
  constexpr int L0 = S::kALoads;
  uint32_t off[S::kLoads];
#pragma unroll
  for (int i = 0; i < L0; ++i) {
    const int row = i * 8 + (lane >> 3);
    off[i] = (uint32_t)(min(mt * S::kTileM + row, a.M - 1) - mt * S::kTileM) * (uint32_t)a.K * 2u +
             (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u + (uint32_t)kp * 128u;
  }
#pragma unroll
  for (int i = 0; i < S::kWLoads; ++i) {
    const int o = i * 1024 + (CB == 2 && i ? lane & 31 : lane) * 16, row = 6 * kp + o / (S::kTileN * 4), col = o % (S::kTileN * 4) / 4;
    off[L0 + i] = (uint32_t)row * (uint32_t)a.N * 4u + (uint32_t)min(ct * S::kTileN + col, a.N - 4) * 4u;
  }
  const int t_last = a.T - 1;
  const int missing = max(0, 2 * KS * t_last + 2 * kp + 2 - G);  // k-groups of this wave's last step, 2 and more: all
  auto back = [&](int l) {  // how far the last step's offset lies in front of off[l]
    const int shift = max(missing - 2, 0) + (missing > 1 ? 1 : 0);  // whole k-groups: the wave's first becomes the last of K
    bool second;                                                     // does the lane load for the wave's second k-group?
    if (l < L0) second = ((lane >> 2) ^ l) & 1;
    else second = ((l - L0) * 1024 + (CB == 2 && l > L0 ? lane & 31 : lane) * 16) / (S::kTileN * 4) >= 3;
    const int groups = shift + (second && missing > 0 ? 1 : 0);
    return (uint32_t)groups * (l < L0 ? 64u : 12u * (uint32_t)a.N);
  };
  // operands of step t into a stage
  auto dma = [&](int stage, int t, bool may_be_last) {
    const unsigned char* const ax = abase + (size_t)t * (128 * KS);
    const unsigned char* const wx = reinterpret_cast<const unsigned char*>(a.w) + (size_t)(6 * KS * t) * a.N * 4u;
#pragma unroll
    for (int l = 0; l < S::kLoads; ++l) {
      uint32_t o = off[l];
      if (may_be_last && t == t_last) o -= back(l);
      const uint32_t at = lds0 + stage * S::kStageBytes + l * 1024;
      if (l < L0) load_lds(at, o, ax);
      else if (CB != 2 || l == L0 || lane < 32) load_lds(at, o, wx);
    }
  };
  // waits until at most n of this wave's loads are in flight
  auto wait = [&](auto n) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory");
  };

  f16v acc[CB];
#pragma unroll
  for (int q = 0; q < CB; ++q)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[q][i] = 0.f;
  float rs = 0.f;

  const unsigned char* const ring = lds + kp * S::kWaveBytes;
  const unsigned char* const a_lane = ring + nl * 128;
  const unsigned char* const w_lane = ring + S::kABytes + (3 * kb * S::kTileN + CB * nl) * 4;
  u4v P[2];
  auto read_pieces = [&](int stage, int i0) {  // two of the four of the lane's k-group
#pragma unroll
    for (int i = 0; i < 2; ++i)
      P[i] = *reinterpret_cast<const u4v*>(a_lane + stage * S::kStageBytes + (((4 * kb + i0 + i) ^ ((nl >> 1) & 7)) * 16));
  };
  struct Words { wv_t v[3]; };
  auto read_w = [&](int stage, int t, bool may_be_last, Words& dst) {
    const bool real = !may_be_last || 2 * KS * t + 2 * kp + kb < G;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const wv_t x = *reinterpret_cast<const wv_t*>(w_lane + stage * S::kStageBytes + j * S::kTileN * 4);
#pragma unroll
      for (int c = 0; c < CB; ++c) dst.v[j][c] = real ? x[c] : 0u;
    }
  };
  // Column q's 32 codes as fp16 numbers code / 8: elements 0..15 the even codes, 16..31 the odd ones (odd parts of K negative).
  const uint32_t neg = kp & 1 ? 0xffffffffu : 0u;
  const uint32_t sign[3] = {neg & field_bits(0, 5, 1), neg & field_bits(1, 5, 1), neg & field_bits(2, 5, 1)};
  uint32_t keep[3] = {field_bits(0, 0, 3), field_bits(1, 0, 3), field_bits(2, 0, 3)};
#pragma unroll
  for (int i = 0; i < 3; ++i) asm("" : "+v"(keep[i]));  // in registers, so that the AND and the OR are one instruction
  auto codes = [&](const Words& words, int q) {
    uint32_t w[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) w[j] = words.v[j][q];
    u6v f;
    f[0] = (w[0] & keep[0]) | sign[0];
    f[1] = (w[1] & keep[1]) | sign[1];
    f[2] = (w[2] & keep[2]) | sign[2];
    f[3] = (__builtin_amdgcn_alignbit(w[1], w[0], 3) & keep[0]) | sign[0];
    f[4] = (__builtin_amdgcn_alignbit(w[2], w[1], 3) & keep[1]) | sign[1];
    f[5] = (w[2] >> 3 & keep[2]) | sign[2];
    return __builtin_bit_cast(u16v, __builtin_amdgcn_cvt_scalef32_pk32_f16_fp6(f, 1.f));
  };
  // and the activations in that order: operand j of a lane's 32, out of pieces 2 (j & 1) and the next
  auto rows_operand = [&](int j, u4v& dst) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const u4v& p = P[i >> 1];
      dst[i] = __builtin_amdgcn_perm(p[2 * (i & 1) + 1], p[2 * (i & 1)], j < 2 ? 0x05040100u : 0x07060302u);
    }
  };

  u4v A[4];
  u16v B;
  Words w;
  dma(0, t0, true);
  if (len > 1) dma(1, t0 + 1, true);
  if (len > 1) wait(std::integral_constant<int, S::kLoads>());
  else wait(std::integral_constant<int, 0>());
  read_w(0, t0, true, w);
  read_pieces(0, 0);
  rows_operand(0, A[0]);
  rows_operand(2, A[2]);
  read_pieces(0, 2);
  rows_operand(1, A[1]);
  rows_operand(3, A[3]);
  int stage = 0, s = 0;
  // A step: column by column of a lane's CB the codes and the products; under the last column the next step's operands come out
  // of LDS and are made.  MODE 2: loads the step after the next, 1: which may be the last of K, 0: none.
  auto step = [&](auto mode) {
    constexpr int MODE = decltype(mode)::value;
    // this step's operands are in registers, its stage is free
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (MODE) dma(stage, t0 + s + 2, MODE == 1);
    __builtin_amdgcn_sched_barrier(0);
    stage ^= 1;
    const h2 one = MODE == 2 || 2 * KS * (t0 + s) + 2 * kp + kb < G ? h2{(_Float16)1.f, (_Float16)1.f} : h2{(_Float16)0.f, (_Float16)0.f};
#pragma unroll
    for (int q = 0; q < CB; ++q) {
      B = codes(w, q);
      if (q == CB - 1) {
        wait(std::integral_constant<int, MODE ? S::kLoads : 0>());  // the next step's operands have to be in LDS
        read_pieces(stage, 0);
        read_w(stage, t0 + s + 1, MODE < 2, w);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        constexpr int kOrder[4] = {0, 2, 1, 3};  // operands 0 and 2 are made of the same pieces
        const int j = kOrder[jj];
        const u4v b = {B[4 * j], B[4 * j + 1], B[4 * j + 2], B[4 * j + 3]};
        acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, A[j]), __builtin_bit_cast(h8, b), acc[q], 0, 0, 0);
        if (q == (CB == 2 ? 0 : j & 1))
#pragma unroll
          for (int i = 0; i < 4; ++i)  // the sums of the rows
            rs = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, (uint32_t)A[j][i]), one, rs, false);
        if (q == CB - 1) {
          rows_operand(j, A[j]);
          if (jj == 1) read_pieces(stage, 2);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    ++s;
  };
  while (s < len - 3) step(std::integral_constant<int, 2>());
  while (s < len - 2) step(std::integral_constant<int, 1>());
  while (s < len) step(std::integral_constant<int, 0>());

  // ---- the parts of K meet: wave p finishes units p * kFinal and up (no load is in flight into LDS any more: the last steps
  // waited for theirs) ----
  constexpr int F = S::kFinal;
  constexpr int V = F < CB ? F : CB;  // adjacent columns of a wave's units
  typedef float fv_t __attribute__((ext_vector_type(V)));
  float* const sums = reinterpret_cast<float*>(lds + S::kBulk);  // [2 KS][kTileM], then the rows' sums
  float* const total = sums + S::kSums;
  f4v* const meet = reinterpret_cast<f4v*>(lds) + lane;
  auto first_row = [&](int i) { return (kp * F + i) / CB * 8 + 4 * kb; };  // of this wave's unit i
  const int first_col = ct * S::kTileN + CB * nl + kp * F % CB;
  f4v fin[F];
  sums[(2 * kp + kb) * S::kTileM + nl] = rs;
  __syncthreads();  // every wave is done with its stages
#pragma unroll
  for (int u = 0; u < S::kUnits; ++u) {
    f4v x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = acc[u % CB][4 * (u / CB) + e];
    meet[(u * KS + kp) * 64] = x;
  }
  if (tid < S::kTileM) {  // (the sums' parts were written ahead of the barrier)
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) t += sums[i * S::kTileM + tid];
    total[tid] = t;
  }
  asm volatile("" ::"s"(a.counters));  // the last arguments are here with the others, not behind the first LDS reads' wait
  __syncthreads();
  const int nc = min(first_col, a.N - V);
  const fv_t sc = *reinterpret_cast<const fv_t*>(a.scales + nc), zr = *reinterpret_cast<const fv_t*>(a.zeros + nc);
#pragma unroll
  for (int i = 0; i < F; ++i) {
    f4v x = meet[((kp * F + i) * KS) * 64];
#pragma unroll
    for (int p = 1; p < KS; ++p) {
      const f4v other = meet[((kp * F + i) * KS + p) * 64];
      x = p & 1 ? x - other : x + other;  // odd parts are the negated ones
    }
    const f4v t = *reinterpret_cast<const f4v*>(total + first_row(i));
#pragma unroll
    for (int e = 0; e < 4; ++e) fin[i][e] = sc[i % V] * (x[e] * 8.f) - zr[i % V] * t[e];  // codes enter as eighths
  }

  if (a.nshare > 1) {
    // A share of a divided tile: its results go out, every wave waits for their acknowledgement, the workgroup counts
    // itself at the memory side, and the last to arrive adds the shares in order of k.
    auto slot_of_share = [&](int c) {
      return reinterpret_cast<f4v*>(a.partial) + (size_t)(tile * a.nshare + c) * (S::kTileM * S::kTileN / 4) + tid;
    };
    f4v* dst = slot_of_share(share);
#pragma unroll
    for (int i = 0; i < F; ++i) hq_store_share(dst + i * S::kThreads, fin[i]);
    unsigned* last = reinterpret_cast<unsigned*>(total + S::kTileM);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const unsigned old = __hip_atomic_fetch_add(&a.counters[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *last = old == (unsigned)(a.nshare - 1);
      if (old == (unsigned)(a.nshare - 1))  // ready for the next call
        __hip_atomic_store(&a.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*last) return;
    constexpr int kAtOnce = F >= 4 ? 4 : 8;
    for (int c0 = 0; c0 < a.nshare; c0 += kAtOnce) {
      f4v x[kAtOnce * F];
#pragma unroll
      for (int k = 0; k < kAtOnce; ++k)
#pragma unroll
        for (int i = 0; i < F; ++i)
          x[k * F + i] = hq_load_share(slot_of_share(min(c0 + k, a.nshare - 1)) + i * S::kThreads);
      hq_wait_shares(x);
#pragma unroll
      for (int k = 0; k < kAtOnce; ++k)
        if (c0 + k < a.nshare) {
#pragma unroll
          for (int i = 0; i < F; ++i) fin[i] = c0 + k == 0 ? x[k * F + i] : fin[i] + x[k * F + i];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < F; i += V) {
    const int m0 = mt * S::kTileM + first_row(i), n = first_col;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (m0 + e < a.M && n < a.N) {
        fv_t* p = reinterpret_cast<fv_t*>(a.out + (size_t)(m0 + e) * a.N + n);
        fv_t o;
#pragma unroll
        for (int c = 0; c < V; ++c) o[c] = fin[i + c][e];
        if (a.flags & HQ_FLAG_ACCUMULATE) o += *p;
        __builtin_nontemporal_store(o, p);
      }
    }
  }
}

__global__ __launch_bounds__(256) void clear_counters(unsigned* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// Host arithmetic of a launch (the launch, the choice between the kernels and the size query share it).

// The workgroups and what they cost, fitted to 5700 timings of 520 problems on MI355X (spread about the fit: 7 %; the bases 0.25 lower since the arguments come
// in registers): a workgroup
// takes base_us and step_us for every step of 64 ks elements; workgroups that share a compute unit take their steps one after
// the other (their operands come through one queue), beyond per_cu of them in rounds; dividing a tile's K among c workgroups costs
// share_us + c * per_share_us.  Eight waves per workgroup where every compute unit has but one, four otherwise; 128 columns load
// fewer activations per weight, 64 divide smaller problems.
struct DirectKind {
  int tm, tn, ks, per_cu;
  float base_us, step_us, share_us, per_share_us;
};
constexpr DirectKind kKinds[4] = {{32, 64, 4, 3, 3.58f, 0.385f, 1.36f, 0.17f}, {32, 64, 8, 1, 3.95f, 0.575f, 1.54f, 0.12f},
                                  {32, 128, 4, 2, 3.81f, 0.574f, 1.2f, 0.35f}, {32, 128, 8, 1, 4.65f, 0.904f, 1.9f, 0.15f}};
constexpr int kMaxShares = 8;

HqQ3DirectPlan direct_plan_of(int cus, int K, int N, int M, int kind, int nshare) {
  const DirectKind& kd = kKinds[kind];
  HqQ3DirectPlan p;
  p.kind = kind;
  p.tm = kd.tm; p.tn = kd.tn; p.ks = kd.ks;
  p.nmt = (M + p.tm - 1) / p.tm;
  p.ntiles = p.nmt * ((N + p.tn - 1) / p.tn);
  p.T = (K / 32 + 2 * p.ks - 1) / (2 * p.ks);
  p.nshare = nshare < p.T ? nshare : p.T;
  p.L = (p.T + p.nshare - 1) / p.nshare;
  p.nshare = (p.T + p.L - 1) / p.L;
  const int wgs = p.ntiles * p.nshare, per_cu = (wgs + cus - 1) / cus;
  const float side = per_cu <= kd.per_cu ? (float)per_cu : (float)wgs / cus + 1.1f;
  p.us = kd.base_us + p.L * side * kd.step_us + (p.nshare > 1 ? kd.share_us + p.nshare * kd.per_share_us : 0.f);
  p.partial_floats = p.nshare > 1 ? (size_t)wgs * p.tm * p.tn : 0;
  p.counters = p.nshare > 1 ? p.ntiles : 0;
  return p;
}

template <int CB, int KS>
int launch(const DirectArgs& a, hipStream_t stream) {
  using S = Form<CB, KS>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&q3_direct_kernel<CB, KS>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, S::kSmem);
  if (attr != hipSuccess) return (int)attr;
  return hq_launch(q3_direct_kernel<CB, KS>, dim3(a.nwg), dim3(S::kThreads), S::kSmem, stream, a.w, a.x, a.M, a.N, a.K, a.nmt, a.T,
                   a.nshare, a.L, a.nwg, a.ct0, a.flags, a.scales, a.zeros, a.out, a.partial, a.counters);
}

}  // namespace

bool hq_q3_direct_can(int K, int N) { return K <= (1 << 24) && N <= (1 << 22); }  // offsets inside a step are 32-bit
bool hq_q3_direct_forced() {
  const int force = hq_tune(HQ_TUNE_Q3_TILES, -1);  // tests: 3 + kind + 10 * shares
  return force >= 0 && force % 10 >= 3 && force % 10 < 7;
}

HqQ3DirectPlan hq_q3_direct_plan(int cus, int K, int N, int M, bool undivided) {
  if (hq_q3_direct_forced()) {
    const int force = hq_tune(HQ_TUNE_Q3_TILES, -1);
    return direct_plan_of(cus, K, N, M, force % 10 - 3, undivided || force < 10 ? 1 : force / 10);
  }
  HqQ3DirectPlan best = direct_plan_of(cus, K, N, M, 0, 1);
  for (int kind = 0; kind < 4; ++kind)
    for (int c = 1; c <= (undivided ? 1 : kMaxShares); ++c) {
      const HqQ3DirectPlan p = direct_plan_of(cus, K, N, M, kind, c);
      if (p.nshare != c) continue;
      const int64_t wgs = (int64_t)p.ntiles * c;
      if (c > 1 && wgs > 2 * cus) break;                       // bounds the workspace: 2 * cus * 32 * 128 floats
      if (kKinds[kind].per_cu == 1 && wgs > cus) continue;
      if (p.us < best.us) best = p;
    }
  return best;
}

int hq_q3_direct_launch(HqQ3DirectPlan p, int cus, const void* x, const int32_t* qweight, const float* scales, const float* zeros,
                        float* y, int K, int N, int M, int col0, unsigned flags, hipStream_t stream, const HqQ3Scratch* fixed) {
  // without room for the shares' sums no tile is divided
  if (p.nshare > 1 && (fixed ? p.partial_floats > fixed->tiles_floats || p.counters > fixed->ncounters
                             : hq_workspace_out_of_reach(stream, p.partial_floats, p.counters)))
    p = hq_q3_direct_plan(cus, K, N - col0, M, true);
  int rc = HQ_OK;
  DirectArgs a;
  a.partial = nullptr; a.counters = nullptr;
  if (p.nshare > 1 && fixed) {
    a.partial = fixed->tiles;
    a.counters = fixed->counters;
    // shared by every call on this device: a call that was cut short may have left counts behind
    hipLaunchKernelGGL(clear_counters, dim3((p.ntiles + 255) / 256), dim3(256), 0, stream, a.counters, p.ntiles);
    rc = hq_launch_status();
    if (rc != HQ_OK) return rc;
  } else if (p.nshare > 1) {
    HqWorkspace ws;
    rc = hq_get_workspace(stream, p.partial_floats, p.counters, &ws);
    if (rc != HQ_OK) return rc;
    a.partial = ws.partial;
    a.counters = ws.counters;
  }
  a.w = reinterpret_cast<const uint32_t*>(qweight);
  a.x = reinterpret_cast<const _Float16*>(x);
  a.scales = scales; a.zeros = zeros; a.out = y;
  a.M = M; a.N = N; a.K = K; a.nmt = p.nmt; a.T = p.T; a.nshare = p.nshare; a.L = p.L; a.nwg = p.ntiles * p.nshare;
  a.ct0 = col0 / p.tn;
  a.flags = flags;
  switch (p.kind) {
    case 0: return launch<2, 4>(a, stream);
    case 1: return launch<2, 8>(a, stream);
    case 2: return launch<4, 4>(a, stream);
    default: return launch<4, 8>(a, stream);
  }
}
