// Per-token int8 activation quantisation (static / dynamic scale, with or without an
// asymmetric zero point) for gfx950.
//
// Replaces static_scaled_int8_quant / dynamic_scaled_int8_quant and their four kernels
// (src/quantVLLM-hip/main.cu:11-168 in the HeCBench tree; helpers in
// src/quantVLLM-cuda/utils.h).  Bit-exact contract: fp32 IEEE division, round to nearest
// even, saturation, exactly as the reference's host loops (src/quantVLLM-cuda/reference.h).
//
// HBM-bound: 3 bytes per fp16 / bf16 element, 5 per fp32 element.  The tensor is cut into units of
// eight consecutive elements on a grid anchored at element 0 of the tensor, not of the row, so that a
// unit is one aligned 128-bit load (two for fp32) and one 64-bit store whatever the hidden size is
// (the reference's run size is 5137); a unit that straddles a row boundary is masked.
//   static : no row structure at all, a flat grid-stride loop over the units.
//   dynamic: a wave per row up to 1536 elements, a workgroup per row beyond; the row stays in registers
//            between the max / min pass and the quantise pass (one read of x, up to 10240 elements);
//            one launch slot per row, many workgroups per CU.
// The division by a scale shared by many elements: fp32 elements are multiplied by its reciprocal wherever that provably
// rounds to the same integer (the product is further from a tie than its error bound, or saturates either way), the other
// lanes divide; 16-bit elements, among which ties are common, get the rounded quotient in three operations (fast8).
// 4096 x 5137, us, before -> now: bf16 static 14.7 -> 11.6, with zero point 15.7 -> 11.7, dynamic with zero point 17.5 -> 13.5;
// fp16 12.4 -> 11.8, 13.0 -> 12.0, 15.9 -> 14.0.
#include "hq_internal.h"

namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

struct bf16_t { uint16_t bits; };  // bfloat16 = the upper half of an fp32

// src/quantVLLM-cuda/utils.h:9-24
// The saturation is done on the converted integer (the hardware conversion saturates at the int32 range
// and turns a NaN into 0, as the conversion of the clamped float did): one integer median instead of
// two compares and two selects per element.
__device__ __forceinline__ int float_to_int8_rn(float x) {
  const float dst = rintf(x);
  int r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(dst));
  return min(max(r, -128), 127);
}
// src/quantVLLM-cuda/utils.h:26-50: round to nearest even, saturating at the int32 range.  The
// hardware conversion saturates by itself (and turns a NaN into 0); it is written as an instruction
// because the C conversion of an out-of-range value is undefined.
__device__ __forceinline__ int float_to_int32_rn(float x) {
  const float dst = rintf(x);
  int r;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(dst));
  return r;
}
// src/quantVLLM-cuda/utils.h:52-61 (saturating add of the zero point happens in int32)
__device__ __forceinline__ int int32_to_int8(int x) { return x < -128 ? -128 : (127 < x ? 127 : x); }

constexpr int kVec = 8;  // elements per unit

// One unit of raw data: 16 bytes of fp16 / bf16 or 32 bytes of fp32.
template <typename T> struct Raw { u4v w[sizeof(T) == 4 ? 2 : 1]; };

template <typename T>
__device__ __forceinline__ Raw<T> load_unit(const T* __restrict__ base, int64_t unit) {
  Raw<T> r;
  const u4v* p = reinterpret_cast<const u4v*>(base + unit * kVec);
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) == 4 ? 2 : 1); ++i) r.w[i] = __builtin_nontemporal_load(p + i);
  return r;
}
// A unit that reaches past the end of the tensor: element by element, zeros beyond.
template <typename T>
__device__ __forceinline__ Raw<T> load_unit_tail(const T* __restrict__ base, int64_t unit, int64_t total) {
  Raw<T> r;
  T tmp[kVec];
#pragma unroll
  for (int i = 0; i < kVec; ++i) {
    const int64_t e = unit * kVec + i;
    tmp[i] = e < total ? base[e] : T{};
  }
  __builtin_memcpy(&r, tmp, sizeof(r));
  return r;
}
__device__ __forceinline__ void unpack(const Raw<float>& r, float (&v)[kVec]) {
#pragma unroll
  for (int i = 0; i < kVec; ++i) v[i] = __uint_as_float(r.w[i >> 2][i & 3]);
}
__device__ __forceinline__ void unpack(const Raw<_Float16>& r, float (&v)[kVec]) {
#pragma unroll
  for (int i = 0; i < kVec; ++i)
    v[i] = (float)__builtin_bit_cast(_Float16, (uint16_t)(r.w[0][i >> 1] >> (16 * (i & 1))));
}
__device__ __forceinline__ void unpack(const Raw<bf16_t>& r, float (&v)[kVec]) {
#pragma unroll
  for (int i = 0; i < kVec; ++i)
    v[i] = __uint_as_float((i & 1) ? (r.w[0][i >> 1] & 0xffff0000u) : (r.w[0][i >> 1] << 16));
}

// y[i] = element i * m.  An fp16 element is converted and multiplied by one mixed-precision instruction
// (the added +0 only turns a product of -0 into +0, which rounds to the same integer).
template <typename T>
__device__ __forceinline__ void products(const Raw<T>& r, float m, float (&y)[kVec]) {
  float v[kVec];
  unpack(r, v);
#pragma unroll
  for (int i = 0; i < kVec; ++i) y[i] = v[i] * m;
}
__device__ __forceinline__ void products(const Raw<_Float16>& r, float m, float (&y)[kVec]) {
#pragma unroll
  for (int i = 0; i < kVec / 2; ++i) {
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(y[2 * i]) : "v"(r.w[0][i]), "v"(m));
    asm("v_fma_mix_f32 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(y[2 * i + 1]) : "v"(r.w[0][i]), "v"(m));
  }
}

// Running maximum and minimum of whole units.  fp16 units are scanned as packed halves (the maximum of
// magnitudes on the bits with the signs cleared), everything else as converted floats.
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
template <typename T, bool AZP>
struct UnitScan {
  __device__ __forceinline__ void add(const Raw<T>& r, float& mx, float& mn) {
    float v[kVec];
    unpack(r, v);
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
      if (AZP) { mx = fmaxf(mx, v[i]); mn = fminf(mn, v[i]); }
      else mx = fmaxf(mx, fabsf(v[i]));
    }
  }
  __device__ __forceinline__ void fold(float&, float&) {}
};
template <bool AZP>
struct UnitScan<_Float16, AZP> {
  h2v hi, lo;
  __device__ __forceinline__ UnitScan() {
    const _Float16 inf = (_Float16)__builtin_inff();
    hi = AZP ? h2v{-inf, -inf} : h2v{(_Float16)0.f, (_Float16)0.f};
    lo = h2v{inf, inf};
  }
  __device__ __forceinline__ void add(const Raw<_Float16>& r, float&, float&) {
#pragma unroll
    for (int i = 0; i < kVec / 2; ++i) {
      const h2v x = __builtin_bit_cast(h2v, AZP ? r.w[0][i] : (r.w[0][i] & 0x7fff7fffu));
      hi = __builtin_elementwise_max(hi, x);
      if (AZP) lo = __builtin_elementwise_min(lo, x);
    }
  }
  __device__ __forceinline__ void fold(float& mx, float& mn) {
    mx = fmaxf(mx, fmaxf((float)hi.x, (float)hi.y));
    if (AZP) mn = fminf(mn, fminf((float)lo.x, (float)lo.y));
  }
};

// Running maximum and minimum of bf16 units as packed integers, a unit of eight in twelve instructions (as converted floats in 16; without
// a zero point eight, 12): a float is a sign and a magnitude, so the largest number, where one is positive, is the largest signed
// integer (the maximum begins above zero), and the smallest the largest unsigned one, or, where none is negative, the smallest.  What is
// not in the row counts as zeros, or as ones for that smallest.  A wave with a NaN scans again as floats, which drop it; that the others
// have none spares the second pass its test.
// With zero point, us, floats -> bits: 4096 x 5137 14.2 -> 13.6, 2000 x 1399 5.61 -> 5.29, 8192 x 401 8.30 -> 7.87, 1452 x 14519 14.6 ->
// 13.65, without 6001 x 1003 6.61 -> 6.26.  Rows of whole 512 elements up to 4096 do not gain (4096 x 4096 10.5 -> 10.6, 6000 x 2048
// 10.2 -> 10.2, but 4096 x 8192 18.7 -> 18.1), nor those that divide 512, whose lanes have one unit each (8000 x 128 4.47 -> 4.59, 20000 x
// 32 8.10 -> 8.28), nor, without a zero point, those of whole units (1992 x 168 2.78 -> 2.83, 4000 x 264 3.61 -> 3.66): these are scanned
// as floats, as is fp16, whose packed maximum is as short.
typedef short s2v __attribute__((ext_vector_type(2)));
typedef unsigned short us2v __attribute__((ext_vector_type(2)));
template <bool AZP>
struct BitScan {
  static constexpr uint32_t kInf = 0x7f80u;
  s2v hi = {0, 0};
  us2v most = {0, 0}, least = {0xffff, 0xffff};  // most, without a zero point: of the magnitudes
  // The bits of word i that belong to the row: elements [lo, end) of the unit.
  static __device__ __forceinline__ uint32_t inside(int i, int lo, int end) {
    return (lo <= 2 * i && end > 2 * i ? 0xffffu : 0u) | (lo <= 2 * i + 1 && end > 2 * i + 1 ? 0xffff0000u : 0u);
  }
  template <bool CUT>  // the row's first or last unit
  __device__ __forceinline__ void add(const Raw<bf16_t>& r, int lo, int end) {
#pragma unroll
    for (int i = 0; i < kVec / 2; ++i) {
      const uint32_t in = CUT ? inside(i, lo, end) : 0xffffffffu;
      const uint32_t x = r.w[0][i] & (AZP ? in : in & 0x7fff7fffu);
      if (AZP) {
        hi = __builtin_elementwise_max(hi, __builtin_bit_cast(s2v, x));
        least = __builtin_elementwise_min(least, __builtin_bit_cast(us2v, x | ~in));
      }
      most = __builtin_elementwise_max(most, __builtin_bit_cast(us2v, x));
    }
  }
  // The lane's maximum and minimum; whether the wave has a NaN.
  __device__ __forceinline__ bool fold(float& mx, float& mn) {
    const uint32_t h = (uint32_t)max((int)hi.x, (int)hi.y), m = max((uint32_t)most.x, (uint32_t)most.y);
    const uint32_t l = m >= 0x8000u ? m : min((uint32_t)least.x, (uint32_t)least.y);
    mx = fmaxf(mx, __uint_as_float((AZP ? h : m) << 16));
    if (AZP && l != 0xffffu) mn = fminf(mn, __uint_as_float(l << 16));  // (all ones: no element at all)
    return __builtin_amdgcn_ballot_w64(h > kInf || m > ((AZP ? 0x8000u : 0u) | kInf)) != 0;
  }
};

// Makes the compiler forget what it knows about a unit's bits, so that the values converted for the
// first pass are not kept alive (at twice the registers of the raw data) for the second.
template <typename T>
__device__ __forceinline__ void forget(Raw<T>& r) {
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) == 4 ? 2 : 1); ++i)
    asm volatile("" : "+v"(r.w[i]));
}

// The low bytes of four integers as one word, a first: byte selects instead of masks and shifts.
__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
  const uint32_t lo = __builtin_amdgcn_perm((uint32_t)b, (uint32_t)a, 0x0c0c0400u);
  const uint32_t hi = __builtin_amdgcn_perm((uint32_t)d, (uint32_t)c, 0x04000c0cu);
  return lo | hi;
}

// Stores elements [lo, hi) of a unit's eight results; all eight as one 64-bit store.  STREAM: as a
// write-through nontemporal store, which the one-pass static kernels gain from (14.2 -> 13.5 us at 4096 x 5137
// fp16) and the two-pass dynamic kernels lose by (18.5 -> 22.9 us).
template <bool STREAM>
__device__ __forceinline__ void store_unit(int8_t* __restrict__ out, int64_t unit, const int (&q)[kVec], int lo, int hi,
                                           bool aligned) {
  int8_t* p = out + unit * kVec;
  if (lo == 0 && hi == kVec && aligned) {
    u2v w;
    w.x = pack4(q[0], q[1], q[2], q[3]);
    w.y = pack4(q[4], q[5], q[6], q[7]);
    if (STREAM) hq_store_stream(reinterpret_cast<hq_u2v*>(p), w);
    else __builtin_nontemporal_store(w, reinterpret_cast<u2v*>(p));
  } else if (aligned) {
    // a unit shared with the neighbouring row: the fewest naturally aligned pieces that cover [lo, hi)
    // (a store instruction costs the same whatever it carries, and the other lanes wait for it)
    uint32_t w[2];
    w[0] = pack4(q[0], q[1], q[2], q[3]);
    w[1] = pack4(q[4], q[5], q[6], q[7]);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const bool whole = lo <= 4 * d && hi >= 4 * d + 4;
      if (whole) reinterpret_cast<uint32_t*>(p)[d] = w[d];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int b = 4 * d + 2 * h;
        const bool half = !whole && lo <= b && hi >= b + 2;
        if (half) reinterpret_cast<uint16_t*>(p)[2 * d + h] = (uint16_t)(w[d] >> (16 * h));
        if (!whole && !half) {
          if (lo <= b && hi > b) p[b] = (int8_t)q[b];
          if (lo <= b + 1 && hi > b + 1) p[b + 1] = (int8_t)q[b + 1];
        }
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < kVec; ++i)
      if (i >= lo && i < hi) p[i] = (int8_t)q[i];
  }
}

// Division by a scale that many elements share.  y = v * (1 / s) differs from the rounded quotient q by
// less than 1.5 * 2^-23 |q| (2^-24 relative each for the reciprocal, the product and the quotient itself),
// so both round to the same integer unless y is within that of a tie; the checks below allow twice as
// much, 3 * 2^-23 |y|, which also covers their own rounding.  Where the result saturates the quotient
// need not be known at all.  The reciprocal must be a normal number for that bound.
struct Divisor {
  float s, r;
  bool usable;
  __device__ __forceinline__ explicit Divisor(float scale) : s(scale), r(1.0f / scale) {
    const float a = fabsf(scale);
    usable = a >= 0x1p-100f && a <= 0x1p100f;
  }
};

// float_to_int8_rn(v / s) or, with AZP, int32_to_int8(float_to_int32_rn(v / s) + azp), for eight values.
template <bool AZP, typename T>
__device__ __forceinline__ void quantise8(const Raw<T>& raw, const Divisor& d, int azp, int (&q)[kVec]) {
  float y[kVec];
  products(raw, d.r, y);
  auto divide = [&]() {
    float v[kVec];
    unpack(raw, v);
#pragma unroll
    for (int i = 0; i < kVec; ++i) y[i] = v[i] / d.s;
  };
  if (!AZP) {
    // Without a zero point only |y| < 129 can end anywhere but at a bound, and there 3 * 2^-23 |y| is less
    // than 2^-15: one constant margin for all eight, taken on the largest distance of a product from its
    // nearest integer.  The subtraction is exact and must stay one (contracted into a multiply-add it
    // would return the rounding error of products beyond 2^23 and send those to the division).  A NaN
    // distance - an infinite or NaN input - drops out of the maximum: such a product converts to the same
    // bound, or to 0, as the quotient.
#pragma clang fp contract(off)
    float worst = 0.f;
#pragma unroll
    for (int i = 0; i < kVec; ++i) worst = fmaxf(worst, fabsf(y[i] - rintf(y[i])));
    const bool exact = !d.usable || !(worst <= 0.5f - 0x1p-15f);
    if (__builtin_amdgcn_ballot_w64(exact)) divide();
#pragma unroll
    for (int i = 0; i < kVec; ++i) q[i] = float_to_int8_rn(y[i]);
    return;
  }
  // With a zero point any quotient may matter: the margin is relative (a subnormal product has no
  // relative bound and no tie near it either); it reaches 0.5, i.e. sends the unit to the division, from
  // |y| = 2^20.4 on.  One comparison for the largest of the eight; a NaN drops out as above.
  float worst = 0.f;
  {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
      const float dist = fabsf(y[i] - rintf(y[i]));  // distance to the nearest integer
      worst = fmaxf(worst, fmaf(fabsf(y[i]), 0x1.8p-22f, dist));
    }
  }
  const bool exact = !d.usable || !(worst < 0.5f - 0x1p-24f);
  if (__builtin_amdgcn_ballot_w64(exact)) divide();
#pragma unroll
  for (int i = 0; i < kVec; ++i) q[i] = int32_to_int8(float_to_int32_rn(y[i]) + azp);
}

// ---- rows of 16-bit elements with an ordinary scale ----------------------------------------------------------------
// 16-bit elements are few distinct numbers, and a row's scale is made of two of them: exact ties are common (one element
// in 500 of a bf16 row), and with 512 elements in a wave's unit the division of quantise8 ran for most units - 17.6
// against 13.1 us without it at 4096 x 5137 bf16 with zero point.  Here every quotient is the rounded one, in three
// operations: with r the rounded reciprocal of s and q0 = v * r, q0 + r * (v - q0 * s) in fused operations is the correctly
// rounded v / s (Markstein's theorem; s must not have a mantissa of all ones, and nothing may overflow).
// Integers up to 2^22 in magnitude are the low bits of 1.5 * 2^23 + integer, so one addition rounds to the nearest
// integer and leaves its low byte in place: no conversion and no rounding instruction.
constexpr float kMagic = 12582912.f;

// What a row's results are: products with a multiplier, rounded quotients, or those with a zero point on top.
enum FastMode { kProduct, kQuotient, kQuotientAzp };
template <FastMode MODE>
struct FastRow {
  bool usable;
  float m, s, azp;  // multiplier or 1 / s
  // a scale of ordinary magnitude (its element of largest magnitude `most`, where that is known, as well)
  __device__ __forceinline__ FastRow(float mul, const Divisor& d, int azp_, float most = 1.f) {
    usable = d.usable && most >= 0x1p-100f && most <= 0x1p100f;
    // zero points beyond saturate whatever the quotient; a quotient beyond 2^22 saturates whatever its last bit
    if (MODE != kProduct)
      usable = usable && (__float_as_uint(d.s) & 0x7fffffu) != 0x7fffffu && azp_ >= -65536 - 256 && azp_ <= 65536 + 256;
    m = MODE == kProduct ? mul : d.r; s = d.s; azp = (float)azp_;
  }
};

// y[i] = element i - q[i] * s, rounded once
template <typename T>
__device__ __forceinline__ void residues(const Raw<T>& r, const float (&q)[kVec], float s, float (&y)[kVec]) {
  float v[kVec];
  unpack(r, v);
#pragma unroll
  for (int i = 0; i < kVec; ++i) y[i] = fmaf(-q[i], s, v[i]);
}
__device__ __forceinline__ void residues(const Raw<_Float16>& r, const float (&q)[kVec], float s, float (&y)[kVec]) {
#pragma unroll
  for (int i = 0; i < kVec / 2; ++i) {
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel_hi:[0,0,1]" : "=v"(y[2 * i]) : "v"(q[2 * i]), "v"(s), "v"(r.w[0][i]));
    asm("v_fma_mix_f32 %0, -%1, %2, %3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(y[2 * i + 1]) : "v"(q[2 * i + 1]), "v"(s), "v"(r.w[0][i]));
  }
}

// The eight results of a unit, as low bytes; CHECKED: false if a quotient is a NaN (a NaN element, or an overflow on the way).
template <bool CHECKED, FastMode MODE, typename T>
__device__ __forceinline__ bool fast8(const Raw<T>& raw, const FastRow<MODE>& row, int (&q)[kVec]) {
  float t[kVec];
  bool ordered = true;
  if (MODE != kProduct) {
    float q0[kVec], rest[kVec], any = 0.f;
    products(raw, row.m, q0);
    residues(raw, q0, row.s, rest);
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
#pragma clang fp contract(off)
      t[i] = fmaf(rest[i], row.m, q0[i]) + kMagic;
      if (MODE == kQuotientAzp) t[i] = t[i] + row.azp;
      if (CHECKED) any = __builtin_elementwise_maximum(any, t[i]);  // a NaN stays
    }
    ordered = any == any;
#pragma unroll
    for (int i = 0; i < kVec; ++i) t[i] = __builtin_amdgcn_fmed3f(t[i], kMagic - 128.f, kMagic + 127.f);
  } else {
    // |product| <= 127 (1 + 2^-22), which rounds to 127 at most; two roundings, as in the definition.  A NaN leaves zero in
    // the low byte: a 16-bit NaN's payload ends above it.
    products(raw, row.m, t);
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
#pragma clang fp contract(off)
      t[i] = t[i] + kMagic;
    }
  }
#pragma unroll
  for (int i = 0; i < kVec; ++i) q[i] = (int)__float_as_uint(t[i]);
  return ordered;
}

// ---- static scale: elementwise over the whole tensor ---------------------------------------------
constexpr int kStaticUnroll = 2;

template <typename T, bool AZP>
__device__ __forceinline__ void static_quant_body(const T* __restrict__ in, int8_t* __restrict__ out, float scale, int azp,
                                                  int64_t total, int aligned) {
  const Divisor d(scale);
  const FastRow<AZP ? kQuotientAzp : kQuotient> row(0.f, d, azp);
  const int64_t units = (total + kVec - 1) / kVec;
  const int64_t full = aligned ? total / kVec : 0;  // units loaded whole: inside the tensor, pointers aligned
  const int64_t stride = (int64_t)gridDim.x * 256;
  for (int64_t u0 = (int64_t)blockIdx.x * 256 + threadIdx.x; u0 < units; u0 += stride * kStaticUnroll) {
    Raw<T> raw[kStaticUnroll];
#pragma unroll
    for (int k = 0; k < kStaticUnroll; ++k) {
      const int64_t u = u0 + k * stride;
      if (u < full) raw[k] = load_unit(in, u);
      else if (u < units) raw[k] = load_unit_tail(in, u, total);
      else raw[k] = Raw<T>{};
    }
#pragma unroll
    for (int k = 0; k < kStaticUnroll; ++k) {
      const int64_t u = u0 + k * stride;
      int q[kVec];
      if (!(sizeof(T) == 2 && row.usable && !__builtin_amdgcn_ballot_w64(!fast8<true>(raw[k], row, q))))
        quantise8<AZP>(raw[k], d, azp, q);
      if (u < units) store_unit<true>(out, u, q, 0, (int)min((int64_t)kVec, total - u * kVec), aligned);
    }
  }
}
template <typename T, bool AZP>
__global__ __launch_bounds__(256) void static_quant_kernel(HQ_ARGS12) {
  HqReader r(HQ_PASS12);
  const T* const in = r;
  int8_t* const out = r;
  const float scale = r;
  const int azp = r;
  const int64_t total = r;
  const int aligned = r;
  static_quant_body<T, AZP>(in, out, scale, azp, total, aligned);
}

// ---- dynamic scale: LANES threads per row --------------------------------------------------------
// Maximum of a and minimum of b over the LANES threads of a row.
// (Neither is a NaN: the scans drop them.)  Within a wave six rounds of shuffles took about three times as long.
template <int LANES>
__device__ __forceinline__ void row_max_min(float& a, float& b, float* lds) {
  a = hq_wave(a, HqMax());
  b = hq_wave(b, HqMin());
  if (LANES > 64) {  // the row spans the workgroup
    const int wv = threadIdx.x >> 6;
    constexpr int W = LANES / 64;
    if ((threadIdx.x & 63) == 0) { lds[wv] = a; lds[W + wv] = b; }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w) { a = fmaxf(a, lds[w]); b = fminf(b, lds[W + w]); }
  }
}

// LANES threads per row (a wave, or the workgroup), so 256 / LANES rows per workgroup and one workgroup
// for every 256 / LANES rows: nothing loops over rows.  KEEP units per thread stay in registers between
// the max / min pass and the quantise pass; a longer row streams the rest twice.  (Workgroups that walked
// over several rows, the next rows' loads in flight during the reduction, the quantisation and the stores,
// needed twice the registers for half the waves per CU and measured 18.8 us where this takes 14.0, 4096
// rows of 5137 fp16: the hardware overlaps one row's stores with another's loads by itself when enough
// workgroups fit a CU.)
// WHOLE: both pointers are aligned and the tensor is a whole number of units, so every unit is loaded whole; EVEN: so is every row, of up
// to 4096 elements, as far as floats scan it as fast (bf16 only, see BitScan); TAIL: aligned,
// but the tensor's last unit is cut (it alone, in the last row, is loaded element by element); ANY: other pointers.  (With
// ANY in the place of TAIL 1452 rows of 14519 bf16 took 35.6 us.)
// 64 registers for the 16-bit types, i.e. eight waves per SIMD, where nothing spills for it (one more register cost bf16 rows of 16384 22.3 -> 26.2 us).
enum RowMode { WHOLE, EVEN, TAIL, ANY };
constexpr int row_threads(int lanes) { return lanes < 256 ? 256 : lanes; }

template <typename T, bool AZP, int LANES, int KEEP, RowMode MODE>
__device__ __forceinline__ void dynamic_quant_body(const T* __restrict__ in, int8_t* __restrict__ out, float* __restrict__ scales,
                                                   int32_t* __restrict__ azps, int64_t tokens, int hidden) {
  constexpr bool aligned = MODE != ANY;
  __shared__ float lds[2 * LANES / 64];
  const int lane = threadIdx.x % LANES;
  const int64_t total = tokens * hidden;
  // uniform over the wave (LANES == 64) or the workgroup
  const int64_t token = LANES == 64 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  if (token >= tokens) return;
  // The row's units, and the multiple of 64 at or before its first: lanes are laid over the units from
  // there, so that a wave's loads and stores cover whole 128-byte lines of the output (256 of the
  // input) except at the row's ends.  Everything per row is uniform: base pointers at that multiple of
  // 64, and 32-bit unit numbers j relative to it (valid in [first, end)).
  const int64_t g0 = token * hidden;
  const int64_t u_first = g0 / kVec;
  const int64_t ubase = u_first & ~(int64_t)63;
  const int first = (int)(u_first - ubase);
  const int end = (int)((g0 + hidden + kVec - 1) / kVec - ubase);
  const int head = (int)(g0 - u_first * kVec);  // elements of the first unit that belong to the row before
  const T* row_in = in + ubase * kVec;
  int8_t* row_out = out + ubase * kVec;
  // the last unit of the row that lies in the tensor whole (the tensor has one)
  const int last = MODE == TAIL ? (int)(min(ubase + end, total / kVec) - ubase) - 1 : end - 1;
  auto fetch = [&](int j) {
    return MODE == WHOLE || MODE == EVEN || (MODE == TAIL && j <= last) ? load_unit(row_in, j) : load_unit_tail(in, ubase + j, total);
  };

  Raw<T> keep[KEEP];
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    const int j = lane + k * LANES;
    // whole units are loaded without a branch, so that the loads stay one straight run the waits can
    // count; a unit outside the row repeats the row's first or last
    if (MODE != ANY) keep[k] = load_unit(row_in, min(max(j, first), last));
    else if (j >= first && j < end) keep[k] = fetch(j);
  }
  if (MODE == TAIL && last < end - 1) {  // the rows that reach it only
#pragma unroll
    for (int k = 0; k < KEEP; ++k)
      if (lane + k * LANES == end - 1) keep[k] = load_unit_tail(in, ubase + end - 1, total);
  }

  // reference initial values: max starts at FLT_MIN (smallest positive normal), min at FLT_MAX
  // (reference.h:71-72); the symmetric variant starts its absmax at 0 (reference.h:43)
  float mx = AZP ? 1.17549435e-38f : 0.f;
  float mn = 3.40282347e+38f;
  auto part = [&](int j, int& lo, int& hi) {  // elements of unit j that belong to the row
    const int rel = (j - first) * kVec - head;  // row position of the unit's element 0
    lo = max(-rel, 0);
    hi = min(hidden - rel, kVec);
  };
  auto scan_kept = [&](auto&& scan) {
#pragma unroll
    for (int k = 0; k < KEEP; ++k) {
      const int j = lane + k * LANES;
      if (j >= first && j < end) scan(keep[k], j);
    }
  };
  auto scan_rest = [&](auto&& scan) {
    for (int j = lane + KEEP * LANES; j < end; j += LANES) scan(fetch(j), j);
  };
  auto scan_floats = [&](const Raw<T>& raw, int j) {
    int lo, hi;
    part(j, lo, hi);
    float v[kVec];
    unpack(raw, v);
#pragma unroll
    for (int i = 0; i < kVec; ++i)
      if (i >= lo && i < hi) {
        if (AZP) { mx = fmaxf(mx, v[i]); mn = fminf(mn, v[i]); }
        else mx = fmaxf(mx, fabsf(v[i]));
      }
  };
  constexpr bool by_bits = __is_same(T, bf16_t) && MODE != EVEN;
  bool nan = false;  // by_bits: among the elements of the wave
  if constexpr (by_bits) {
    const float mx0 = mx, mn0 = mn;
    BitScan<AZP> bits;
    auto add = [&](const Raw<T>& raw, int j) {
      int lo, hi;
      part(j, lo, hi);
      if (lo == 0 && hi == kVec) bits.template add<false>(raw, 0, kVec);  // all but the row's first and last unit
      else bits.template add<true>(raw, lo, hi);
    };
    scan_kept(add);
    scan_rest(add);
    nan = bits.fold(mx, mn);
    if (nan) {
      mx = mx0;
      mn = mn0;
      scan_kept(scan_floats);
      scan_rest(scan_floats);
    }
  } else {
    UnitScan<T, AZP> whole;
    auto scan = [&](const Raw<T>& raw, int j) {
      int lo, hi;
      part(j, lo, hi);
      if (lo == 0 && hi == kVec) whole.add(raw, mx, mn);  // all but the row's first and last unit
      else scan_floats(raw, j);
    };
    scan_kept(scan);
    scan_rest(scan);
    whole.fold(mx, mn);
  }
  row_max_min<LANES>(mx, mn, lds);

  float scale_val, mul = 0.f;
  int azp_val = 0;
  if (AZP) {
    scale_val = (mx - mn) / 255.0f;
    azp_val = (int)rintf(-128.0f - mn / scale_val);
  } else {
    scale_val = mx / 127.0f;
    mul = 127.0f / mx;
  }
  if (lane == 0) {
    scales[token] = scale_val;
    if (AZP) azps[token] = azp_val;
  }
  const Divisor d(scale_val);
  const FastRow<AZP ? kQuotientAzp : kProduct> row(mul, d, azp_val, AZP ? fmaxf(fabsf(mx), fabsf(mn)) : mx);
  auto emit = [&](Raw<T> raw, int j) {
    int q[kVec];
    forget(raw);
    bool done = false;
    if constexpr (by_bits) {
      // no NaN among the wave's elements, and none on the way: the largest magnitude is ordinary and a quotient within 2^20
      if (row.usable && !(AZP && nan)) {
        fast8<false>(raw, row, q);
        done = true;
      }
    } else if (sizeof(T) == 2 && row.usable) {
      done = !__builtin_amdgcn_ballot_w64(!fast8<true>(raw, row, q));
    }
    if (done) {
    } else if (AZP) {
      quantise8<true>(raw, d, azp_val, q);
    } else {
      float y[kVec];
      products(raw, mul, y);
#pragma unroll
      for (int i = 0; i < kVec; ++i) q[i] = float_to_int8_rn(y[i]);
    }
    const int rel = (j - first) * kVec - head;
    store_unit<false>(row_out, j, q, max(-rel, 0), min(hidden - rel, kVec), aligned);
  };
#pragma unroll
  for (int k = 0; k < KEEP; ++k) {
    const int j = lane + k * LANES;
    if (j >= first && j < end) emit(keep[k], j);
  }
  for (int j = lane + KEEP * LANES; j < end; j += LANES) emit(fetch(j), j);
}
template <typename T, bool AZP, int LANES, int KEEP, RowMode MODE>
__global__ __launch_bounds__(row_threads(LANES)) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 2 && LANES >= 256 ? (MODE == WHOLE || MODE == EVEN || !AZP ? 8 : 7) : 1)))
void dynamic_quant_kernel(HQ_ARGS12) {
  HqReader r(HQ_PASS12);
  const T* const in = r;
  int8_t* const out = r;
  float* const scales = r;
  int32_t* const azps = r;
  const int64_t tokens = r;
  const int hidden = r;
  dynamic_quant_body<T, AZP, LANES, KEEP, MODE>(in, out, scales, azps, tokens, hidden);
}

// The 128-bit loads and 64-bit stores need both base pointers on their grid; other pointers are served
// element by element.
__host__ inline int pointers_aligned(const void* in, const void* out) {
  return !((uintptr_t)in & 15) && !((uintptr_t)out & 7);
}

template <typename T>
int launch_static(const T* in, int8_t* out, int64_t tokens, int hidden, float scale, int has_azp, int azp,
                  const HqDevice* dev, hipStream_t stream) {
  const int aligned = pointers_aligned(in, out);
  const int64_t total = tokens * hidden;
  const int64_t units = (total + kVec - 1) / kVec;
  int64_t blocks = (units + 256 * kStaticUnroll - 1) / (256 * kStaticUnroll);
  // six workgroups per CU, grid-stride beyond that (us per call at 32 / 6 per CU, fp16: 4096 x 5137 13.8 / 12.8,
  // 4096 x 4096 11.3 / 10.7, 8192 x 5120 24.3 / 23.3, 16384 x 8192 72.4 / 71.6; four and eight per CU, and grids
  // sized so that every workgroup makes the same number of trips, measured in between)
  const int64_t cap = (int64_t)dev->cus * 6;
  if (blocks > cap) blocks = cap;
  if (has_azp)
    return hq_launch(static_quant_kernel<T, true>, dim3((unsigned)blocks), dim3(256), 0, stream, in, out, scale, azp, total, aligned);
  return hq_launch(static_quant_kernel<T, false>, dim3((unsigned)blocks), dim3(256), 0, stream, in, out, scale, azp, total, aligned);
}

template <typename T, bool AZP, RowMode MODE>
int launch_dynamic_mode(const T* in, int8_t* out, float* scales, int32_t* azps, int64_t tokens, int hidden,
                         const HqDevice* dev, hipStream_t stream) {
  // Short rows get a wave each, the others a workgroup of as many threads as keep the whole row in registers with at most
  // five units each: rows past five units of 256 threads used to be read twice (2048 rows of 16384 bf16 with zero point
  // 21.4 -> 18.9 us; 3001 of 10241 fp32 69.6 -> 29.2; 1023 of 12289 fp16 22.6 -> 9.2, both of these also cut at the tensor's end).
  // With no more rows than compute units the latency of one row is all there is, and more threads shorten it (5 rows of 14883
  // bf16 9.7 -> 4.6 us).
  const bool wave_rows = hidden <= 64 * kVec * 3;
  const int span = (hidden + kVec - 1) / kVec + 1 + 63;  // units from the 64-unit boundary before a ragged row to its end
#define HQ_ROWS(LANES, KEEP)                                                                                          \
  return hq_launch(dynamic_quant_kernel<T, AZP, LANES, KEEP, MODE>, dim3((unsigned)(LANES == 64 ? (tokens + 3) / 4 : tokens)), \
                   dim3(row_threads(LANES)), 0, stream, in, out, scales, azps, tokens, hidden)
  if (wave_rows) {
    if (span <= 64 * 2) HQ_ROWS(64, 2);
    else if (span <= 64 * 3) HQ_ROWS(64, 3);
    else HQ_ROWS(64, 5);
  } else if (tokens <= dev->cus && span > 512) {
    if (span <= 1024) HQ_ROWS(512, 2);
    else if (span <= 2048) HQ_ROWS(1024, 2);
    else HQ_ROWS(1024, 5);
  } else {
    if (span <= 256 * 2) HQ_ROWS(256, 2);
    else if (span <= 256 * 3) HQ_ROWS(256, 3);
    else if (span <= 256 * 5) HQ_ROWS(256, 5);
    else if (span <= 512 * 5) HQ_ROWS(512, 5);
    else HQ_ROWS(1024, 5);
  }
#undef HQ_ROWS
}

template <typename T, bool AZP>
int launch_dynamic_azp(const T* in, int8_t* out, float* scales, int32_t* azps, int64_t tokens, int hidden,
                        const HqDevice* dev, hipStream_t stream) {
  const int64_t total = tokens * hidden;
  if (!pointers_aligned(in, out) || total < kVec)
    return launch_dynamic_mode<T, AZP, ANY>(in, out, scales, azps, tokens, hidden, dev, stream);
  if (total % kVec)
    return launch_dynamic_mode<T, AZP, TAIL>(in, out, scales, azps, tokens, hidden, dev, stream);
  if constexpr (__is_same(T, bf16_t)) {
    // with a zero point only rows that begin and end with blocks of 64 units, or never cross one
    const bool even = !AZP || hidden % (64 * kVec) == 0 || (64 * kVec) % hidden == 0;
    if (hidden % kVec == 0 && even && hidden <= 4096)
      return launch_dynamic_mode<T, AZP, EVEN>(in, out, scales, azps, tokens, hidden, dev, stream);
  }
  return launch_dynamic_mode<T, AZP, WHOLE>(in, out, scales, azps, tokens, hidden, dev, stream);
}

template <typename T>
int launch_dynamic(const T* in, int8_t* out, float* scales, int32_t* azps, int64_t tokens, int hidden,
                   const HqDevice* dev, hipStream_t stream) {
  if (azps) return launch_dynamic_azp<T, true>(in, out, scales, azps, tokens, hidden, dev, stream);
  return launch_dynamic_azp<T, false>(in, out, scales, azps, tokens, hidden, dev, stream);
}

int check_common(const void* x, int x_dtype, const int8_t* out, int64_t tokens, int hidden) {
  if (tokens < 0 || hidden <= 0) return HQ_ERR_BAD_SHAPE;
  if (x_dtype != HQ_DTYPE_F32 && x_dtype != HQ_DTYPE_F16 && x_dtype != HQ_DTYPE_BF16) return HQ_ERR_BAD_ENUM;
  if (tokens == 0) return HQ_OK;
  if (!x || !out) return HQ_ERR_NULL_POINTER;
  if (tokens > 0x7fffffff) return HQ_ERR_TOO_LARGE;
  const int esz = x_dtype == HQ_DTYPE_F32 ? 4 : 2;
  if ((uintptr_t)x & (esz - 1)) return HQ_ERR_MISALIGNED;
  return HQ_OK;
}

}  // namespace

extern "C" int hq_int8_quant_static(const void* x, int x_dtype, int8_t* out, int64_t num_tokens, int hidden_size,
                                    float scale, int has_azp, int32_t azp, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  int rc = check_common(x, x_dtype, out, num_tokens, hidden_size);
  if (rc != HQ_OK || num_tokens == 0) return rc;
  const HqDevice* dev = nullptr;
  rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  if (x_dtype == HQ_DTYPE_F32)
    return launch_static((const float*)x, out, num_tokens, hidden_size, scale, has_azp, azp, dev, stream);
  if (x_dtype == HQ_DTYPE_F16)
    return launch_static((const _Float16*)x, out, num_tokens, hidden_size, scale, has_azp, azp, dev, stream);
  return launch_static((const bf16_t*)x, out, num_tokens, hidden_size, scale, has_azp, azp, dev, stream);
}

extern "C" int hq_int8_quant_dynamic(const void* x, int x_dtype, int8_t* out, float* scales, int32_t* azp,
                                     int64_t num_tokens, int hidden_size, void* stream_) {
  hipStream_t stream = (hipStream_t)stream_;
  int rc = check_common(x, x_dtype, out, num_tokens, hidden_size);
  if (rc != HQ_OK || num_tokens == 0) return rc;
  if (!scales) return HQ_ERR_NULL_POINTER;
  if (((uintptr_t)scales & 3) || ((uintptr_t)azp & 3)) return HQ_ERR_MISALIGNED;
  const HqDevice* dev = nullptr;
  rc = hq_current_device(&dev);
  if (rc != HQ_OK) return rc;
  if (x_dtype == HQ_DTYPE_F32)
    return launch_dynamic((const float*)x, out, scales, azp, num_tokens, hidden_size, dev, stream);
  if (x_dtype == HQ_DTYPE_F16)
    return launch_dynamic((const _Float16*)x, out, scales, azp, num_tokens, hidden_size, dev, stream);
  return launch_dynamic((const bf16_t*)x, out, scales, azp, num_tokens, hidden_size, dev, stream);
}
