// Weight preparation on the device: the reference's pure-torch quantizers
// (x/fp4x_kernels.py: quantize_w8 :138-144, quantize_w6 :179-202 with or
// without the clip search, quantize_nv4 :277-300, quantize_int2 :330-351 with fp16 scales,
// or e4m3 scales under an fp32 row scale) as one thread per 16 weights: the
// 1, 2 or 4 lanes of a quantization group share its maximum.  (One thread per
// group for the clip search, one wave per row for the e4m3 INT2 target.)
//
// The source rows are fp32, bf16, or packed MXFP8 / NVFP4 rows decoded in
// registers with the exact dequant of mx8_dequant (:261-267) or dequant_nv4
// (:420-426), so a packed head is requantized without its fp32 copy.
//
// Arithmetic follows the reference's formulas with IEEE fp32 division, the
// semantics of its torch ops on CPU tensors (where its golden vectors were
// taken): torch's GPU division by a Python scalar multiplies by the
// reciprocal instead, which can move a result by one fp32 ulp.  A division per
// weight is about 11 instructions, and was what these kernels spent their time
// on; exact_quot gives the same quotient in 3 from the scale's reciprocal, and
// the INT2 codes need comparisons only.  Groups with infinities, NaN or scales
// at the ends of their range still divide.  us, before -> after, kernels alone
// (MXFP8 rows, traced): the 248,320 x 2560 head's INT2 copy 416 -> 160 (893
// MB); [16384 x 2560] to W8 35 -> 18, to W6 35 -> 20, to NVFP4 44 -> 20, its
// global maximum 100 -> 14 (one atomic per workgroup that raises it, instead
// of one per wave, all on one word).
#include <cmath>

#include "fp4x_kernels.h"
#include "../../include/fp4x.h"

namespace fp4x {

int device_cus();

// ------------------------------------------------------------------ sources
// load<G>(row, k0, f): the G fp32 weights [k0, k0 + G) of a row (k0 % 16 == 0).
// load16(t, f): weights [16 t, 16 t + 16) of the whole matrix (every plane is
// one run of memory, K being a multiple of 64).
struct SrcF32 {
  const float* w;
  int64_t ld;
  __device__ void load16(int64_t t, float (&f)[16]) const { SrcF32{w + 16 * t, 0}.load<16>(0, 0, f); }
  template <int G>
  __device__ void load(int64_t row, int k0, float (&f)[G]) const {
    const float4* p = reinterpret_cast<const float4*>(w + row * ld + k0);
#pragma unroll
    for (int i = 0; i < G / 4; ++i) {
      const float4 v = p[i];
      f[4 * i] = v.x; f[4 * i + 1] = v.y; f[4 * i + 2] = v.z; f[4 * i + 3] = v.w;
    }
  }
};

struct SrcBF16 {
  const uint16_t* w;
  int64_t ld;
  __device__ void load16(int64_t t, float (&f)[16]) const { SrcBF16{w + 16 * t, 0}.load<16>(0, 0, f); }
  template <int G>
  __device__ void load(int64_t row, int k0, float (&f)[G]) const {
    const uint4* p = reinterpret_cast<const uint4*>(w + row * ld + k0);
#pragma unroll
    for (int i = 0; i < G / 8; ++i) {
      const uint4 v = p[i];
      const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f[8 * i + 2 * j] = bf16_lo(d[j]);
        f[8 * i + 2 * j + 1] = bf16_hi(d[j]);
      }
    }
  }
};

// MXFP8: e4m3fn [N, K] and e8m0 [N, K/32]; e4m3 * 2^(s - 127) is exact.
struct SrcMX8 {
  const uint8_t* w;
  const uint8_t* s;
  int K;
  __device__ void load16(int64_t t, float (&f)[16]) const { SrcMX8{w + 16 * t, s + (t >> 1), 32}.load<16>(0, 0, f); }
  template <int G>
  __device__ void load(int64_t row, int k0, float (&f)[G]) const {
#pragma unroll
    for (int c = 0; c < G / 16; ++c) {
      const int k = k0 + 16 * c;
      const uint4 q = *reinterpret_cast<const uint4*>(w + row * K + k);
      const uint32_t e = s[row * (K / 32) + k / 32];
      const float sc = e8m0_to_f32(e);
      const uint32_t d[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x2_t a = fp8x2_to_f32x2<false>(d[i], sc), b = fp8x2_to_f32x2<true>(d[i], sc);
        f[16 * c + 4 * i] = a.x; f[16 * c + 4 * i + 1] = a.y;
        f[16 * c + 4 * i + 2] = b.x; f[16 * c + 4 * i + 3] = b.y;
      }
      if (e == 255u) {                                    // exp2(128) = +inf, as mx8_dequant (FmtMX8)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          f[16 * c + j] = __uint_as_float(FmtMX8::inf_bf16((d[j / 4] >> (8 * (j % 4))) & 0xffu) << 16);
      }
    }
  }
};

// NVFP4: e2m1 pairs [N, K/2] (low nibble = even k), e4m3 [N, K/16], gs:
// (e2m1 * e4m3) * gs in fp32, the product exact and one rounding by gs.
struct SrcNV4 {
  const uint8_t* P;
  const uint8_t* S;
  float gs;
  int K;
  __device__ void load16(int64_t t, float (&f)[16]) const { SrcNV4{P + 8 * t, S + t, gs, 16}.load<16>(0, 0, f); }
  template <int G>
  __device__ void load(int64_t row, int k0, float (&f)[G]) const {
#pragma unroll
    for (int c = 0; c < G / 16; ++c) {
      const int k = k0 + 16 * c;
      const uint2 q = *reinterpret_cast<const uint2*>(P + row * (K / 2) + k / 2);
      const float sc = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8((uint32_t)S[row * (K / 16) + k / 16], 1.0f,
                                                                false)[0];
      const uint32_t d[2] = {q.x, q.y};
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x2_t v0 = fp4x2_to_f32x2<0>(d[h]), v1 = fp4x2_to_f32x2<1>(d[h]);
        const f32x2_t v2 = fp4x2_to_f32x2<2>(d[h]), v3 = fp4x2_to_f32x2<3>(d[h]);
        const float v[8] = {v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
#pragma unroll
        for (int j = 0; j < 8; ++j) f[16 * c + 8 * h + j] = (v[j] * sc) * gs;
      }
    }
  }
};

__device__ __forceinline__ float f16_round(float v) { return (float)(_Float16)v; }

// Non-negative fp32 v < 464 -> e4m3fn code, round to nearest even (below
// 2^-6 the subnormal step 2^-9; below 2^-10, and at it, code 0).
__device__ __forceinline__ uint32_t e4m3_code(float v) {
  int e = (int)((__float_as_uint(v) >> 23) & 0xff) - 127;
  if (e < -6) e = -6;                                  // subnormal step 2^-9
  float q = rintf(v * __uint_as_float((uint32_t)(127 + 3 - e) << 23));   // v * 2^(3 - e)
  if (q >= 16.0f) { q = 8.0f; ++e; }
  const uint32_t m = (uint32_t)q;
  return m < 8 ? m : ((uint32_t)(e + 7) << 3) | (m - 8);
}
__device__ __forceinline__ float e4m3_value(uint32_t code) {
  const uint32_t e = code >> 3, m = code & 7;
  return e ? (float)(8 + m) * __uint_as_float((uint32_t)(127 + (int)e - 10) << 23) : (float)m * 0x1p-9f;
}

template <int G>
__device__ __forceinline__ float group_amax(const float (&f)[G]) {
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < G; ++i) a = fmaxf(a, fabsf(f[i]));
  return a;
}

// Maximum of |f| over the 16 LPG weights of a group's LPG lanes (1, 2 or 4
// neighbours); a NaN weight makes it NaN (v_maximum3_f32).
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_mov_dpp((int)__float_as_uint(v), CTRL, 0xf, 0xf, true));
}
template <int LPG>
__device__ __forceinline__ float lanes_maximum(const float (&f)[16]) {
  float a = fabsf(f[0]);
#pragma unroll
  for (int i = 1; i < 16; ++i) a = __builtin_elementwise_maximum(a, fabsf(f[i]));
  if constexpr (LPG >= 2) a = __builtin_elementwise_maximum(a, dpp_f32<0xB1>(a));   // lane ^ 1
  if constexpr (LPG >= 4) a = __builtin_elementwise_maximum(a, dpp_f32<0x4E>(a));   // lane ^ 2
  return a;
}
// The reference's maximum, which skips NaN weights.
template <int LPG>
__device__ __forceinline__ float lanes_amax(const float (&f)[16]) {
  float a = group_amax(f);
  if constexpr (LPG >= 2) a = fmaxf(a, dpp_f32<0xB1>(a));
  if constexpr (LPG >= 4) a = fmaxf(a, dpp_f32<0x4E>(a));
  return a;
}
__device__ __forceinline__ bool finite_max(float m) { return m < __builtin_inff(); }   // false for NaN

// Targets: put(t, f) quantizes weights [16 t, 16 t + 16) of the matrix; lanes
// t of one group run together.
constexpr float kRint = 12582912.0f;               // 1.5 * 2^23: v + kRint holds rint(v) in its low bits

// RN(f / s) from rs = RN(1 / s) (Markstein: a quotient within an ulp, its exact
// remainder by fma, and one correction with the rounded reciprocal give the
// rounded quotient), for 2^-100 <= s < 2^100 and finite f; a quotient so small
// that the remainder underflows is still within an ulp, which no code notices.
// -0 gives +0.
__device__ __forceinline__ float exact_quot(float f, float s, float rs) {
  const float q = f * rs;
  return __builtin_fmaf(__builtin_fmaf(-q, s, f), rs, q);
}
__device__ __forceinline__ bool mid_range(float s) { return s >= 0x1p-100f && s < 0x1p100f; }

// ------------------------------------------------------------------ targets
// W8 g64: s = max(amax, 1e-12) / 127, q = clamp(rint(w / s), -127, 127).
// The clamp never acts on a finite group: its maximum gives 127.
struct QW8 {
  static constexpr int G = 64, LPG = 4;
  int8_t* q;
  float* s;
  __device__ void put(int64_t t, const float (&f)[16]) const {
    float m = lanes_maximum<LPG>(f);
    const bool fin = finite_max(m);
    if (!fin) m = lanes_amax<LPG>(f);
    const float sc = fmaxf(m, 1e-12f) / 127.0f;
    uint32_t b[16];
    if (fin && mid_range(sc)) {
      const float rc = 1.0f / sc;
#pragma unroll
      for (int i = 0; i < 16; ++i) b[i] = __float_as_uint(exact_quot(f[i], sc, rc) + kRint);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) b[i] = (uint32_t)(int)fminf(fmaxf(rintf(f[i] / sc), -127.0f), 127.0f);
    }
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = perm_b32(perm_b32(b[4 * i + 3], b[4 * i + 2], 0x0c0c0400u), perm_b32(b[4 * i + 1], b[4 * i], 0x0c0c0400u),
                      0x05040100u);
    reinterpret_cast<uint4*>(q)[t] = make_uint4(w[0], w[1], w[2], w[3]);
    if ((t & 3) == 0) s[t >> 2] = sc;
  }
};

// W6 g32: s = max(fp16(amax / qmax), 6.2e-5), c = clamp(rint(w / s), -qmax-1,
// qmax) + 32, split into the nibble plane L and the bit-pair plane H.
struct W6Planes {
  uint8_t* L;
  uint8_t* H;
  uint16_t* S;
  int qmax;
};
// By 16 weights.  fp16's rounding of the scale moves the quotient of a finite
// group's maximum by at most 2^-11 of it (a scale raised to 6.2e-5 makes
// quotients smaller), so the clamp never acts.
struct QW6 : W6Planes {
  static constexpr int G = 32, LPG = 2;
  __device__ void put(int64_t t, const float (&f)[16]) const {
    float m = lanes_maximum<LPG>(f);
    const bool fin = finite_max(m);
    if (!fin) m = lanes_amax<LPG>(f);
    const float sc = fmaxf(f16_round(m / (float)qmax), 6.2e-5f);
    uint32_t c[16];
    if (fin && finite_max(sc)) {                   // (fp16 can overflow)
      const float rc = 1.0f / sc;
#pragma unroll
      for (int i = 0; i < 16; ++i) c[i] = __float_as_uint(exact_quot(f[i], sc, rc) + (kRint + 32.0f));
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        c[i] = (uint32_t)((int)fminf(fmaxf(rintf(f[i] / sc), (float)(-qmax - 1)), (float)qmax) + 32);
    }
    uint32_t l[2] = {0, 0}, h = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {                  // four codes a byte each, then their nibbles and bit pairs
      const uint32_t b = perm_b32(perm_b32(c[4 * i + 3], c[4 * i + 2], 0x0c0c0400u),
                                  perm_b32(c[4 * i + 1], c[4 * i], 0x0c0c0400u), 0x05040100u);
      const uint32_t n = b & 0x0f0f0f0fu, n2 = n | (n >> 4), p = (b >> 4) & 0x03030303u;
      l[i >> 1] |= ((n2 & 0xffu) | ((n2 >> 8) & 0xff00u)) << (16 * (i & 1));
      h |= ((p | (p >> 14) | (p >> 4) | (p >> 18)) & 0xffu) << (8 * i);
    }
    reinterpret_cast<uint2*>(L)[t] = make_uint2(l[0], l[1]);
    reinterpret_cast<uint32_t*>(H)[t] = h;
    if ((t & 1) == 0) S[t >> 1] = __builtin_bit_cast(uint16_t, (_Float16)sc);
  }
};
// By groups.
struct QW6Group : W6Planes {
  static constexpr int G = 32;
  __device__ static float base_scale(const float (&f)[G], int qmax) {
    return fmaxf(f16_round(group_amax(f) / (float)qmax), 6.2e-5f);
  }
  // codes clamp(rint(w / sc), -qmax - 1, qmax) + 32 into the two planes, fp16(sc) into S
  __device__ void put_scaled(int64_t row, int gi, int K, const float (&f)[G], float sc) const {
    uint32_t c[G];
#pragma unroll
    for (int i = 0; i < G; ++i)
      c[i] = (uint32_t)((int)fminf(fmaxf(rintf(f[i] / sc), (float)(-qmax - 1)), (float)qmax) + 32);
    uint32_t l[4] = {0, 0, 0, 0}, h[2] = {0, 0};
#pragma unroll
    for (int j = 0; j < 16; ++j) l[j >> 2] |= ((c[2 * j] & 15) | ((c[2 * j + 1] & 15) << 4)) << (8 * (j & 3));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t b = (c[4 * j] >> 4) | ((c[4 * j + 2] >> 4) << 2) | ((c[4 * j + 1] >> 4) << 4) |
                         ((c[4 * j + 3] >> 4) << 6);
      h[j >> 2] |= b << (8 * (j & 3));
    }
    *reinterpret_cast<uint4*>(L + row * (K / 2) + gi * 16) = make_uint4(l[0], l[1], l[2], l[3]);
    *reinterpret_cast<uint2*>(H + row * (K / 4) + gi * 8) = make_uint2(h[0], h[1]);
    S[row * (K / G) + gi] = __builtin_bit_cast(uint16_t, (_Float16)sc);
  }
};

// W6 with the clip search: the group's scale is the first of s, sc_1 .. sc_n
// (sc_i = max(fp16(s * c_i), 6.2e-5), c_i the fp32 factors of the clip grid)
// whose squared error sum((clamp(rint(w / sc), -qmax - 1, qmax) * sc - w)^2)
// is strictly the smallest.  Every operation is rounded to fp32 on its own
// (no fused multiply-add); the 32 squares are summed as 8 lanes of 4
// (lane j: elements j, j + 8, j + 16, j + 24 in turn), then lanes 0..7 in
// turn: the order of torch's CPU sum over a 32-element row.
constexpr int kW6MaxClip = 64;
struct W6Clip {
  int n;
  float c[kW6MaxClip];
};
__device__ __forceinline__ float w6_sq_err(const float (&f)[32], float sc, int qmax) {
#pragma clang fp contract(off)
  float lane[8];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const float d = fminf(fmaxf(rintf(f[i] / sc), (float)(-qmax - 1)), (float)qmax) * sc - f[i];
    const float d2 = d * d;
    if (i < 8) lane[i] = d2;
    else lane[i & 7] = lane[i & 7] + d2;
  }
  float e = lane[0];
#pragma unroll
  for (int j = 1; j < 8; ++j) e = e + lane[j];
  return e;
}
struct QW6Clip : QW6Group {
  W6Clip clip;
  __device__ void put(int64_t row, int gi, int K, const float (&f)[G]) const {
#pragma clang fp contract(off)
    const float s = base_scale(f, qmax);
    float best = w6_sq_err(f, s, qmax), bs = s;
    for (int i = 0; i < clip.n; ++i) {
      // the fp32 product is rounded before its fp16 rounding: without the
      // register barrier the compiler fuses both into one v_fma_mixlo_f16,
      // a single rounding that differs at fp16 midpoints of the fp32 product
      float p = s * clip.c[i];
      asm volatile("" : "+v"(p));
      const float sc = fmaxf(f16_round(p), 6.2e-5f);
      const float e = w6_sq_err(f, sc, qmax);
      if (e < best) {
        best = e;
        bs = sc;
      }
    }
    put_scaled(row, gi, K, f, bs);
  }
};

// NVFP4 g16: sc = e4m3(clamp(amax / 6 / gs, 2^-9, 448)), v = clamp(w / (sc * gs),
// -6, 6), magnitude = the number of e2m1 midpoints below |v| (ties go down),
// sign bit 3 for v < 0.  The e2m1 conversion rounds ties to even, which goes up
// at 0.75, 1.75 and 3.5 alone of the midpoints, those whose leading fraction bit
// is set: one fp32 step less for such quotients sends them down and moves no
// other quotient across a midpoint.  Taken for sf in [2^-100, 1), where no
// nonzero quotient underflows to a zero (whose sign would be lost), and amax <=
// 6.9 sf, where the conversion rounds to 6 by itself.
__device__ __forceinline__ float nv4_global_scale(float amax) {
  return (float)fmax((double)amax / 6.0 / 448.0, 1e-30);   // as the host computes it
}
struct QNV4 {
  static constexpr int G = 16, LPG = 1;
  uint8_t* P;
  uint8_t* S;
  float gs;
  __device__ void put(int64_t t, const float (&f)[16]) const { put_gs(t, f, gs); }
  __device__ void put_gs(int64_t t, const float (&f)[16], float gsv) const {
    float m = lanes_maximum<1>(f);
    const bool fin = finite_max(m);
    if (!fin) m = group_amax(f);
    const float sc = fminf(fmaxf(m / 6.0f / gsv, 0x1p-9f), 448.0f);
    const uint32_t code = e4m3_code(sc);
    const float sf = e4m3_value(code) * gsv;
    uint32_t p[2] = {0, 0};
    if (fin && sf >= 0x1p-100f && sf < 1.0f && m <= 6.9f * sf) {
      const float rs = 1.0f / sf;
      float v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t b = __float_as_uint(exact_quot(f[i], sf, rs));
        v[i] = __uint_as_float(b - ((b >> 22) & 1u));
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        p[h] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(p[h], v[8 * h], v[8 * h + 1], 1.0f, 0);
        p[h] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(p[h], v[8 * h + 2], v[8 * h + 3], 1.0f, 1);
        p[h] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(p[h], v[8 * h + 4], v[8 * h + 5], 1.0f, 2);
        p[h] = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(p[h], v[8 * h + 6], v[8 * h + 7], 1.0f, 3);
      }
    } else {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const float v = fminf(fmaxf(f[i] / sf, -6.0f), 6.0f), a = fabsf(v);
        const uint32_t mag = (a > 0.25f) + (a > 0.75f) + (a > 1.25f) + (a > 1.75f) + (a > 2.5f) + (a > 3.5f) +
                             (a > 5.0f);
        p[i >> 3] |= (mag | (v < 0.0f ? 8u : 0u)) << (4 * (i & 7));
      }
    }
    reinterpret_cast<uint2*>(P)[t] = make_uint2(p[0], p[1]);
    S[t] = (uint8_t)code;
  }
};

// The G 2-bit codes clamp(floor(w / sf) + 2, 0, 3) of one INT2 group (0 where
// w / sf is NaN: a zero element of a group whose scale underflows), element j
// of a 4-group in bit pair (0, 2, 1, 3)[j], stored at o (G / 4 bytes).
template <int G>
__device__ __forceinline__ void put_int2_codes(const float (&f)[G], float sf, uint8_t* o) {
  uint32_t b[G / 16];
#pragma unroll
  for (int i = 0; i < G / 16; ++i) b[i] = 0;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    const uint32_t c = (uint32_t)fminf(fmaxf(floorf(f[i] / sf) + 2.0f, 0.0f), 3.0f);
    const int pair = (i & 3) == 1 ? 2 : (i & 3) == 2 ? 1 : (i & 3);
    b[i >> 4] |= c << (2 * pair + 8 * ((i >> 2) & 3));
  }
  uint32_t* o32 = reinterpret_cast<uint32_t*>(o);
#pragma unroll
  for (int i = 0; i < G / 16; ++i) o32[i] = b[i];
}

// The 16 codes of one word without a division, for finite weights and a normal
// scale 0 < sf < 2: the rounded quotient reaches 1 exactly where w >= sf and
// stays above -1 exactly where w >= -sf (the quotients of sf's two fp32
// neighbours round to 1 - 2^-24 or less and to 1 + 2^-23), and it keeps the
// sign of w (nothing underflows to zero).  So 3 - code has the bits (w < 0, w -
// copysign(sf, w) < 0), shifted in from the last element's to the first's.
__device__ __forceinline__ uint32_t int2_word(const float (&f)[16], float sf) {
  uint32_t acc = 0;
#pragma unroll
  for (int b = 3; b >= 0; --b)
#pragma unroll
    for (int j = 3; j >= 0; --j) {                 // bit pairs 3..0 hold elements 3, 1, 2, 0
      const int i = 4 * b + (j == 1 ? 2 : j == 2 ? 1 : j);
      const float w = f[i] + 0.0f;                 // -0 as +0
      acc = __builtin_amdgcn_alignbit(acc, __float_as_uint(w), 31);
      acc = __builtin_amdgcn_alignbit(acc, __float_as_uint(w - __builtin_copysignf(sf, w)), 31);
    }
  return ~acc;
}

// INT2 with fp16 group scales: s = fp16(max(amax, 1e-8) / 1.5) (a zero group's
// scale underflows fp16 to 0, and its codes are 0).
template <int GG>
struct QInt2 {
  static constexpr int G = GG, LPG = GG / 16;
  uint8_t* P;
  uint16_t* S;
  __device__ void put(int64_t t, const float (&f)[16]) const {
    float m = lanes_maximum<LPG>(f);
    const bool fin = finite_max(m);
    if (!fin) m = lanes_amax<LPG>(f);
    const _Float16 s16 = (_Float16)(fmaxf(m, 1e-8f) / 1.5f);
    const float sf = (float)s16;
    if (fin && sf > 0.0f && sf < 2.0f) reinterpret_cast<uint32_t*>(P)[t] = int2_word(f, sf);
    else put_int2_codes<16>(f, sf, P + 4 * t);
    if (t % LPG == 0) S[t / LPG] = __builtin_bit_cast(uint16_t, s16);
  }
};

// INT2 with e4m3fn group scales under an fp32 row scale rs (R[row], written by
// int2e_kernel): S = e4m3(s / rs) for s = max(amax, 1e-8) / 1.5,
// codes against sf = float(S) * rs.  A group whose s / rs rounds to e4m3 0
// (amax below about 2^-10 / 448 of the row's largest) has sf = 0: its codes
// are 3, 0 and 0 for positive, negative and zero elements.
template <int GG>
struct QInt2E {
  static constexpr int G = GG;
  uint8_t* P;
  uint8_t* S;
  float* R;
  __device__ void put(int64_t row, int gi, int K, const float (&f)[G]) const { put_rs(row, gi, K, f, R[row]); }
  __device__ void put_rs(int64_t row, int gi, int K, const float (&f)[G], float rs) const {
    const uint32_t code = e4m3_code((fmaxf(group_amax(f), 1e-8f) / 1.5f) / rs);
    put_int2_codes(f, e4m3_value(code) * rs, P + row * (K / 4) + gi * (G / 4));
    S[row * (K / G) + gi] = (uint8_t)code;
  }
};

// One thread per group (the clip search).
template <class Src, class Q>
__global__ __launch_bounds__(256) void quant_group_kernel(Src src, Q q, int64_t N, int K) {
  const int gpr = K / Q::G;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= N * gpr) return;
  const int64_t row = t / gpr;
  const int gi = (int)(t - row * gpr);
  float f[Q::G];
  src.template load<Q::G>(row, gi * Q::G, f);
  q.put(row, gi, K, f);
}

// One thread per 16 weights; n16 (a multiple of 4, so of every LPG) of them.
template <class Src, class Q>
__global__ __launch_bounds__(256) void quant_kernel(Src src, Q q, int64_t n16) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= n16) return;
  float f[16];
  src.load16(t, f);
  q.put(t, f);
}

// The NVFP4 target with the global scale of *amax, worked out once per workgroup.
template <class Src>
__global__ __launch_bounds__(256) void quant_nv4_amax_kernel(Src src, QNV4 q, int64_t n16, const float* amax) {
  __shared__ float gs;
  if (threadIdx.x == 0) gs = nv4_global_scale(*amax);
  __syncthreads();
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n16; t += (int64_t)gridDim.x * 256) {
    float f[16];
    src.load16(t, f);
    q.put_gs(t, f, gs);
  }
}

// max |w| over the whole matrix into *out (zeroed by the caller): per-thread
// maxima over pieces of 16 weights, the workgroup's maximum, and an atomic max
// of its fp32 bits (ordered as unsigned for non-negative values) where it is
// above what *out already holds: atomics on one word queue, about 10 ns each.
template <class Src>
__global__ __launch_bounds__(512) void absmax_kernel(Src src, int64_t n16, uint32_t* out) {
  __shared__ float part[8];
  const int64_t step = (int64_t)gridDim.x * 512;
  float m = 0.0f;
  int64_t t = (int64_t)blockIdx.x * 512 + threadIdx.x;
  for (; t + 3 * step < n16; t += 4 * step) {          // four pieces in flight
    float f[4][16];
#pragma unroll
    for (int u = 0; u < 4; ++u) src.load16(t + u * step, f[u]);
#pragma unroll
    for (int u = 0; u < 4; ++u) m = fmaxf(m, group_amax(f[u]));
  }
  for (; t < n16; t += step) {
    float f[16];
    src.load16(t, f);
    m = fmaxf(m, group_amax(f));
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 8; ++w) m = fmaxf(m, part[w]);
    if (__float_as_uint(m) > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(out, __float_as_uint(m));
  }
}

template <class Src>
static void launch_absmax(const Src& src, int64_t N, int K, float* out, hipStream_t st) {
  const int64_t n16 = N * (K / 16);
  const unsigned grid = (unsigned)std::min<int64_t>((n16 + 511) / 512, (int64_t)device_cus() * 2);
  hipLaunchKernelGGL(absmax_kernel<Src>, dim3(grid), dim3(512), 0, st, src, n16, reinterpret_cast<uint32_t*>(out));
}

// The e4m3 INT2 target, one wave per row: the row scale R[row] =
// (max(row amax, 1e-8) / 1.5) / 448, the largest group scale of the row over
// 448 (the rounded quotient max(a, 1e-8) / 1.5 is monotonic in a, so the row
// maximum of the group scales is the scale of the row's amax), then the
// row's groups against it.  The second read of the row comes from the caches
// the first one filled.
template <class Src, int G>
__global__ __launch_bounds__(256) void int2e_kernel(Src src, QInt2E<G> q, int64_t N, int K) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;                                  // uniform over the wave
  const int lane = threadIdx.x & 63;
  float m = 0.0f;
  for (int g = lane; g < K / 16; g += 64) {
    float f[16];
    src.template load<16>(row, g * 16, f);
    m = fmaxf(m, group_amax(f));
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  const float rs = (fmaxf(m, 1e-8f) / 1.5f) / 448.0f;
  if (lane == 0) q.R[row] = rs;
  for (int gi = lane; gi < K / G; gi += 64) {
    float f[G];
    src.template load<G>(row, gi * G, f);
    q.put_rs(row, gi, K, f, rs);
  }
}

static bool al(const void* p, int a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

template <class Src, class Q>
static int launch_q(const Src& src, const Q& q, int64_t N, int K, hipStream_t st) {
  const int64_t n16 = N * (K / 16);
  if (n16 == 0) return FP4X_OK;
  hipLaunchKernelGGL((quant_kernel<Src, Q>), dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, st, src, q, n16);
  return check_launch("quantize");
}
template <class Src, class Q>
static int launch_q_groups(const Src& src, const Q& q, int64_t N, int K, hipStream_t st) {
  const int64_t groups = N * (K / Q::G);
  if (groups == 0) return FP4X_OK;
  hipLaunchKernelGGL((quant_group_kernel<Src, Q>), dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, src, q, N,
                     K);
  return check_launch("quantize");
}
template <class Src>
static int launch_nv4_amax(const Src& src, int64_t N, int K, float* amax, uint8_t* P, uint8_t* S, hipStream_t st) {
  const int64_t n16 = N * (K / 16);
  if (n16 == 0) return FP4X_OK;
  launch_absmax(src, N, K, amax, st);
  const unsigned grid = (unsigned)std::min<int64_t>((n16 + 255) / 256, (int64_t)device_cus() * 16);
  hipLaunchKernelGGL(quant_nv4_amax_kernel<Src>, dim3(grid), dim3(256), 0, st, src, QNV4{P, S, 0.0f}, n16, amax);
  return check_launch("quantize_nv4");
}

template <class Src>
static int dispatch_q(const Src& src, int64_t N, int K, int dst, int G, int qmax, float gs, void* o0, void* o1,
                      void* o2, hipStream_t st) {
  switch (dst) {
    case FP4X_Q_W8:
      return launch_q(src, QW8{static_cast<int8_t*>(o0), static_cast<float*>(o1)}, N, K, st);
    case FP4X_Q_W6:
      return launch_q(
          src, QW6{{static_cast<uint8_t*>(o0), static_cast<uint8_t*>(o1), static_cast<uint16_t*>(o2), qmax}}, N, K, st);
    case FP4X_Q_NV4:
      return launch_q(src, QNV4{static_cast<uint8_t*>(o0), static_cast<uint8_t*>(o1), gs}, N, K, st);
    case FP4X_Q_INT2_E4M3: {
      uint8_t* P = static_cast<uint8_t*>(o0);
      uint8_t* S = static_cast<uint8_t*>(o1);
      float* R = static_cast<float*>(o2);
      if (N == 0) return FP4X_OK;
      const dim3 grid((unsigned)((N + 3) / 4));
      if (G == 16) hipLaunchKernelGGL((int2e_kernel<Src, 16>), grid, dim3(256), 0, st, src, QInt2E<16>{P, S, R}, N, K);
      else if (G == 32) hipLaunchKernelGGL((int2e_kernel<Src, 32>), grid, dim3(256), 0, st, src, QInt2E<32>{P, S, R}, N, K);
      else hipLaunchKernelGGL((int2e_kernel<Src, 64>), grid, dim3(256), 0, st, src, QInt2E<64>{P, S, R}, N, K);
      return check_launch("quantize (INT2 e4m3)");
    }
    default:
      if (G == 16) return launch_q(src, QInt2<16>{static_cast<uint8_t*>(o0), static_cast<uint16_t*>(o1)}, N, K, st);
      if (G == 32) return launch_q(src, QInt2<32>{static_cast<uint8_t*>(o0), static_cast<uint16_t*>(o1)}, N, K, st);
      return launch_q(src, QInt2<64>{static_cast<uint8_t*>(o0), static_cast<uint16_t*>(o1)}, N, K, st);
  }
}

static int src_check(int src, const void* a, const void* b, int64_t N, int K) {
  if (N < 0 || K <= 0 || K % 64) { set_error("quantize: need N >= 0 and K % 64 == 0"); return FP4X_ERR_ARG; }
  if (src < FP4X_SRC_F32 || src > FP4X_SRC_NV4) { set_error("quantize: unknown source kind"); return FP4X_ERR_ARG; }
  if (!al(a, 16) || ((src == FP4X_SRC_MX8 || src == FP4X_SRC_NV4) && !b)) {
    set_error("quantize: source rows must be 16-byte aligned (and packed sources need their scales)");
    return FP4X_ERR_ARG;
  }
  return FP4X_OK;
}

}  // namespace fp4x

using namespace fp4x;

extern "C" {

int fp4x_quantize(int src, const void* src_a, const void* src_b, float src_gs, int64_t N, int K, int dst, int G,
                  int qmax, float dst_gs, void* out0, void* out1, void* out2, void* stream) {
  int rc = src_check(src, src_a, src_b, N, K);
  if (rc) return rc;
  const bool int2 = dst == FP4X_Q_INT2 || dst == FP4X_Q_INT2_E4M3;
  if (dst < FP4X_Q_W8 || dst > FP4X_Q_INT2_E4M3 || (int2 && G != 16 && G != 32 && G != 64) ||
      (dst == FP4X_Q_W6 && (qmax < 1 || qmax > 31)) || (dst == FP4X_Q_NV4 && !(dst_gs > 0.0f))) {
    set_error("quantize: bad target (INT2 group 16, 32 or 64; W6 qmax 1..31; NVFP4 gs > 0)");
    return FP4X_ERR_ARG;
  }
  if (!al(out0, 16) || !out1 || ((dst == FP4X_Q_W6 || dst == FP4X_Q_INT2_E4M3) && !out2) ||
      (dst == FP4X_Q_INT2_E4M3 && !al(out2, 4))) {
    set_error("quantize: the packed output must be 16-byte aligned, and every output plane given");
    return FP4X_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  switch (src) {
    case FP4X_SRC_F32:
      return dispatch_q(SrcF32{static_cast<const float*>(src_a), K}, N, K, dst, G, qmax, dst_gs, out0, out1, out2, st);
    case FP4X_SRC_BF16:
      return dispatch_q(SrcBF16{static_cast<const uint16_t*>(src_a), K}, N, K, dst, G, qmax, dst_gs, out0, out1, out2,
                        st);
    case FP4X_SRC_MX8:
      return dispatch_q(SrcMX8{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), K}, N, K, dst,
                        G, qmax, dst_gs, out0, out1, out2, st);
    default:
      return dispatch_q(SrcNV4{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), src_gs, K}, N,
                        K, dst, G, qmax, dst_gs, out0, out1, out2, st);
  }
}

int fp4x_quantize_w6_clip(int src, const void* src_a, const void* src_b, float src_gs, int64_t N, int K, int qmax,
                          int clip_search, void* L, void* H, void* S, void* stream) {
  int rc = src_check(src, src_a, src_b, N, K);
  if (rc) return rc;
  if (qmax < 1 || qmax > 31 || clip_search < 0 || clip_search > kW6MaxClip) {
    set_error("quantize_w6_clip: need qmax 1..31 and clip_search 0..64");
    return FP4X_ERR_ARG;
  }
  if (!al(L, 16) || !al(H, 8) || !S) {
    set_error("quantize_w6_clip: L must be 16-byte and H 8-byte aligned, and S given");
    return FP4X_ERR_ARG;
  }
  // the clip grid as torch.linspace(0.70, 0.98, n) in fp32: step = (0.98f - 0.70f) / (n - 1),
  // c_i = fma(step, i, 0.70f) below n / 2, else fma(-step, n - 1 - i, 0.98f)
  QW6Clip q;
  q.L = static_cast<uint8_t*>(L);
  q.H = static_cast<uint8_t*>(H);
  q.S = static_cast<uint16_t*>(S);
  q.qmax = qmax;
  q.clip.n = clip_search;
  const float c0 = 0.70f, c1 = 0.98f;
  const float step = clip_search > 1 ? (c1 - c0) / (float)(clip_search - 1) : 0.0f;
  for (int i = 0; i < clip_search; ++i)
    q.clip.c[i] = i < clip_search / 2 || clip_search == 1 ? std::fma(step, (float)i, c0)
                                                          : std::fma(-step, (float)(clip_search - 1 - i), c1);
  for (int i = clip_search; i < kW6MaxClip; ++i) q.clip.c[i] = 0.0f;
  hipStream_t st = (hipStream_t)stream;
  switch (src) {
    case FP4X_SRC_F32:
      return launch_q_groups(SrcF32{static_cast<const float*>(src_a), K}, q, N, K, st);
    case FP4X_SRC_BF16:
      return launch_q_groups(SrcBF16{static_cast<const uint16_t*>(src_a), K}, q, N, K, st);
    case FP4X_SRC_MX8:
      return launch_q_groups(SrcMX8{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), K}, q, N, K, st);
    default:
      return launch_q_groups(SrcNV4{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), src_gs, K}, q, N,
                      K, st);
  }
}

int fp4x_absmax(int src, const void* src_a, const void* src_b, float src_gs, int64_t N, int K, float* out,
                void* stream) {
  int rc = src_check(src, src_a, src_b, N, K);
  if (rc) return rc;
  if (!out) { set_error("absmax: no output"); return FP4X_ERR_ARG; }
  if (N == 0) return FP4X_OK;
  hipStream_t st = (hipStream_t)stream;
  switch (src) {
    case FP4X_SRC_F32: launch_absmax(SrcF32{static_cast<const float*>(src_a), K}, N, K, out, st); break;
    case FP4X_SRC_BF16: launch_absmax(SrcBF16{static_cast<const uint16_t*>(src_a), K}, N, K, out, st); break;
    case FP4X_SRC_MX8:
      launch_absmax(SrcMX8{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), K}, N, K, out, st);
      break;
    default:
      launch_absmax(SrcNV4{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), src_gs, K}, N, K,
                    out, st);
  }
  return check_launch("absmax");
}

int fp4x_quantize_nv4(int src, const void* src_a, const void* src_b, float src_gs, int64_t N, int K, float* amax,
                      void* P, void* S, void* stream) {
  int rc = src_check(src, src_a, src_b, N, K);
  if (rc) return rc;
  if (!al(P, 16) || !S || !amax) {
    set_error("quantize_nv4: P must be 16-byte aligned, and S and amax given");
    return FP4X_ERR_ARG;
  }
  hipStream_t st = (hipStream_t)stream;
  uint8_t* p = static_cast<uint8_t*>(P);
  uint8_t* s = static_cast<uint8_t*>(S);
  switch (src) {
    case FP4X_SRC_F32: return launch_nv4_amax(SrcF32{static_cast<const float*>(src_a), K}, N, K, amax, p, s, st);
    case FP4X_SRC_BF16: return launch_nv4_amax(SrcBF16{static_cast<const uint16_t*>(src_a), K}, N, K, amax, p, s, st);
    case FP4X_SRC_MX8:
      return launch_nv4_amax(SrcMX8{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), K}, N, K,
                             amax, p, s, st);
    default:
      return launch_nv4_amax(SrcNV4{static_cast<const uint8_t*>(src_a), static_cast<const uint8_t*>(src_b), src_gs, K},
                             N, K, amax, p, s, st);
  }
}

}  // extern "C"
