// Blocked GEMM over packed weights (gfx950), any number of rows M:
//   y[m, n] = gs * sum_k x[m, k] * w[n, k],
// x bf16, w decoded to the bf16 operand of its format (fp4x_gemv.h), fp32
// accumulation on v_mfma_f32_16x16x32_bf16.
//
// It serves more than 16 rows, which the other kernels take as one launch per
// 16 rows (each reading every weight again), and the shapes of up to 16 rows
// that only the MFMA core took (rows too few or too long for the streaming
// kernels, K not a multiple of 512), and some of the few-rows kernels' shapes
// at 9 to 16 rows (gemm_before_rows).
//
// A workgroup owns a tile of 16 MT rows of x and 16 NT WN rows of w.  Its WN x
// WK waves split the tile's columns WN ways and K WK ways.  K advances in
// units of 128 values: a wave's unit is NT strips of 16 weight rows as they
// are packed, and the WN waves of a K part share that part's activation unit.
// Both go to LDS by direct loads (no registers) through a ring of D stages,
// so later stages are on their way while one is used.  A wave then decodes
// its strips in registers and multiplies them with every row group, so each
// weight is decoded once per tile.  With WN = 1 a ring belongs to one wave
// and no barrier is needed; otherwise a stage starts with one.
//
// What bounds it (MXFP8 [16384 x 2560], copies with parts left out): at M = 64
// its loads alone take 17 of 19 us and grow by 1.9 us per 16 rows, which is
// the tile's bytes (weights from HBM, activations from L2) at about 40 GB/s
// per CU, whatever the ring's depth; loads that all hit L2 reach 140.  So
// tiles are as large as leaves every CU one.  At M = 256 (26 us of loads, 30
// of decoding and MFMA, 38-40 in all) larger wave tiles, through direct loads
// or registers, took 37-41 and were slower on every narrower matrix; torch's
// bf16 product of that size takes 41 with its weights from HBM.
//
// us per call with weights from HBM (graph replays of 8 to 64 calls on weights
// of their own, 1 GB read before each), one launch per 16 rows -> this:
//   M                     24          64          256
//   MXFP8 [16384 x 2560]  23 -> 14    44 -> 21    169 -> 39
//   MXFP8 [2560 x 6144]   25 -> 12    67 -> 16    263 -> 29
//   W6 [1280 x 2560]      21 -> 6.1   51 -> 7.1   202 -> 11
//   NVFP4 [13312 x 2560]  18 -> 12    38 -> 17    145 -> 39
//   W8 [2560 x 640]       12 -> 4.8   26 -> 5.4   112 -> 6.9
// and against the core: at M = 16 [5000 x 1920] 12-13 -> 6.8-8.3, [2560 x 6144]
// 17-19 -> 10, [1280 x 2560] 9-12 -> 5.8-6.5, [2560 x 640] 6.7-9.0 -> 4.1-4.3;
// at M = 1, 2 and 4 [9000 x 1088] 12-16 -> 7.0-9.1.  Over 29 to 107 such calls
// per row count from 1 to 16 it takes 0.64 to 0.70 of the core's time, 0.92 at
// most (K = 1088 to 4160, 2100 to 16000 rows).
#pragma once
#include <type_traits>
#include "fp4x_stream.h"
#include "../../include/fp4x.h"

namespace fp4x {

// The four 8-value pieces at a[0..3] of G row groups (4096 bytes apart), and
// the wait for them, in one block.
template <int G>
__device__ __forceinline__ void lds_read_x(uint4 (&x)[4 * G], const uint32_t (&a)[4]) {
  static_assert(G >= 1 && G <= 4, "row groups per block");
  if constexpr (G == 1) {
    asm volatile(
        "ds_read_b128 %0, %4\n\t"
        "ds_read_b128 %1, %5\n\t"
        "ds_read_b128 %2, %6\n\t"
        "ds_read_b128 %3, %7\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
  } else if constexpr (G == 2) {
    asm volatile(
        "ds_read_b128 %0, %8\n\t"
        "ds_read_b128 %1, %9\n\t"
        "ds_read_b128 %2, %10\n\t"
        "ds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %8 offset:4096\n\t"
        "ds_read_b128 %5, %9 offset:4096\n\t"
        "ds_read_b128 %6, %10 offset:4096\n\t"
        "ds_read_b128 %7, %11 offset:4096\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
  } else if constexpr (G == 3) {
    asm volatile(
        "ds_read_b128 %0, %12\n\t"
        "ds_read_b128 %1, %13\n\t"
        "ds_read_b128 %2, %14\n\t"
        "ds_read_b128 %3, %15\n\t"
        "ds_read_b128 %4, %12 offset:4096\n\t"
        "ds_read_b128 %5, %13 offset:4096\n\t"
        "ds_read_b128 %6, %14 offset:4096\n\t"
        "ds_read_b128 %7, %15 offset:4096\n\t"
        "ds_read_b128 %8, %12 offset:8192\n\t"
        "ds_read_b128 %9, %13 offset:8192\n\t"
        "ds_read_b128 %10, %14 offset:8192\n\t"
        "ds_read_b128 %11, %15 offset:8192\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7]), "=&v"(x[8]), "=&v"(x[9]), "=&v"(x[10]), "=&v"(x[11])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
  } else {
    asm volatile(
        "ds_read_b128 %0, %16\n\t"
        "ds_read_b128 %1, %17\n\t"
        "ds_read_b128 %2, %18\n\t"
        "ds_read_b128 %3, %19\n\t"
        "ds_read_b128 %4, %16 offset:4096\n\t"
        "ds_read_b128 %5, %17 offset:4096\n\t"
        "ds_read_b128 %6, %18 offset:4096\n\t"
        "ds_read_b128 %7, %19 offset:4096\n\t"
        "ds_read_b128 %8, %16 offset:8192\n\t"
        "ds_read_b128 %9, %17 offset:8192\n\t"
        "ds_read_b128 %10, %18 offset:8192\n\t"
        "ds_read_b128 %11, %19 offset:8192\n\t"
        "ds_read_b128 %12, %16 offset:12288\n\t"
        "ds_read_b128 %13, %17 offset:12288\n\t"
        "ds_read_b128 %14, %18 offset:12288\n\t"
        "ds_read_b128 %15, %19 offset:12288\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3]), "=&v"(x[4]), "=&v"(x[5]), "=&v"(x[6]), "=&v"(x[7]), "=&v"(x[8]), "=&v"(x[9]), "=&v"(x[10]), "=&v"(x[11]), "=&v"(x[12]), "=&v"(x[13]), "=&v"(x[14]), "=&v"(x[15])
        : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
  }
}

constexpr int kGemmKB = 128;                       // k values of a unit

// A unit of a format: 16 weight rows x 128 k values in LDS, filled by direct
// loads.  Strip: the lane's addresses for one strip of 16 rows.  Lane (i, g)
// consumes k values [32 g, 32 g + 32) of row i.
//
// Scales: 16 rows x 2 dwords that hold the row's scales of the unit, the
// first one at byte `off & 3` where the rows' scales are only 2-byte aligned.
struct GemmScales {
  const uint8_t* s;                                // a whole dword of the plane
  uint32_t o;                                      // this lane's row's scale bytes, from s
  int last;                                        // last whole dword of the plane, from s
  // rb: scale bytes of a row; the plane holds at least one whole dword.  A
  // strip of the last row alone can begin past the last whole dword (two bytes
  // a row, K = 64, N odd): s is then that dword, so no offset is below 0.
  __host__ __device__ void set(const uint8_t* plane, int64_t n0, int row, int rb, int64_t N) {
    const int64_t at = n0 * rb, end = N * rb - 4, b = (at < end ? at : end) & ~(int64_t)3;
    s = plane + b;
    o = (uint32_t)(row * rb + (int)(at - b));
    last = (int)(end - b < 0x7ffffffc ? end - b : 0x7ffffffc) & ~3;
  }
  // ub: scale bytes of a row in a unit; d: dword 0 or 1
  __host__ __device__ const uint8_t* at(int ku, int ub, int d) const {
    const int a = (int)((o + ku * ub) & ~3u) + 4 * d;
    return s + (uint32_t)(a < last ? a : last);
  }
  __device__ void issue(char* l, int ku, int ub, int d) const { dma_b32(at(ku, ub, d), l); }
};

template <class F> struct GemmUnit;

// Bytes by which piece p of a unit of n pieces lies past the row's last piece
// when the row ends `cut` pieces before the unit does.
__device__ __forceinline__ uint32_t gemm_past(int p, int n, int cut) {
  const int over = p - (n - 1 - cut);
  return over > 0 ? (uint32_t)over * 16 : 0;
}

// 16 rows x 128 bytes (MXFP8, W8): two 16-byte loads of 8 rows, row r's piece p at p ^ ((r >> 1) & 7)
struct GemmRows128 {
  const uint8_t* w;
  uint32_t o[2];
  __device__ void set(const uint8_t* plane, int64_t n0, int K, int lane, int lim, int nt) {
    w = plane + n0 * K;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = h * 8 + (lane >> 3), rm = (r >> 2) * nt + (r & 3);
      o[h] = (uint32_t)(rm < lim ? rm : lim) * (uint32_t)K + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    }
  }
  // cut: the unit's pieces past the row's end (0 but for a last partial unit), which read the row's last piece
  __device__ void issue(char* l, int ku, int lane, int cut) const {
    const uint8_t* u = w + ku * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint32_t v = o[h];
      if (cut) v -= gemm_past((lane & 7) ^ (((h * 8 + (lane >> 3)) >> 1) & 7), 8, cut);
      dma_b128(u + v, l + h * 1024);
    }
  }
  __device__ static uint32_t at(uint32_t u, int i, int p) { return u + i * 128 + ((p ^ ((i >> 1) & 7)) * 16); }
};
// 16 rows x 64 bytes (W6 low nibbles, NVFP4): one 16-byte load, row r's piece p at p ^ ((r >> 2) & 3)
struct GemmRows64 {
  const uint8_t* w;
  uint32_t o;
  __device__ void set(const uint8_t* plane, int64_t n0, int rb, int lane, int lim, int nt) {
    const int r = lane >> 2, rm = (r >> 2) * nt + (r & 3);
    w = plane + n0 * rb;
    o = (uint32_t)(rm < lim ? rm : lim) * (uint32_t)rb + ((lane & 3) ^ ((r >> 2) & 3)) * 16;
  }
  __device__ void issue(char* l, int ku, int lane, int cut) const {
    uint32_t v = o;
    if (cut) v -= gemm_past((lane & 3) ^ ((lane >> 4) & 3), 4, cut);
    dma_b128(w + ku * 64 + v, l);
  }
  __device__ static uint32_t at(uint32_t u, int i, int p) { return u + i * 64 + ((p ^ ((i >> 2) & 3)) * 16); }
};

template <> struct GemmUnit<FmtMX8> {
  static bool on(const Switches& w) { return w.mx8_stream; }
  static constexpr int BYTES = 2048 + 128, NDMA = 3;
  static constexpr float DEQ = 0.5f;                // VALU operations per weight
  static constexpr int KMULT = 64;
  static constexpr bool MX = true, ODD2 = true;
  GemmRows128 w;
  GemmScales s;
  __device__ void set(const PlaneArgs& a, int64_t n0, int64_t N, int lane, int lim, int nt) {
    w.set(a.w0, n0, a.K, lane, lim, nt);
    const int r = (lane & 31) >> 1, rm = (r >> 2) * nt + (r & 3);
    s.set(a.s, n0, rm < lim ? rm : lim, a.K / 32, N);
  }
  __device__ void issue(char* l, int ku, int lane, int cut) const {
    w.issue(l, ku, lane, cut);
    if (lane < 32) s.issue(l + 2048, ku, 4, lane & 1);
  }
  struct Raw { uint4 q[2]; uint32_t e; };
  // the NT strips' operands of lane (i, g), and the wait for them, in one block
  template <int NT>
  __device__ static void read(Raw (&r)[NT], uint32_t u, int i, int g, uint32_t so) {
    const uint32_t a0 = GemmRows128::at(u, i, 2 * g), a1 = GemmRows128::at(u, i, 2 * g + 1);
    const uint32_t sa = u + 2048 + i * 8 + (so & 3) + g;
    if constexpr (NT == 1) {
      asm volatile(
          "ds_read_b128 %0, %3\n\t"
          "ds_read_b128 %1, %4\n\t"
          "ds_read_u8 %2, %5\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e)
          : "v"(a0), "v"(a1), "v"(sa) : "memory");
    }
    else {
      static_assert(NT == 2, "strips per wave");
      asm volatile(
          "ds_read_b128 %0, %6\n\t"
          "ds_read_b128 %1, %7\n\t"
          "ds_read_u8 %2, %8\n\t"
          "ds_read_b128 %3, %6 offset:%9\n\t"
          "ds_read_b128 %4, %7 offset:%9\n\t"
          "ds_read_u8 %5, %8 offset:%9\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e), "=&v"(r[1].q[0]), "=&v"(r[1].q[1]), "=&v"(r[1].e)
          : "v"(a0), "v"(a1), "v"(sa), "n"(1 * BYTES) : "memory");
    }
  }
  __device__ static uint32_t scale_off(const PlaneArgs& a, int64_t n) { return (uint32_t)(n * (a.K / 32)); }
  static constexpr int UB = 4;
  __device__ static void last_scale(Raw& r, const PlaneArgs& a, int64_t N, int g) {
    if (g < 2)
      asm volatile("global_load_ubyte %0, %1, off\n\ts_waitcnt vmcnt(0)"
                   : "=&v"(r.e) : "v"(a.s + N * (a.K / 32) - 2 + g) : "memory");
  }
  __device__ static void deq(const Raw& r, int h, uint32_t (&w)[8]) {
    const float sc = e8m0_to_f32(r.e);
    const uint4 q = r.q[h];
    w[0] = fp8x2_to_bf16x2<false>(q.x, sc); w[1] = fp8x2_to_bf16x2<true>(q.x, sc);
    w[2] = fp8x2_to_bf16x2<false>(q.y, sc); w[3] = fp8x2_to_bf16x2<true>(q.y, sc);
    w[4] = fp8x2_to_bf16x2<false>(q.z, sc); w[5] = fp8x2_to_bf16x2<true>(q.z, sc);
    w[6] = fp8x2_to_bf16x2<false>(q.w, sc); w[7] = fp8x2_to_bf16x2<true>(q.w, sc);
  }
};

template <bool F16S> struct GemmUnit<FmtW8<F16S>> {
  static bool on(const Switches& w) { return w.w8_stream; }
  static constexpr int BYTES = 2048 + 128, NDMA = 3, SB = F16S ? 2 : 4;
  static constexpr float DEQ = 2.5f;
  static constexpr int KMULT = 64;
  static constexpr bool MX = false, ODD2 = F16S;
  GemmRows128 w;
  GemmScales s;
  __device__ void set(const PlaneArgs& a, int64_t n0, int64_t N, int lane, int lim, int nt) {
    w.set(a.w0, n0, a.K, lane, lim, nt);
    const int r = (lane & 31) >> 1, rm = (r >> 2) * nt + (r & 3);
    s.set(a.s, n0, rm < lim ? rm : lim, a.K / 64 * SB, N);
  }
  __device__ void issue(char* l, int ku, int lane, int cut) const {
    w.issue(l, ku, lane, cut);
    if (lane < 32) s.issue(l + 2048, ku, 2 * SB, lane & 1);
  }
  struct Raw { uint4 q[2]; uint32_t e; };
  // the NT strips' operands of lane (i, g), and the wait for them, in one block
  template <int NT>
  __device__ static void read(Raw (&r)[NT], uint32_t u, int i, int g, uint32_t so) {
    const uint32_t a0 = GemmRows128::at(u, i, 2 * g), a1 = GemmRows128::at(u, i, 2 * g + 1);
    const uint32_t sa = u + 2048 + i * 8 + (so & 3) + (g >> 1) * SB;
    if constexpr (F16S) {
    if constexpr (NT == 1) {
      asm volatile(
          "ds_read_b128 %0, %3\n\t"
          "ds_read_b128 %1, %4\n\t"
          "ds_read_u16 %2, %5\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e)
          : "v"(a0), "v"(a1), "v"(sa) : "memory");
    }
    else {
      static_assert(NT == 2, "strips per wave");
      asm volatile(
          "ds_read_b128 %0, %6\n\t"
          "ds_read_b128 %1, %7\n\t"
          "ds_read_u16 %2, %8\n\t"
          "ds_read_b128 %3, %6 offset:%9\n\t"
          "ds_read_b128 %4, %7 offset:%9\n\t"
          "ds_read_u16 %5, %8 offset:%9\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e), "=&v"(r[1].q[0]), "=&v"(r[1].q[1]), "=&v"(r[1].e)
          : "v"(a0), "v"(a1), "v"(sa), "n"(1 * BYTES) : "memory");
    }
    } else {
    if constexpr (NT == 1) {
      asm volatile(
          "ds_read_b128 %0, %3\n\t"
          "ds_read_b128 %1, %4\n\t"
          "ds_read_b32 %2, %5\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e)
          : "v"(a0), "v"(a1), "v"(sa) : "memory");
    }
    else {
      static_assert(NT == 2, "strips per wave");
      asm volatile(
          "ds_read_b128 %0, %6\n\t"
          "ds_read_b128 %1, %7\n\t"
          "ds_read_b32 %2, %8\n\t"
          "ds_read_b128 %3, %6 offset:%9\n\t"
          "ds_read_b128 %4, %7 offset:%9\n\t"
          "ds_read_b32 %5, %8 offset:%9\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[0].e), "=&v"(r[1].q[0]), "=&v"(r[1].q[1]), "=&v"(r[1].e)
          : "v"(a0), "v"(a1), "v"(sa), "n"(1 * BYTES) : "memory");
    }
    }
  }
  __device__ static uint32_t scale_off(const PlaneArgs& a, int64_t n) { return (uint32_t)(n * (a.K / 64) * SB); }
  static constexpr int UB = 2 * SB;
  __device__ static void last_scale(Raw& r, const PlaneArgs& a, int64_t N, int g) {
    if (g < 2)
      asm volatile("global_load_ushort %0, %1, off\n\ts_waitcnt vmcnt(0)"
                   : "=&v"(r.e) : "v"(a.s + N * (a.K / 64) * SB - 2) : "memory");
  }
  __device__ static void deq(const Raw& r, int h, uint32_t (&w)[8]) {
    w8_chunk_bf16(r.q[h], FmtW8<F16S>::scale(r.e), w);
  }
};

template <> struct GemmUnit<FmtW6> {
  static bool on(const Switches& w) { return w.w6_stream; }
  static constexpr int BYTES = 1024 + 512 + 128, NDMA = 3;
  static constexpr float DEQ = 3.9f;                // VALU operations per weight
  static constexpr int KMULT = 64;
  static constexpr bool MX = false, ODD2 = false;
  GemmRows64 l;
  const uint8_t* hp;
  uint32_t ho;
  GemmScales s;
  __device__ void set(const PlaneArgs& a, int64_t n0, int64_t N, int lane, int lim, int nt) {
    l.set(a.w0, n0, a.K / 2, lane, lim, nt);
    const int r = (lane & 31) >> 1, rm = (r >> 2) * nt + (r & 3), rc = rm < lim ? rm : lim;
    hp = a.w1 + n0 * (a.K / 4);
    ho = (uint32_t)rc * (uint32_t)(a.K / 4) + ((lane & 1) ^ (r >> 3)) * 16;
    s.set(a.s, n0, rc, a.K / 16, N);
  }
  __device__ void issue(char* d, int ku, int lane, int cut) const {
    l.issue(d, ku, lane, cut >> 1);
    if (lane < 32) {
      uint32_t v = ho;
      if (cut) v -= gemm_past((lane & 1) ^ (lane >> 4), 2, cut >> 2);
      dma_b128(hp + ku * 32 + v, d + 1024);
      s.issue(d + 1536, ku, 8, lane & 1);
    }
  }
  struct Raw { uint4 lo; uint2 hi; uint32_t e; };
  // the NT strips' operands of lane (i, g), and the wait for them, in one block
  template <int NT>
  __device__ static void read(Raw (&r)[NT], uint32_t u, int i, int g, uint32_t so) {
    const uint32_t a0 = GemmRows64::at(u, i, g), a1 = u + 1024 + i * 32 + (((g >> 1) ^ (i >> 3)) * 16) + (g & 1) * 8;
    const uint32_t sa = u + 1536 + i * 8 + (so & 3) + g * 2;
    if constexpr (NT == 1) {
      asm volatile(
          "ds_read_b128 %0, %3\n\t"
          "ds_read_b64 %1, %4\n\t"
          "ds_read_u16 %2, %5\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].lo), "=&v"(r[0].hi), "=&v"(r[0].e)
          : "v"(a0), "v"(a1), "v"(sa) : "memory");
    }
    else {
      static_assert(NT == 2, "strips per wave");
      asm volatile(
          "ds_read_b128 %0, %6\n\t"
          "ds_read_b64 %1, %7\n\t"
          "ds_read_u16 %2, %8\n\t"
          "ds_read_b128 %3, %6 offset:%9\n\t"
          "ds_read_b64 %4, %7 offset:%9\n\t"
          "ds_read_u16 %5, %8 offset:%9\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].lo), "=&v"(r[0].hi), "=&v"(r[0].e), "=&v"(r[1].lo), "=&v"(r[1].hi), "=&v"(r[1].e)
          : "v"(a0), "v"(a1), "v"(sa), "n"(1 * BYTES) : "memory");
    }
  }
  __device__ static uint32_t scale_off(const PlaneArgs& a, int64_t n) { return (uint32_t)(n * (a.K / 16)); }
  static constexpr int UB = 8;
  __device__ static void last_scale(Raw&, const PlaneArgs&, int64_t, int) {}
  __device__ static void deq(const Raw& r, int h, uint32_t (&w)[8]) {
    FmtW6::Chunk c;
    c.lo = r.lo;
    c.hi = r.hi;
    c.s = r.e;
    FmtW6::deq16(c, h, w);
  }
};

template <> struct GemmUnit<FmtNV4> {
  static bool on(const Switches& w) { return w.nv4_stream; }
  static constexpr int BYTES = 1024 + 128, NDMA = 2;
  static constexpr float DEQ = 2.0f;                // VALU operations per weight
  static constexpr int KMULT = 64;
  static constexpr bool MX = false, ODD2 = false;
  GemmRows64 w;
  GemmScales s;
  __device__ void set(const PlaneArgs& a, int64_t n0, int64_t N, int lane, int lim, int nt) {
    w.set(a.w0, n0, a.K / 2, lane, lim, nt);
    const int r = (lane & 31) >> 1, rm = (r >> 2) * nt + (r & 3);
    s.set(a.s, n0, rm < lim ? rm : lim, a.K / 16, N);
  }
  __device__ void issue(char* d, int ku, int lane, int cut) const {
    w.issue(d, ku, lane, cut >> 1);
    if (lane < 32) s.issue(d + 1024, ku, 8, lane & 1);
  }
  struct Raw { uint4 q; uint32_t e; };
  // the NT strips' operands of lane (i, g), and the wait for them, in one block
  template <int NT>
  __device__ static void read(Raw (&r)[NT], uint32_t u, int i, int g, uint32_t so) {
    const uint32_t a0 = GemmRows64::at(u, i, g), sa = u + 1024 + i * 8 + (so & 3) + g * 2;
    if constexpr (NT == 1) {
      asm volatile(
          "ds_read_b128 %0, %2\n\t"
          "ds_read_u16 %1, %3\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q), "=&v"(r[0].e)
          : "v"(a0), "v"(sa) : "memory");
    }
    else {
      static_assert(NT == 2, "strips per wave");
      asm volatile(
          "ds_read_b128 %0, %4\n\t"
          "ds_read_u16 %1, %5\n\t"
          "ds_read_b128 %2, %4 offset:%6\n\t"
          "ds_read_u16 %3, %5 offset:%6\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(r[0].q), "=&v"(r[0].e), "=&v"(r[1].q), "=&v"(r[1].e)
          : "v"(a0), "v"(sa), "n"(1 * BYTES) : "memory");
    }
  }
  __device__ static uint32_t scale_off(const PlaneArgs& a, int64_t n) { return (uint32_t)(n * (a.K / 16)); }
  static constexpr int UB = 8;
  __device__ static void last_scale(Raw&, const PlaneArgs&, int64_t, int) {}
  __device__ static void deq(const Raw& r, int h, uint32_t (&w)[8]) {
    FmtNV4::Chunk c;
    c.q = r.q;
    c.s = r.e;
    FmtNV4::deq16(c, h, w);
  }
};

template <> struct GemmUnit<FmtBF16> {
  static bool on(const Switches&) { return true; }
  static constexpr int BYTES = 4096, NDMA = 4;
  static constexpr float DEQ = 0.0f;                // VALU operations per weight
  static constexpr int KMULT = 16;
  static constexpr bool MX = false, ODD2 = false;
  const uint8_t* w;
  uint32_t o[4];
  __device__ void set(const PlaneArgs& a, int64_t n0, int64_t, int lane, int lim, int nt) {
    w = a.w0 + n0 * a.K * 2;
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int r = h * 4 + (lane >> 4), rm = (r >> 2) * nt + (r & 3);
      o[h] = (uint32_t)(rm < lim ? rm : lim) * (uint32_t)(a.K * 2) + ((lane & 15) ^ r) * 16;
    }
  }
  __device__ void issue(char* d, int ku, int lane, int cut) const {
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      uint32_t v = o[h];
      if (cut) v -= gemm_past((lane & 15) ^ (h * 4 + (lane >> 4)), 16, 2 * cut);
      dma_b128(w + ku * 256 + v, d + h * 1024);
    }
  }
  struct Raw { uint4 q[4]; };
  template <int NT>
  __device__ static void read(Raw (&r)[NT], uint32_t u, int i, int g, uint32_t) {
    const uint32_t b = u + i * 256;
    const uint32_t a[4] = {b + (((4 * g) ^ i) * 16), b + (((4 * g + 1) ^ i) * 16), b + (((4 * g + 2) ^ i) * 16),
                           b + (((4 * g + 3) ^ i) * 16)};
    uint4 q[4 * NT];
    lds_read_x<NT>(q, a);                          // strips are 4096 bytes apart, as row groups are
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) r[t].q[j] = q[t * 4 + j];
  }
  __device__ static uint32_t scale_off(const PlaneArgs&, int64_t) { return 0; }
  static constexpr int UB = 0;
  __device__ static void last_scale(Raw&, const PlaneArgs&, int64_t, int) {}
  __device__ static void deq(const Raw& r, int h, uint32_t (&w)[8]) {
    const uint4 a = r.q[2 * h], b = r.q[2 * h + 1];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
    w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
  }
};

template <class F, int MT, int NT, int WN, int WK, int D>
struct GemmShape {
  static constexpr int BM = 16 * MT, BN = 16 * NT * WN, THREADS = 64 * WN * WK;
  static constexpr int XU = MT * 4096, WU = NT * GemmUnit<F>::BYTES;
  static constexpr int STAGE = WK * XU + WN * WK * WU;
  static constexpr int XI = 4 * MT / WN;                   // activation loads per wave and stage
  static constexpr int C = XI + NT * GemmUnit<F>::NDMA;    // loads per wave and stage
  static constexpr int RED = WK > 1 ? WK * WN * MT * NT * 1024 : 0;   // K parts' sums, then a word per wave
  static constexpr int LDS = D * STAGE > RED + 64 ? D * STAGE : RED + 64;
};

// Output (m, n) when row n has MXFP8's exponent 255, which the reference
// takes as the scale +inf (+-inf, or NaN for a zero or NaN code) and the
// scaled convert as NaN: such a sum is +-inf or NaN, in any order.
__device__ __forceinline__ void gemm_inf_fix(const GemvLaunch& p, int m, int64_t n) {
  bool met = false;
  for (int c = 0; c < p.pa.K / 32; ++c) met |= p.pa.s[n * (p.pa.K / 32) + c] == 255;
  if (!met) return;
  float acc = 0.0f;
  for (int c = 0; c < p.pa.K / 16; ++c) {
    uint32_t w[8];
    FmtMX8::deq16(FmtMX8::load(p.pa, n, c), 0, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t v = *reinterpret_cast<const uint32_t*>(p.x + m * p.x_stride + c * 16 + 2 * i);
      acc = __builtin_fmaf(bf16_lo(w[i]), bf16_lo(v), acc);
      acc = __builtin_fmaf(bf16_hi(w[i]), bf16_hi(v), acc);
    }
  }
  store_out(p.out, m * p.out_stride + n, p.out_dtype, acc * p.gs);
}

__device__ __forceinline__ void gemm_store4(const GemvLaunch& p, int m, int64_t n, f32x4_t v, bool vec) {
  const int64_t at = m * p.out_stride + n;
  v[0] *= p.gs; v[1] *= p.gs; v[2] *= p.gs; v[3] *= p.gs;
  if (vec) {
    if (p.out_dtype == DT_BF16) {
      uint2 o = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(p.out) + at) = o;
      return;
    }
    if (p.out_dtype == DT_F32) {
      *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(p.out) + at) = v;
      return;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < p.N) store_out(p.out, at + r, p.out_dtype, v[r]);
}

// Waits until at most `later` stages of C loads are outstanding.
template <int C, int MAX>
__device__ __forceinline__ void gemm_wait(int later) {
  if constexpr (MAX > 0) {
    if (later >= MAX) wait_vmcnt<MAX * C>();
    else gemm_wait<C, MAX - 1>(later);
  } else {
    wait_vmcnt<0>();
  }
}

template <class F, int MT, int NT, int WN, int WK, int D>
__global__ __launch_bounds__(64 * WN * WK) __attribute__((amdgpu_waves_per_eu(2))) void gemm_kernel(GemvLaunch p, int mtiles, int ntiles, int vec, int odd) {
  using S = GemmShape<F, MT, NT, WN, WK, D>;
  using U = GemmUnit<F>;
  constexpr bool MX = U::MX, ODD2 = U::ODD2;
  extern __shared__ __align__(16) uint16_t lds[];
  char* base = reinterpret_cast<char*>(lds);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int i16 = lane & 15, g = lane >> 4;
  // workgroups that share an XCD (equal index mod 8) take consecutive tiles, row tiles of one column tile together
  const int total = mtiles * ntiles, per = (total + 7) / 8;
  const int item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (item >= total || (int)(blockIdx.x >> 3) >= per) return;
  const int nt0 = item / mtiles, m0 = (item - nt0 * mtiles) * S::BM;
  const int64_t n0 = (int64_t)nt0 * S::BN + wn * 16 * NT;
  const int K = p.pa.K, nu = (K + kGemmKB - 1) / kGemmKB;
  const int steps = (nu + WK - 1) / WK, cnt = (nu - wk + WK - 1) / WK;
  // strip t's row i is output column n0 + (i >> 2) * 4 NT + 4 t + (i & 3): a lane's sums are then 4 NT consecutive columns
  U unit[NT];
  uint32_t so = 0;                                         // strips differ by multiples of 4 rows: one byte offset
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int64_t ns = n0 + 4 * t < p.N ? n0 + 4 * t : p.N - 1;
    const int64_t left = p.N - 1 - ns;
    const int lim = left < 16 * NT ? (int)left : 16 * NT, rm = (i16 >> 2) * 4 * NT + (i16 & 3);
    unit[t].set(p.pa, ns, p.N, lane, lim, 4 * NT);
    if (t == 0) so = U::scale_off(p.pa, ns + (rm < lim ? rm : lim));
  }
  // activation rows m0 + 4 (wn XI + h) + (lane >> 4): bytes from row m0, piece (lane & 15) ^ row at position lane & 15
  const uint16_t* x0 = p.x + m0 * p.x_stride;
  uint32_t xo[S::XI];
#pragma unroll
  for (int h = 0; h < S::XI; ++h) {
    const int row = (wn * S::XI + h) * 4 + (lane >> 4), m = m0 + row < p.M ? row : p.M - 1 - m0;
    xo[h] = (uint32_t)(m * p.x_stride * 2) + ((lane & 15) ^ (row & 15)) * 16;
  }
  auto issue_unit = [&](int slot, int ku, auto cut_c) {
    constexpr bool CUT = decltype(cut_c)::value;
    char* xb = base + slot * S::STAGE + wk * S::XU + wn * S::XI * 1024;
    char* wb = base + slot * S::STAGE + WK * S::XU + wave * S::WU;
    const int cut = CUT ? ((ku + 1) * kGemmKB - K) / 16 : 0;
#pragma unroll
    for (int t = 0; t < NT; ++t) unit[t].issue(wb + t * U::BYTES, ku, lane, cut);
    const uint8_t* xu = reinterpret_cast<const uint8_t*>(x0) + ku * (kGemmKB * 2);
#pragma unroll
    for (int h = 0; h < S::XI; ++h) {
      uint32_t v = xo[h];
      if (CUT) v -= gemm_past((lane & 15) ^ (((wn * S::XI + h) * 4 + (lane >> 4)) & 15), 16, 2 * cut);
      dma_b128(xu + v, xb + h * 1024);
    }
  };
  auto issue = [&](int slot, int s) {
    if (s >= cnt) return;
    const int ku = s * WK + wk;
    if ((ku + 1) * kGemmKB > K) issue_unit(slot, ku, std::true_type{});
    else issue_unit(slot, ku, std::false_type{});
  };
  // zeroes this wave's activation pieces past K of a partial unit
  auto clear_past = [&](int slot, int s) {
    const int ku = s * WK + wk, left = K - ku * kGemmKB;
    if (s >= cnt || left >= kGemmKB) return;
    const uint32_t xb = lds_addr(base) + slot * S::STAGE + wk * S::XU + wn * S::XI * 1024 + lane * 16;
#pragma unroll
    for (int h = 0; h < S::XI; ++h) {
      const int row = (wn * S::XI + h) * 4 + (lane >> 4);
      if ((((lane & 15) ^ row) & 15) * 8 >= left) lds_put_f32x4(xb + h * 1024, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
    }
  };
  uint32_t seen = 0;                                       // MXFP8: the largest exponent met
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mt][t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const uint32_t l0 = lds_addr(base);
  auto consume = [&](int slot, int s) {
    const int ku = s * WK + wk;
    const uint32_t xb = l0 + slot * S::STAGE + wk * S::XU + i16 * 256, wb = l0 + slot * S::STAGE + WK * S::XU + wave * S::WU;
    typename U::Raw raw[NT];
    U::template read<NT>(raw, wb, i16, g, so + ku * U::UB);
    const int left = K - ku * kGemmKB;                     // k values of the row from this unit on
    if (ODD2 && left <= kGemmKB && odd) {                  // the plane's last two bytes lie past its last whole dword
#pragma unroll
      for (int t = 0; t < NT; ++t)
        if (n0 + (i16 >> 2) * 4 * NT + t * 4 + (i16 & 3) == p.N - 1) U::last_scale(raw[t], p.pa, p.N, g);
    }
    const bool dead = g * 32 >= left;
    uint4 w[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (U::UB > 0) {
        if constexpr (MX) seen = raw[t].e > seen ? raw[t].e : seen;
        raw[t].e = dead ? 0 : raw[t].e;
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t d[8];
        U::deq(raw[t], h, d);
        if constexpr (U::UB == 0) {
          const bool gone = g * 32 + h * 16 >= left;
#pragma unroll
          for (int i = 0; i < 8; ++i) d[i] = gone ? 0 : d[i];
        }
        w[t][2 * h] = make_uint4(d[0], d[1], d[2], d[3]);
        w[t][2 * h + 1] = make_uint4(d[4], d[5], d[6], d[7]);
      }
    }
    constexpr int MG = MT <= 4 ? MT : 4;                   // row groups per read block
#pragma unroll
    for (int m1 = 0; m1 < MT; m1 += MG) {
      uint4 x[4 * MG];
      uint32_t a[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = xb + m1 * 4096 + (((4 * g + j) ^ i16) * 16);
      lds_read_x<MG>(x, a);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mm = 0; mm < MG; ++mm)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[m1 + mm][t] = mfma16(w[t][j], x[mm * 4 + j], acc[m1 + mm][t]);
    }
  };
  if constexpr (WN == 1) {                                 // wave-private rings: no barrier
#pragma unroll
    for (int d = 0; d < D; ++d) issue(d, d);
    for (int s = 0, slot = 0; s < cnt; ++s) {
      gemm_wait<S::C, D - 1>(cnt - 1 - s < D - 1 ? cnt - 1 - s : D - 1);
      clear_past(slot, s);
      consume(slot, s);
      issue(slot, s + D);
      if (++slot == D) slot = 0;
    }
  } else {
#pragma unroll
    for (int d = 0; d < D - 1; ++d) issue(d, d);
    for (int s = 0, slot = 0; s < steps; ++s) {
      const int later = cnt - 1 - s < D - 2 ? cnt - 1 - s : D - 2;
      gemm_wait<S::C, D - 2>(later > 0 ? later : 0);
      clear_past(slot, s);
      wg_barrier_raw();
      issue(slot == 0 ? D - 1 : slot - 1, s + D - 1);
      if (s < cnt) consume(slot, s);
      if (++slot == D) slot = 0;
    }
  }

  const int mrow = m0 + i16;
  bool inf = MX && __builtin_amdgcn_ballot_w64(seen == 255u) != 0;
  if constexpr (WK == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int64_t n = n0 + g * 4 * NT + t * 4;
        if (mrow + mt * 16 < p.M) gemm_store4(p, mrow + mt * 16, n, acc[mt][t], vec && n + 3 < p.N);
      }
  } else {
    // the rings are drained: their LDS holds the K parts, added in part order
    wg_barrier_raw();
    const uint32_t rb = l0 + lane * 16;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < NT; ++t) lds_put_f32x4(rb + ((wk * WN + wn) * MT * NT + mt * NT + t) * 1024, acc[mt][t]);
    if constexpr (MX) {
      if (lane == 0)
        asm volatile("ds_write_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" ::"v"(l0 + S::RED + wave * 4), "v"((int)inf) : "memory");
    }
    wg_barrier_raw();
    if constexpr (MX) {                                    // any of the K parts' waves
      typedef const __attribute__((address_space(3))) int* lds_int_ptr;
      int any = 0;
#pragma unroll
      for (int w = 0; w < WK; ++w) any |= *reinterpret_cast<lds_int_ptr>((uintptr_t)(l0 + S::RED + (w * WN + wn) * 4));
      inf = __builtin_amdgcn_readfirstlane(any) != 0;
    }
    for (int f = wk; f < MT * NT; f += WK) {
      typedef const __attribute__((address_space(3))) f32x4_t* lds_f32x4_ptr;
      f32x4_t o[WK];
#pragma unroll
      for (int w = 0; w < WK; ++w)
        o[w] = *reinterpret_cast<lds_f32x4_ptr>((uintptr_t)(rb + ((w * WN + wn) * MT * NT + f) * 1024));
      f32x4_t v = o[0];
#pragma unroll
      for (int w = 1; w < WK; ++w) { v[0] += o[w][0]; v[1] += o[w][1]; v[2] += o[w][2]; v[3] += o[w][3]; }
      const int mt = f / NT, t = f - mt * NT;
      const int64_t n = n0 + g * 4 * NT + t * 4;
      if (mrow + mt * 16 < p.M) gemm_store4(p, mrow + mt * 16, n, v, vec && n + 3 < p.N);
    }
  }
  if constexpr (MX) {
    if (inf) {
#pragma clang loop unroll(disable)
      for (int f = wk * 4; f < MT * NT * 4; f += f % 4 == 3 ? 4 * WK - 3 : 1) {   // the columns this wave stored
        const int m = mrow + f / (4 * NT) * 16;
        const int64_t n = n0 + g * 4 * NT + f % (4 * NT);
        if (m < p.M && n < p.N) gemm_inf_fix(p, m, n);
      }
    }
  }
}

// Scale bytes of a weight row.
template <class F> constexpr int gemm_scale_row(int K) { return GemmUnit<F>::UB * K / kGemmKB; }

template <int MT_, int NT_, int WN_, int WK_, int D_> struct GemmCfg {
  static constexpr int MT = MT_, NT = NT_, WN = WN_, WK = WK_, D = D_;
};

template <class F, class C>
bool launch_gemm_cfg(const GemvLaunch& p, hipStream_t st) {
  using S = GemmShape<F, C::MT, C::NT, C::WN, C::WK, C::D>;
  static_assert(C::WN == 1 || C::D >= 2, "a shared ring needs a buffer ahead");
  static_assert(S::XI * C::WN == 4 * C::MT, "activation loads divide over the waves");
  auto kern = gemm_kernel<F, C::MT, C::NT, C::WN, C::WK, C::D>;
  if constexpr (S::LDS > 64 * 1024) {
    static bool attr_set = false;
    if (!attr_set) {
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                              S::LDS) != hipSuccess) {
        (void)hipGetLastError();                           // not the next launch's error
        return false;
      }
      attr_set = true;
    }
  }
  const int mtiles = (p.M + S::BM - 1) / S::BM, ntiles = (p.N + S::BN - 1) / S::BN;
  const int total = mtiles * ntiles, grid = (total + 7) / 8 * 8;
  const int odd = (int64_t)p.N * gemm_scale_row<F>(p.pa.K) % 4 != 0;
  // four columns per store where every output row starts at a multiple of them
  const int vec = p.out_stride % 4 == 0 &&
                  (reinterpret_cast<uintptr_t>(p.out) & (p.out_dtype == DT_F32 ? 15 : 7)) == 0;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(S::THREADS), S::LDS, st, p, mtiles, ntiles, vec, odd);
  return true;
}

// Estimated us of a call with tile shape C, good enough to choose by: over 450
// calls (MXFP8, W8, W6, NVFP4 and bf16, 9 matrices from [96 x 2560] to [16384 x
// 2560], 10 row counts from 17 to 256, weights from HBM) the shape that it
// chooses takes 1.01 times the fastest one's time on (geometric) average and
// 1.12 times at worst.  The busiest CU's workgroups run in rounds of as many as
// its LDS holds; a step costs the longer of a memory round trip over the stages
// in flight and the stage's bytes, then the MFMAs and the decoding; the five
// constants are a fit to timings of 20 tile shapes.
template <class F, class C>
float gemm_cost(const GemvLaunch& p, int cus) {
  using S = GemmShape<F, C::MT, C::NT, C::WN, C::WK, C::D>;
  constexpr int waves = C::WN * C::WK;
  constexpr int fit = 160 * 1024 / S::LDS, lim = waves > 8 ? 2 : 4, resident = fit < lim ? fit : lim;
  const int64_t tiles = (int64_t)((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
  const int64_t per = (tiles + cus - 1) / cus, act = per < resident ? per : resident, rounds = (per + act - 1) / act;
  const int steps = ((p.pa.K + kGemmKB - 1) / kGemmKB + C::WK - 1) / C::WK;
  constexpr int ahead = C::WN > 1 ? C::D - 1 : C::D < 3 ? C::D : 3;
  const float mfma = C::MT * C::NT * waves * (16 / 2400.0f);                       // us per SIMD and step
  const float deq = GemmUnit<F>::DEQ * 32 * C::NT * waves / 2400.0f;
  const float load = act * (S::STAGE / 1000.0f) * 0.00958f, trip = 0.2436f / ahead;
  return rounds * (1.27f + steps * ((trip > load ? trip : load) + act * (3.344f * mfma + 0.485f * deq)));
}

struct GemmChoice {
  float cost = 3.0e38f;
  bool (*fn)(const GemvLaunch&, hipStream_t) = nullptr;
};
template <class F, class... Cs>
GemmChoice gemm_choose(const GemvLaunch& p, int cus) {
  GemmChoice best;
  auto look = [&](float cost, bool (*fn)(const GemvLaunch&, hipStream_t)) {
    if (cost < best.cost) {
      best.cost = cost;
      best.fn = fn;
    }
  };
  (look(gemm_cost<F, Cs>(p, cus), &launch_gemm_cfg<F, Cs>), ...);
  return best;
}

// Launches the call (ksplit is only a shape precondition here) when the
// kernel can take it: whole 128-byte weight rows' alignment as checked below,
// offsets within a tile in 32 bits, the scale plane in whole dwords from its
// start (its last two bytes apart).  False, and nothing launched, otherwise.
template <class F>
bool launch_gemm(const GemvLaunch& p, hipStream_t st) {
  // a switch that sends the format's calls to the core turns this kernel off too
  const Switches& sw = switches();
  if (!sw.gemm || !sw.rows || !GemmUnit<F>::on(sw) || p.M < 1 || p.N < 1) return false;
  auto al = [](const void* q, int n) { return (reinterpret_cast<uintptr_t>(q) & (uintptr_t)(n - 1)) == 0; };
  const int K = p.pa.K;
  if (!al(p.x, 16) || p.x_stride % 8 || !al(p.pa.w0, 16)) return false;
  if (K > 1 << 20 || p.x_stride > 1 << 23) return false;
  if (GemmUnit<F>::KMULT > 16 && K % GemmUnit<F>::KMULT) return false;
  if (GemmUnit<F>::UB) {
    if (!al(p.pa.s, 4) || (int64_t)p.N * gemm_scale_row<F>(K) < 4) return false;
  }
  if (p.pa.w1 && !al(p.pa.w1, 16)) return false;
  const GemmChoice c =
      gemm_choose<F, GemmCfg<1, 1, 1, 8, 1>, GemmCfg<1, 1, 1, 10, 2>, GemmCfg<1, 2, 1, 8, 1>, GemmCfg<2, 1, 1, 8, 1>,
                  GemmCfg<2, 2, 1, 8, 1>, GemmCfg<2, 1, 4, 2, 3>, GemmCfg<3, 1, 4, 2, 2>, GemmCfg<3, 1, 2, 4, 2>,
                  GemmCfg<4, 1, 4, 2, 2>, GemmCfg<4, 1, 8, 1, 2>, GemmCfg<8, 1, 8, 1, 2>>(p, device_cus());
  return c.fn(p, st);
}

// Matrices under half a tile per CU that the few-rows kernels leave (over 4
// rows per CU, or rows too long for them): this kernel rather than the core at
// M > 8, but for short rows at M > 12, also for calls with a K split.
inline bool gemm_small(const GemvLaunch& p) {
  const int tiles = (p.N + 15) / 16;
  return tiles * 2 < device_cus() && p.M > (p.pa.K < 2048 ? 12 : 8) && (p.ksplit == 1 || p.pa.K <= 4096);
}

// Those of the few-rows kernels' shapes that this kernel takes first: from M
// on by format and K, since its time goes up in steps of its K parts and hardly
// with M, and theirs with K and M.  us with weights from HBM (graph replays of
// up to 64 matrices, 1 GB read before each), few-rows kernel / this, [512 x K]
// at M = 9, 13 and 16:
//   K       1088                             2560                             6144
//   NVFP4   4.8 / 4.3  5.0 / 4.3  5.2 / 4.4  5.5 / 5.2  6.0 / 5.3  6.2 / 5.7  7.8 / 8.4  8.8 / 8.5  9.5 / 8.6
//   W6      4.8 / 4.6  5.1 / 4.7  5.3 / 4.8  5.6 / 5.9  6.1 / 6.3  6.3 / 6.4  8.1 / 9.5  9.1 / 9.6  9.8 / 9.7
//   W8      4.5 / 4.5  4.7 / 4.6  4.9 / 4.7  5.5 / 5.5  5.9 / 5.8  6.1 / 6.0  8.1 / 9.2  9.0 / 9.3  9.6 / 9.4
//   MXFP8   4.5 / 4.6  4.7 / 4.7  4.9 / 4.8  5.5 / 5.4  5.8 / 5.7  6.1 / 6.0  7.9 / 9.2  8.9 / 9.3  9.5 / 9.5
//   bf16    4.6 / 4.6  4.8 / 4.8  5.0 / 4.8  5.5 / 5.8  5.9 / 6.0  6.2 / 6.2  8.0 / 9.0  9.1 / 9.4  9.7 / 9.7
// Over 16 K from 512 to 8192, N = 96, 512 and 1000 and M from 9 to 16 these
// lines cost 0.8-1.4% against the better of the two on average and 10% at worst
// (14% for NVFP4 below K = 2048 at 9 to 12 rows).
inline bool gemm_before_rows(const GemvLaunch& p, int fmt) {
  const int K = p.pa.K;
  const int above = fmt == FP4X_FMT_NV4   ? K < 2048 ? 12 : K < 4096 ? 8 : 10
                    : K >= 4096           ? 14
                    : K >= 2048           ? 10
                    : fmt == FP4X_FMT_MX8 ? 16
                                          : 12;
  return gemm_small(p) && p.M > above;
}

}  // namespace fp4x
