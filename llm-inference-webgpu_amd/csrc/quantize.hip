// The loader's per-tensor conversion (GpuModel.load, src/gpu/model.js:147-207) on the
// device: checkpoint values (bf16 bits, widened exactly, or f32) quantized with the
// reference quantizer's arithmetic (src/core/quantize.js:36-132) or narrowed to f16
// (src/core/dtype.js:81-113). The codes, scales and zero points equal the host
// restatement's (qh_quantize_int8 / qh_quantize_int4 in host.cpp) bit for bit: the same
// f64 expressions -- the peak or the group range, scale = peak/127 or (hi-lo)/15, the
// inverse of the f64 scale, round half away from zero, Math.min/Math.max semantics for
// NaN and signed zeros -- evaluated per element; only the max/min reductions run in
// parallel, and they are order-free (the maximum of a set, NaN skipped as the host's
// `v > peak` skips it).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "qh_internal.h"

namespace qh {

namespace {

constexpr int kQBlock = 256;

__device__ __forceinline__ double js_min(double a, double b) {
  if (a != a || b != b) return NAN;
  if (a == 0 && b == 0) return (signbit(a) || signbit(b)) ? -0.0 : 0.0;
  return a < b ? a : b;
}
__device__ __forceinline__ double js_max(double a, double b) {
  if (a != a || b != b) return NAN;
  if (a == 0 && b == 0) return (signbit(a) && signbit(b)) ? -0.0 : 0.0;
  return a > b ? a : b;
}
// A typed-array store of a Number: NaN becomes 0.
__device__ __forceinline__ int store_int(double v) { return v != v ? 0 : (int)v; }

template <bool BF16>
__device__ __forceinline__ float src_at(const void* src, size_t i) {
  if constexpr (BF16) return __uint_as_float((uint32_t)static_cast<const uint16_t*>(src)[i] << 16);
  else return static_cast<const float*>(src)[i];
}

// The larger of two candidates as `if (v > best) best = v` keeps it: NaN never wins.
__device__ __forceinline__ double keep_max(double best, double v) { return v > best ? v : best; }
__device__ __forceinline__ double keep_min(double best, double v) { return v < best ? v : best; }

template <typename F>
__device__ __forceinline__ double wave_reduce(double v, F f) {
  for (int off = 32; off > 0; off >>= 1) v = f(v, __shfl_xor(v, off));
  return v;
}

// src/core/quantize.js:36-58, one block per row.
template <bool BF16>
__global__ __launch_bounds__(kQBlock) void k_quant_int8(const void* __restrict__ src, int cols,
                                                        int8_t* __restrict__ q, float* __restrict__ scales) {
  __shared__ double red[kQBlock / 64];
  const int r = blockIdx.x;
  const size_t base = (size_t)r * cols;
  double peak = 0;
  for (int c = threadIdx.x; c < cols; c += kQBlock) peak = keep_max(peak, fabs((double)src_at<BF16>(src, base + c)));
  peak = wave_reduce(peak, keep_max);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = peak;
  __syncthreads();
  peak = 0;
  for (int w = 0; w < kQBlock / 64; w++) peak = keep_max(peak, red[w]);
  const double scale = peak / 127;
  if (threadIdx.x == 0) scales[r] = (float)scale;
  const double inverse = 1 / scale;
  for (int c = threadIdx.x; c < cols; c += kQBlock) {
    int8_t code = 0;
    if (scale != 0) {
      code = (int8_t)store_int(js_max(-127, js_min(127, round((double)src_at<BF16>(src, base + c) * inverse))));
    }
    q[base + c] = code;
  }
}

// src/core/quantize.js:80-132, one wave per (row, group); an even group, so the two
// codes of a byte are in the same group: lane l packs elements 2p, 2p+1 of pair p.
template <bool BF16>
__global__ __launch_bounds__(kQBlock) void k_quant_int4(const void* __restrict__ src, int rows, int cols, int group,
                                                        uint8_t* __restrict__ q, float* __restrict__ scales,
                                                        float* __restrict__ zeros) {
  const int gpr = cols / group;
  const size_t item = (size_t)blockIdx.x * (kQBlock / 64) + (threadIdx.x >> 6);
  if (item >= (size_t)rows * gpr) return;
  const int lane = threadIdx.x & 63;
  const size_t base = (item / gpr) * (size_t)cols + (item % gpr) * (size_t)group;
  double lo = INFINITY, hi = -INFINITY;
  for (int i = lane; i < group; i += 64) {
    const double v = src_at<BF16>(src, base + i);
    lo = keep_min(lo, v);
    hi = keep_max(hi, v);
  }
  lo = wave_reduce(lo, keep_min);
  hi = wave_reduce(hi, keep_max);
  lo = js_min(lo, 0);
  hi = js_max(hi, 0);
  const double scale = (hi - lo) / 15;
  const double zero = scale == 0 ? 0.0 : js_max(0, js_min(15, round(-lo / scale)));
  if (lane == 0) {
    scales[item] = (float)scale;
    zeros[item] = (float)zero;
  }
  const double inverse = 1 / scale;
  for (int p = lane; p < group / 2; p += 64) {
    uint32_t code[2] = {0, 0};
    if (scale != 0) {
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const double level =
            js_max(0, js_min(15, round((double)src_at<BF16>(src, base + 2 * p + k) * inverse) + zero));
        code[k] = (uint32_t)store_int(level) & 0xfu;
      }
    }
    q[(base >> 1) + p] = (uint8_t)(code[0] | (code[1] << 4));
  }
}

// ------------------------------------------------------------------ row-per-wave forms
// The kernels above are the general forms. Where a row is a whole number of 16-byte chunks
// (8 bf16 or 4 f32 values) and the buffers are aligned, one wave takes a row: each lane loads
// its chunks (chunk lane + 64k) once into registers, the peak or the group ranges are reduced
// in f32 compare-selects (exact for a maximum or minimum; NaN never taken, as above), and the
// codes come from the held values with the same f64 expressions, written as one store per chunk.

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <bool BF16>
struct Chunk {
  static constexpr int kVals = BF16 ? 8 : 4;
  // Value j (0..kVals-1) of a 16-byte chunk, widened exactly.
  static __device__ __forceinline__ float at(const u32x4& c, int j) {
    const uint32_t w = j < (BF16 ? 2 : 1) ? c.x : j < (BF16 ? 4 : 2) ? c.y : j < (BF16 ? 6 : 3) ? c.z : c.w;
    if constexpr (BF16) return __uint_as_float((j & 1) ? (w & 0xffff0000u) : (w << 16));
    else return __uint_as_float(w);
  }
};

__device__ __forceinline__ float take_max(float best, float v) { return v > best ? v : best; }
__device__ __forceinline__ float take_min(float best, float v) { return v < best ? v : best; }

// round(t), half away from zero, as an int for |t| < 2^31: the integer part and the exact
// remainder t - trunc(t) decide it.
__device__ __forceinline__ int round_away(double t) {
#pragma clang fp contract(off)
  const int i = (int)t;
  const double f = t - (double)i;
  return i + (f >= 0.5 ? 1 : 0) - (f <= -0.5 ? 1 : 0);
}

// The code expressions above, restated in integers. Every product t = x * inverse that is not
// NaN is bounded: |x| <= peak gives |t| <= 127 (1 + 2^-51) for int8, and lo <= x <= hi gives
// |t| <= 15 (1 + 2^-51) for int4 (an infinite x makes the scale infinite, the inverse 0 and t
// NaN). So round(t) fits an int, the clamps are integer clamps, and NaN -- of t, or of an int4
// zero point, which is otherwise an integer in [0, 15] -- is the typed-array store's 0.
// The product is rounded on its own: fused into the remainder's subtraction, a product that
// rounds to a half-integer would be judged by its unrounded value.
__device__ __forceinline__ int code_int8(float x, double inverse) {
#pragma clang fp contract(off)
  const double t = (double)x * inverse;
  if (t != t) return 0;
  return min(max(round_away(t), -127), 127);
}
__device__ __forceinline__ uint32_t code_int4(float x, double inverse, double zero) {
#pragma clang fp contract(off)
  const double t = (double)x * inverse;
  if (t != t || zero != zero) return 0;
  return (uint32_t)min(max(round_away(t) + (int)zero, 0), 15);
}

// The same codes from an f32 product where that is safe. t32 = x * f32(inverse) differs from
// the f64 product t the expressions above round by at most |t| 2^-23 (the two roundings to f32,
// 2^-24 each relative; f32(inverse) is never subnormal: |x| < 2^128 bounds the scale), and
// |t| <= 16 (int4) or 128 (int8). So wherever t32 lies farther than kSafe from every
// half-integer, t rounds half away from zero to the integer nearest t32; nearer a half-integer,
// and for NaN or an infinite t32, the f64 expression decides. The codes are those of the f64
// expressions bit for bit, at a fraction of their arithmetic. int4 of bf16 tests each value, of
// f32 each chunk of four values (65536 x 1792: bf16 76 us by value, 88 by chunk of eight; f32 112
// by value, 105 by chunk).
constexpr float kSafeInt4 = 0x1p-16f;  // > 16 * 2^-23
constexpr float kSafeInt8 = 0x1p-13f;  // > 128 * 2^-23
// The nearest integer to x * inv32, and whether t32 is too near a half-integer (or NaN).
__device__ __forceinline__ float nearest(float x, float inv32, float safe, bool& unsafe) {
#pragma clang fp contract(off)
  const float t = x * inv32;
  const float r = __builtin_rintf(t);
  unsafe |= !(fabsf(t - r) <= 0.5f - safe);
  return r;
}
// Codes of a chunk's four values from value j0 as bytes.
template <bool BF16>
__device__ __forceinline__ uint32_t codes_int8(const u32x4& c, int j0, float inv32, double inverse) {
  uint32_t w = 0;
  bool unsafe = false;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const float r = __builtin_amdgcn_fmed3f(nearest(Chunk<BF16>::at(c, j0 + j), inv32, kSafeInt8, unsafe), -127.f, 127.f);
    w = __builtin_amdgcn_cvt_pk_u8_f32(r + 128.f, j, w);  // an integer in [1, 255]
  }
  w ^= 0x80808080u;
  if (unsafe) {
    w = 0;
    for (int j = 0; j < 4; j++) w |= (uint32_t)(uint8_t)(int8_t)code_int8(Chunk<BF16>::at(c, j0 + j), inverse) << (8 * j);
  }
  return w;
}
// A bf16 chunk's eight codes as nibbles, value 0 lowest; zf: the zero point, an integer in
// [0, 15], or NaN.
__device__ __forceinline__ uint32_t codes_int4_bf16(const u32x4& c, float inv32, double inverse, float zf) {
  uint32_t w = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const float x = Chunk<true>::at(c, j);
    bool unsafe = false;
    const float r = nearest(x, inv32, kSafeInt4, unsafe);
    w |= (unsafe ? code_int4(x, inverse, (double)zf)
                 : (uint32_t)fminf(fmaxf(r + zf, 0.f), 15.f)) << (4 * j);  // small integers: exact
  }
  return w;
}
// An f32 chunk's four codes where `unsafe` stays false, for values without NaN or infinity. The
// zero point is added before rounding (exactly what adding it after gives, farther than kSafeInt4
// from a half-integer: t32 + zf is off by 2^-20 more).
__device__ __forceinline__ uint32_t codes_int4_f32(const u32x4& c, float inv32, float zf, bool& unsafe) {
  uint32_t w = 0;
  float far = 0.f;
#pragma unroll
  for (int j = 0; j < 4; j += 2) {
    const float a = fmaf(Chunk<false>::at(c, j), inv32, zf), b = fmaf(Chunk<false>::at(c, j + 1), inv32, zf);
    const float ra = __builtin_rintf(a), rb = __builtin_rintf(b);
    far = fmaxf(far, fmaxf(fabsf(a - ra), fabsf(b - rb)));
    // an integer in [0, 255]
    w = __builtin_amdgcn_cvt_pk_u8_f32(fmaf(__builtin_amdgcn_fmed3f(rb, 0.f, 15.f), 16.f,
                                            __builtin_amdgcn_fmed3f(ra, 0.f, 15.f)), j / 2, w);
  }
  unsafe |= !(far <= 0.5f - kSafeInt4);
  return w;
}
__device__ __forceinline__ uint32_t codes_int4_f64(const u32x4& c, double inverse, float zf) {
  uint32_t w = 0;
  for (int j = 0; j < 4; j++) w |= code_int4(Chunk<false>::at(c, j), inverse, (double)zf) << (4 * j);
  return w;
}
template <bool BF16>
__device__ __forceinline__ void store_int4(uint8_t* out, int ci, uint32_t w) {
  if constexpr (BF16) *reinterpret_cast<uint32_t*>(out + (size_t)ci * 4) = w;
  else *reinterpret_cast<uint16_t*>(out + (size_t)ci * 2) = (uint16_t)w;
}

// The range of each segment of G lanes' chunks (NaN never taken, as above). bf16: the values as
// order-preserving 16-bit keys, two to a register (a quarter of the f32 compare-selects), unless
// some value is NaN, whose keys lie outside the infinities'.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
typedef short s16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ s16x2 keys_of(uint32_t u) {  // two bf16 bit patterns; its own inverse
  const s16x2 x = __builtin_bit_cast(s16x2, u);
  return x ^ ((x >> 15) & (s16x2){0x7fff, 0x7fff});
}
__device__ __forceinline__ float key_value(short k) {
  const uint16_t u = (uint16_t)(k ^ ((k >> 15) & 0x7fff));
  return __uint_as_float((uint32_t)u << 16);
}
// Returns whether the wave met a NaN.
template <bool BF16>
__device__ __forceinline__ bool segment_range(const u32x4& c, int G, float& lo, float& hi) {
  if constexpr (BF16) {
    s16x2 mx = keys_of(c.x), mn = mx;
#pragma unroll
    for (int j = 1; j < 4; j++) {
      const s16x2 k = keys_of(c[j]);
      mx = __builtin_elementwise_max(mx, k);
      mn = __builtin_elementwise_min(mn, k);
    }
    auto step = [&](auto other) {
      mx = __builtin_elementwise_max(mx, __builtin_bit_cast(s16x2, other(__builtin_bit_cast(uint32_t, mx))));
      mn = __builtin_elementwise_min(mn, __builtin_bit_cast(s16x2, other(__builtin_bit_cast(uint32_t, mn))));
    };
    if (G > 1) step([](uint32_t v) { return dpp_u32<0xB1>(v); });    // quad_perm: lane ^ 1
    if (G > 2) step([](uint32_t v) { return dpp_u32<0x4E>(v); });    // quad_perm: lane ^ 2
    if (G > 4) step([](uint32_t v) { return dpp_u32<0x141>(v); });   // row_half_mirror
    if (G > 8) step([](uint32_t v) { return dpp_u32<0x140>(v); });   // row_mirror
    for (int off = 16; off < G; off <<= 1) step([&](uint32_t v) { return (uint32_t)__shfl_xor((int)v, off); });
    const short top = mx.x > mx.y ? mx.x : mx.y, bottom = mn.x < mn.y ? mn.x : mn.y;
    constexpr short kInf = 0x7f80, kNegInf = (short)0x807f;
    if (!__any(top > kInf || bottom < kNegInf)) {
      lo = key_value(bottom);
      hi = key_value(top);
      return false;
    }
  }
  bool nan = false;
  lo = INFINITY;
  hi = -INFINITY;
#pragma unroll
  for (int j = 0; j < Chunk<BF16>::kVals; j++) {
    const float v = Chunk<BF16>::at(c, j);
    nan |= v != v;
    lo = take_min(lo, v);
    hi = take_max(hi, v);
  }
  for (int off = 1; off < G; off <<= 1) {
    lo = take_min(lo, __shfl_xor(lo, off));
    hi = take_max(hi, __shfl_xor(hi, off));
  }
  return __any(nan);
}

// src/core/quantize.js:36-58, one wave per row, four rows per block; MAXC chunks per lane.
template <bool BF16, int MAXC>
__global__ __launch_bounds__(kQBlock) void k_quant_int8_rows(const void* __restrict__ src, int rows, int cols,
                                                             int8_t* __restrict__ q, float* __restrict__ scales) {
  using C = Chunk<BF16>;
  const int row = blockIdx.x * (kQBlock / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int nchunks = cols / C::kVals;
  const u32x4* in = reinterpret_cast<const u32x4*>(src) + (size_t)row * nchunks;
  u32x4 c[MAXC];
  float peak = 0;
#pragma unroll
  for (int k = 0; k < MAXC; k++) {
    const int ci = lane + 64 * k;
    c[k] = ci < nchunks ? __builtin_nontemporal_load(in + ci) : u32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < C::kVals; j++) peak = take_max(peak, fabsf(C::at(c[k], j)));
  }
  for (int off = 32; off > 0; off >>= 1) peak = take_max(peak, __shfl_xor(peak, off));
  const double scale = (double)peak / 127;
  if (lane == 0) scales[row] = (float)scale;
  const double inverse = 1 / scale;
  const float inv32 = (float)inverse;
  int8_t* out = q + (size_t)row * cols;
#pragma unroll
  for (int k = 0; k < MAXC; k++) {
    const int ci = lane + 64 * k;
    if (ci >= nchunks) break;
    uint32_t w[C::kVals / 4];
#pragma unroll
    for (int j = 0; j < C::kVals; j += 4) w[j / 4] = scale != 0 ? codes_int8<BF16>(c[k], j, inv32, inverse) : 0u;
    if constexpr (BF16) *reinterpret_cast<uint2*>(out + (size_t)ci * 8) = uint2{w[0], w[1]};
    else *reinterpret_cast<uint32_t*>(out + (size_t)ci * 4) = w[0];
  }
}

// src/core/quantize.js:80-132, one wave per R rows of at most 64 groups together: a group is
// G = group / chunk-values consecutive chunks (G a power of two up to 64), so at step k of a row
// lanes [G*i, G*i + G) hold its group (64k + G*i) / G and the range is a segmented reduction over
// those lanes. Each group's f64 parameters (the divisions and Math.min / Math.max of
// src/core/quantize.js:95-104: ~200 instructions, over a third of a one-row wave's work at 7
// groups a row) are worked out once, lane l for group l of the R rows, and handed back by shuffles.
// LG: log2 of G where it is compiled in (128-column groups), else -1.
template <bool BF16, int MAXC, int R, int LG>
__global__ __launch_bounds__(kQBlock) void k_quant_int4_rows(const void* __restrict__ src, int rows, int cols,
                                                             int lg, uint8_t* __restrict__ q,
                                                             float* __restrict__ scales, float* __restrict__ zeros) {
  using C = Chunk<BF16>;
  if constexpr (LG >= 0) lg = LG;
  const int G = 1 << lg;
  const int row0 = (blockIdx.x * (kQBlock / 64) + (threadIdx.x >> 6)) * R;
  if (row0 >= rows) return;
  const int lane = threadIdx.x & 63;
  const int nchunks = cols / C::kVals, gpr = nchunks >> lg;
  const int steps = (nchunks + 63) / 64, lp = 6 - lg;  // 2^lp groups per step: segment s of step k is group (k << lp) + s
  u32x4 c[R][MAXC];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const u32x4* in = reinterpret_cast<const u32x4*>(src) + (size_t)min(row0 + r, rows - 1) * nchunks;
#pragma unroll
    for (int k = 0; k < MAXC; k++) {
      const int ci = lane + 64 * k;
      c[r][k] = ci < nchunks ? __builtin_nontemporal_load(in + ci) : u32x4{0, 0, 0, 0};
    }
  }
  // Lane l collects the range of group l % gpr of row l / gpr.
  int own_row = 0;
#pragma unroll
  for (int r = 1; r <= R; r++) own_row += lane >= r * gpr ? 1 : 0;
  const int own = lane - own_row * gpr;
  const int own_step = own >> lp, from = (own & ((1 << lp) - 1)) << lg;
  uint32_t odd = 0;  // chunks with a NaN somewhere in the wave
  float glo = INFINITY, ghi = -INFINITY;
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int k = 0; k < MAXC; k++) {
      if (MAXC > 2 && k >= steps) continue;  // wave-uniform
      float lo, hi, a, b;
      if (segment_range<BF16>(c[r][k], G, lo, hi)) odd |= 1u << (r * MAXC + k);
      if constexpr (BF16) {  // both are bf16 values: one shuffle
        const uint32_t u = (uint32_t)__shfl((int)((__float_as_uint(lo) >> 16) | __float_as_uint(hi)), from);
        a = __uint_as_float(u << 16);
        b = __uint_as_float(u & 0xffff0000u);
      } else {
        a = __shfl(lo, from);
        b = __shfl(hi, from);
      }
      if (r == own_row && k == own_step) {
        glo = a;
        ghi = b;
      }
    }
  double ginverse = 0;
  float ginv32 = 0.f, gzero = -1.f;  // -1: a zero scale, whose codes are 0
  if (own_row < min(R, rows - row0)) {
    const double dlo = js_min(glo, 0), dhi = js_max(ghi, 0);
    const double scale = (dhi - dlo) / 15;
    const double zero = scale == 0 ? 0.0 : js_max(0, js_min(15, round(-dlo / scale)));
    scales[(size_t)row0 * gpr + lane] = (float)scale;
    zeros[(size_t)row0 * gpr + lane] = (float)zero;
    ginverse = 1 / scale;
    ginv32 = (float)ginverse;
    if (scale != 0) gzero = (float)zero;  // an integer in [0, 15], or NaN
  }
  // An infinite range, or one whose f32 inverse overflows: a chunk's f32 products may be NaN.
  const bool infinite = __any(gzero != -1.f && (ginverse == 0 || ginv32 == INFINITY));
#pragma unroll
  for (int r = 0; r < R; r++) {
    uint8_t* out = q + (size_t)(row0 + r) * (cols / 2);
#pragma unroll
    for (int k = 0; k < MAXC; k++) {
      if (MAXC > 2 && k >= steps) continue;
      const int ci = lane + 64 * k, owner = r * gpr + min(ci >> lg, gpr - 1);  // the chunk's group (clamped past the row)
      const float inv32 = __shfl(ginv32, owner), zf = __shfl(gzero, owner);
      uint32_t w = 0;
      if constexpr (BF16) {
        const double inverse = __shfl(ginverse, owner);
        if (zf != -1.f) w = codes_int4_bf16(c[r][k], inv32, inverse, zf);
      } else {
        bool unsafe = infinite || (odd >> (r * MAXC + k) & 1);
        w = codes_int4_f32(c[r][k], inv32, zf, unsafe);
        if (__any(unsafe)) {  // wave-uniform, for the shuffle
          const double inverse = __shfl(ginverse, owner);
          if (unsafe) w = codes_int4_f64(c[r][k], inverse, zf);
        }
      }
      if (ci < nchunks && row0 + r < rows) store_int4<BF16>(out, ci, zf == -1.f ? 0u : w);
    }
  }
}

// The same for rows of more than 64 groups, one wave per row: every lane works its group's
// parameters out at each step.
template <bool BF16, int MAXC>
__global__ __launch_bounds__(kQBlock) void k_quant_int4_steps(const void* __restrict__ src, int rows, int cols,
                                                              int G, uint8_t* __restrict__ q,
                                                              float* __restrict__ scales, float* __restrict__ zeros) {
  using C = Chunk<BF16>;
  const int row = blockIdx.x * (kQBlock / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int nchunks = cols / C::kVals;
  const int gpr = nchunks / G;
  const u32x4* in = reinterpret_cast<const u32x4*>(src) + (size_t)row * nchunks;
  u32x4 c[MAXC];
#pragma unroll
  for (int k = 0; k < MAXC; k++) {
    const int ci = lane + 64 * k;
    c[k] = ci < nchunks ? __builtin_nontemporal_load(in + ci) : u32x4{0, 0, 0, 0};
  }
  uint8_t* out = q + (size_t)row * (cols / 2);
#pragma unroll
  for (int k = 0; k < MAXC; k++) {
    const int ci = lane + 64 * k;
    if (64 * k >= nchunks) break;   // wave-uniform: the segmented reduction needs every lane
    float lo, hi;
    const bool odd = segment_range<BF16>(c[k], G, lo, hi);
    if (ci >= nchunks) continue;
    const double dlo = js_min(lo, 0), dhi = js_max(hi, 0);
    const double scale = (dhi - dlo) / 15;
    const double zero = scale == 0 ? 0.0 : js_max(0, js_min(15, round(-dlo / scale)));
    if ((lane & (G - 1)) == 0) {
      const size_t gi = (size_t)row * gpr + ci / G;
      scales[gi] = (float)scale;
      zeros[gi] = (float)zero;
    }
    const double inverse = 1 / scale;
    const float inv32 = (float)inverse;
    uint32_t w = 0;
    if constexpr (BF16) {
      if (scale != 0) w = codes_int4_bf16(c[k], inv32, inverse, (float)zero);
    } else {
      bool unsafe = odd || inverse == 0 || inv32 == INFINITY;  // f32 products may be NaN
      w = codes_int4_f32(c[k], inv32, (float)zero, unsafe);
      if (unsafe) w = codes_int4_f64(c[k], inverse, (float)zero);
    }
    store_int4<BF16>(out, ci, scale != 0 ? w : 0u);
  }
}

// src/core/dtype.js:81-113: round to nearest even with gradual underflow and overflow to
// infinity, which the hardware conversion does for every number; a NaN keeps its sign and the
// top ten payload bits with the quiet bit set (dtype.js:88-90).
__device__ __forceinline__ uint16_t narrow_f16(float x) {
  const uint32_t u = __float_as_uint(x);
  return x != x ? (uint16_t)(((u >> 16) & 0x8000u) | 0x7c00u | ((u & 0x7fffffu) >> 13) | 0x200u)
                : __builtin_bit_cast(uint16_t, (_Float16)x);
}

template <bool BF16>
__global__ void k_to_f16(const void* __restrict__ src, size_t n, uint16_t* __restrict__ out) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = narrow_f16(src_at<BF16>(src, i));
}

template <bool BF16>
__global__ void k_to_f32(const void* __restrict__ src, size_t n, float* __restrict__ out) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    out[i] = src_at<BF16>(src, i);
}

// Eight values per thread with 16-byte accesses; the n % 8 tail by the first threads.
template <bool BF16, bool F16>
__global__ __launch_bounds__(kQBlock) void k_widen_narrow8(const void* __restrict__ src, size_t n,
                                                           void* __restrict__ out) {
  const size_t n8 = n / 8;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8; i += (size_t)gridDim.x * blockDim.x) {
    float v[8];
    if constexpr (BF16) {
      const u32x4 c = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + i);
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = Chunk<true>::at(c, j);
    } else {
      const u32x4 a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + 2 * i);
      const u32x4 b = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src) + 2 * i + 1);
#pragma unroll
      for (int j = 0; j < 4; j++) v[j] = Chunk<false>::at(a, j), v[4 + j] = Chunk<false>::at(b, j);
    }
    if constexpr (F16) {
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; j++) w[j] = (uint32_t)narrow_f16(v[2 * j]) | ((uint32_t)narrow_f16(v[2 * j + 1]) << 16);
      reinterpret_cast<u32x4*>(out)[i] = u32x4{w[0], w[1], w[2], w[3]};
    } else {
      float4* o = reinterpret_cast<float4*>(out) + 2 * i;
      o[0] = float4{v[0], v[1], v[2], v[3]};
      o[1] = float4{v[4], v[5], v[6], v[7]};
    }
  }
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n - n8 * 8) {
    const float x = src_at<BF16>(src, n8 * 8 + t);
    if constexpr (F16) static_cast<uint16_t*>(out)[n8 * 8 + t] = narrow_f16(x);
    else static_cast<float*>(out)[n8 * 8 + t] = x;
  }
}

unsigned grid_for(size_t n) { return (unsigned)std::min<size_t>((n + kQBlock - 1) / kQBlock, 16384); }

bool aligned(const void* p, size_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; }

// Chunks per lane of the row-per-wave kernels for `nchunks` chunks a row; 0 when too many.
int chunks_per_lane(int nchunks) {
  const int per = (nchunks + 63) / 64;
  return per <= 1 ? 1 : per <= 2 ? 2 : per <= 4 ? 4 : per <= 8 ? 8 : per <= 16 ? 16 : 0;
}

template <bool BF16, int MAXC>
void launch_int8_rows(hipStream_t s, const void* src, int rows, int cols, int8_t* q, float* scales) {
  hipLaunchKernelGGL((k_quant_int8_rows<BF16, MAXC>), dim3((rows + 3) / 4), dim3(kQBlock), 0, s, src, rows, cols, q,
                     scales);
}
// Rows from which a wave takes several: below, the rows after the first only wait for it. bf16 to
// int4, us, one row a wave | four: 896 x 896 3.8 | 7.7, 8192 x 896 8.1 | 9.3, 16384 x 896 14.1 |
// 14.5, 16384 x 512 9.0 | 8.2, 65536 x 896 45.7 | 41.0, 233472 x 896 146 | 126.
constexpr int kSharedRows = 16384;
template <bool BF16, int MAXC, int R>
void launch_int4_rows(hipStream_t s, const void* src, int rows, int cols, int G, uint8_t* q, float* scales,
                      float* zeros) {
  // R rows a wave where there are waves enough without (kSharedRows) and their groups fit the
  // wave's lanes; more than 64 groups a row go step by step.
  const int gpr = cols / Chunk<BF16>::kVals / G;
  const auto blocks = [&](int r) { return dim3((rows + 4 * r - 1) / (4 * r)); };
  int lg = 0;
  while ((1 << lg) < G) lg++;
  constexpr int kLg = BF16 ? 4 : 5;  // chunks of a 128-column group
  if (R > 1 && R * gpr <= 64 && lg == kLg && rows >= kSharedRows)
    hipLaunchKernelGGL((k_quant_int4_rows<BF16, MAXC, R, kLg>), blocks(R), dim3(kQBlock), 0, s, src, rows, cols, lg,
                       q, scales, zeros);
  else if (gpr <= 64 && lg == kLg)
    hipLaunchKernelGGL((k_quant_int4_rows<BF16, MAXC, 1, kLg>), blocks(1), dim3(kQBlock), 0, s, src, rows, cols, lg,
                       q, scales, zeros);
  else if (gpr <= 64)
    hipLaunchKernelGGL((k_quant_int4_rows<BF16, MAXC, 1, -1>), blocks(1), dim3(kQBlock), 0, s, src, rows, cols, lg, q,
                       scales, zeros);
  else
    hipLaunchKernelGGL((k_quant_int4_steps<BF16, MAXC>), blocks(1), dim3(kQBlock), 0, s, src, rows, cols, G, q,
                       scales, zeros);
}

template <bool BF16>
hipError_t convert_t(hipStream_t s, const void* src, int rows, int cols, int format, int group, void* data,
                     float* scales, float* zeros) {
  const size_t n = (size_t)rows * cols;
  constexpr int kVals = Chunk<BF16>::kVals;
  const int nchunks = cols / kVals;
  const bool rows_vec = cols % kVals == 0 && aligned(src, 16);
  const int maxc = rows_vec ? chunks_per_lane(nchunks) : 0;
  switch (format) {
    case QH_FMT_F32:
    case QH_FMT_F16: {
      const bool f16 = format == QH_FMT_F16;
      if (aligned(src, 16) && aligned(data, 16)) {
        const unsigned grid = (unsigned)std::min<size_t>(std::max<size_t>((n / 8 + kQBlock - 1) / kQBlock, 1), 16384);
        if (f16) hipLaunchKernelGGL((k_widen_narrow8<BF16, true>), dim3(grid), dim3(kQBlock), 0, s, src, n, data);
        else hipLaunchKernelGGL((k_widen_narrow8<BF16, false>), dim3(grid), dim3(kQBlock), 0, s, src, n, data);
      } else if (f16) {
        hipLaunchKernelGGL(k_to_f16<BF16>, dim3(grid_for(n)), dim3(kQBlock), 0, s, src, n,
                           static_cast<uint16_t*>(data));
      } else {
        hipLaunchKernelGGL(k_to_f32<BF16>, dim3(grid_for(n)), dim3(kQBlock), 0, s, src, n, static_cast<float*>(data));
      }
      break;
    }
    case QH_FMT_INT8: {
      int8_t* q = static_cast<int8_t*>(data);
      if (maxc && aligned(data, BF16 ? 8 : 4)) {
        if (maxc <= 2) launch_int8_rows<BF16, 2>(s, src, rows, cols, q, scales);
        else if (maxc == 4) launch_int8_rows<BF16, 4>(s, src, rows, cols, q, scales);
        else if (maxc == 8) launch_int8_rows<BF16, 8>(s, src, rows, cols, q, scales);
        else launch_int8_rows<BF16, 16>(s, src, rows, cols, q, scales);
      } else {
        hipLaunchKernelGGL(k_quant_int8<BF16>, dim3(rows), dim3(kQBlock), 0, s, src, cols, q, scales);
      }
      break;
    }
    case QH_FMT_INT4: {
      uint8_t* q = static_cast<uint8_t*>(data);
      const int G = group / kVals;
      if (maxc && group % kVals == 0 && G <= 64 && (G & (G - 1)) == 0 && aligned(data, BF16 ? 4 : 2)) {
        if (maxc == 1) launch_int4_rows<BF16, 1, 4>(s, src, rows, cols, G, q, scales, zeros);
        else if (maxc == 2) launch_int4_rows<BF16, 2, 4>(s, src, rows, cols, G, q, scales, zeros);
        else if (maxc == 4) launch_int4_rows<BF16, 4, 2>(s, src, rows, cols, G, q, scales, zeros);
        else if (maxc == 8) launch_int4_rows<BF16, 8, 1>(s, src, rows, cols, G, q, scales, zeros);
        else launch_int4_rows<BF16, 16, 1>(s, src, rows, cols, G, q, scales, zeros);
      } else {
        const size_t items = (size_t)rows * (cols / group);
        hipLaunchKernelGGL(k_quant_int4<BF16>, dim3((unsigned)((items + 3) / 4)), dim3(kQBlock), 0, s, src, rows,
                           cols, group, q, scales, zeros);
      }
      break;
    }
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_convert(hipStream_t s, bool bf16, const void* src, int rows, int cols, int format, int group,
                          void* data, float* scales, float* zeros) {
  return bf16 ? convert_t<true>(s, src, rows, cols, format, group, data, scales, zeros)
              : convert_t<false>(s, src, rows, cols, format, group, data, scales, zeros);
}

}  // namespace qh
