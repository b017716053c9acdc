// The fast-numerics matvec over many positions on the f32 matrix cores, bit for bit the
// decode step's (the f32 core of device_common.h).
//
// v_mfma_f32_32x32x2f32 evaluates D = C + A B over its two k as ascending fused multiply-adds,
// each rounded to nearest even, subnormals kept: with C carried from one to the next, a run of
// them is the same chain fma(w, x, acc) the f32 core runs per lane, in the same order. So a
// chunk's partial sums come from the matrix cores, and what the f32 core does between chunks (the
// biased code's correction, the int4 scale, the sums over a lane's chunks, the butterfly over the
// team, a balanced tree over the lanes in order) is done on the accumulators in its order: every
// output has the bits of launch_matvec_f32's tiles and of a decode step.
//
// Bound: the f32 matrix rate (140 TFLOP/s in a large product on this card). A block takes 64
// positions x 64 rows, four waves of 32 x 32; a slab of 64 columns per "slot group" (consecutive
// lanes of the decode team, so consecutive chunks) is staged in LDS while the previous one is
// contracted: activations as f32 with their chunk sums, weights as stored (converted in
// registers: a conversion feeds 32 positions). The tree's pending subtrees stay in registers.
#include <algorithm>

#include "device_common.h"

namespace qh {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kChainM = 64;                 // positions per block
constexpr int kChainN = 64;                 // rows per block
constexpr int kChainK = 64;                 // columns per slab
constexpr int kChainXRow = kChainK + 4;     // staged floats per position: the pad spreads rows over the banks

template <int FMT>
struct ChainFmt {
  static constexpr int kW = Fmt<FMT>::kW;
  static constexpr int kS = kChainK / kW;                  // slots (decode lanes) per slab
  static constexpr int kWBytes = 16 * kS;                  // weight bytes of a row in a slab
  static constexpr int kWRow = kWBytes + 16;               // staged, padded against bank conflicts
  static constexpr int kPieces = kChainN * kS;             // 16-byte pieces of a weight slab
  static constexpr int kPer = (kPieces + kBlock - 1) / kBlock;
  static constexpr int kLevels = FMT == QH_FMT_F16 ? 3 : FMT == QH_FMT_INT8 ? 4 : 5;  // log2(64 / kS)
};

struct ChainArgs {
  DMat m;
  const float* x;     // [seq][cols]
  const float* bias;  // [rows] or null
  float* y;           // [seq][rows]; with several splits [splits][seq][rows] roots without scale or bias
  int seq, tl, slots; // decode team width; slots per split (blockIdx.z), a power of two
};

template <int FMT>
struct ChainLds {
  float x[kChainM * kChainXRow];
  float sx[ChainFmt<FMT>::kS][kChainM];
  float sz[FMT == QH_FMT_INT4 ? kChainN * 2 * ChainFmt<FMT>::kS : 4];
  __attribute__((aligned(16))) uint8_t w[kChainN * ChainFmt<FMT>::kWRow];
};

// A slab's loads, in flight in registers while the previous slab is contracted.
template <int FMT>
struct ChainRegs {
  v4f x[4];
  v4u w[ChainFmt<FMT>::kPer];
  float s, z;
};

// Loads of the slab whose first chunk is c0. Indices are clamped into the matrix: rows,
// positions and chunks past the end are staged but never summed or stored.
template <int FMT>
__device__ __forceinline__ void chain_load(const ChainArgs& a, int row0, int pos0, int c0, ChainRegs<FMT>& r) {
  using F = ChainFmt<FMT>;
  const int t = threadIdx.x;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int i = t + j * kBlock, p = min(pos0 + i / 16, a.seq - 1);
    const int col = min(c0 * F::kW + 4 * (i & 15), a.m.cols - 4);
    r.x[j] = *reinterpret_cast<const v4f*>(a.x + (size_t)p * a.m.cols + col);
  }
#pragma unroll
  for (int j = 0; j < F::kPer; j++) {
    const int i = (F::kPieces % kBlock) ? min(t + j * kBlock, F::kPieces - 1) : t + j * kBlock;
    const int row = min(row0 + i / F::kS, a.m.rows - 1), c = min(c0 + i % F::kS, a.m.nchunks - 1);
    r.w[j] = *reinterpret_cast<const v4u*>(a.m.data + (size_t)row * a.m.row_bytes + 16 * (size_t)c);
  }
  if constexpr (FMT == QH_FMT_INT4) {
    const int i = min(t, kChainN * F::kS - 1);
    const int row = min(row0 + i / F::kS, a.m.rows - 1), c = min(c0 + i % F::kS, a.m.nchunks - 1);
    r.s = a.m.scales[(size_t)row * a.m.gpr + c / a.m.cpg];
    r.z = a.m.zeros[(size_t)row * a.m.gpr + c / a.m.cpg];
  }
}

// Stores a loaded slab. Within each 8 columns the two half-waves' operands (lane l / 32 holds
// k = l / 32 of each instruction) are made contiguous, so a lane reads four instructions' A
// operands with one ds_read_b128: f16 and int8 [0 2 4 6 | 1 3 5 7]; int4, whose even and odd
// elements are separate chains, [0 1 4 5 | 2 3 6 7].
template <int FMT>
__device__ __forceinline__ void chain_store(const ChainRegs<FMT>& r, ChainLds<FMT>& l) {
  using F = ChainFmt<FMT>;
  const int t = threadIdx.x;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const int i = t + j * kBlock, p = i / 16, q = i & 15;
    const v4f v = r.x[j];
    float* d = l.x + p * kChainXRow + 8 * (q >> 1) + 2 * (q & 1);
    if constexpr (FMT == QH_FMT_INT4) {
      *reinterpret_cast<float2*>(d) = float2{v.x, v.y};
      *reinterpret_cast<float2*>(d + 4) = float2{v.z, v.w};
    } else {
      *reinterpret_cast<float2*>(d) = float2{v.x, v.z};
      *reinterpret_cast<float2*>(d + 4) = float2{v.y, v.w};
    }
    if constexpr (FMT != QH_FMT_F16) {
      constexpr int G = F::kW / 4;  // consecutive lanes per chunk: the staging's own chunk sum
      const float s4 = chunk_group_sum<G>((v.x + v.y) + (v.z + v.w));
      if ((q & (G - 1)) == 0) l.sx[q / G][p] = s4;
    }
  }
#pragma unroll
  for (int j = 0; j < F::kPer; j++) {
    const int i = t + j * kBlock;
    if (F::kPieces % kBlock == 0 || i < F::kPieces)
      *reinterpret_cast<v4u*>(l.w + (i / F::kS) * F::kWRow + 16 * (i % F::kS)) = r.w[j];
  }
  if constexpr (FMT == QH_FMT_INT4) {
    if (t < kChainN * F::kS) *reinterpret_cast<float2*>(l.sz + 2 * t) = float2{r.s, r.z};
  }
}

__device__ __forceinline__ f32x16 chain_mfma(float x, float w, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, c, 0, 0, 0);
}

// acc (+)= chunk ci of the staged slab for this wave's 32 positions x 32 rows. Accumulator
// register r holds position 8 (r / 4) + 4 (lane / 32) + r % 4, row lane % 32.
template <int FMT>
__device__ __forceinline__ void chain_chunk(const ChainLds<FMT>& l, int ci, int wp, int wr, f32x16& acc) {
  using F = ChainFmt<FMT>;
  const int n = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  const float* xp = l.x + (32 * wp + n) * kChainXRow + ci * F::kW + 4 * h;
  const v4u w = *reinterpret_cast<const v4u*>(l.w + (32 * wr + n) * F::kWRow + 16 * ci);
  v4f xg[F::kW / 8];
#pragma unroll
  for (int g = 0; g < F::kW / 8; g++) xg[g] = *reinterpret_cast<const v4f*>(xp + 8 * g);
  if constexpr (FMT == QH_FMT_F16) {
#pragma unroll
    for (int k = 0; k < 4; k++) acc = chain_mfma(xg[0][k], f16_lo(w[k] >> (16 * h)), acc);
  } else {
    v4f sx[4];
#pragma unroll
    for (int i = 0; i < 4; i++) sx[i] = *reinterpret_cast<const v4f*>(&l.sx[ci][32 * wp + 8 * i + 4 * h]);
    if constexpr (FMT == QH_FMT_INT8) {
      f32x16 d;
#pragma unroll
      for (int r = 0; r < 16; r++) d[r] = -128.f * sx[r / 4][r % 4];  // exact
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t t = (w[k] ^ 0x80808080u) >> (8 * h);  // q + 128: elements 4k + h and 4k + 2 + h
        d = chain_mfma(xg[k >> 1][2 * (k & 1)], ubyte<0>(t), d);
        d = chain_mfma(xg[k >> 1][2 * (k & 1) + 1], ubyte<2>(t), d);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] += d[r];
    } else {
      const float2 sz = *reinterpret_cast<const float2*>(l.sz + 2 * ((32 * wr + n) * F::kS + ci));
      f32x16 pe, po;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        pe[r] = mul_rounded(-sz.y, sx[r / 4][r % 4]) * 0x1p-24f;
        po[r] = 0.f;
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const uint32_t t = w[k] >> (8 * h);  // bytes 0 and 2: element pairs 8k + 2h and 8k + 4 + 2h
        const uint32_t m0 = t & 0x000F000Fu, m1 = t & 0x00F000F0u;
        pe = chain_mfma(xg[k].x, f16_lo(m0), pe);
        po = chain_mfma(xg[k].y, f16_lo(m1), po);
        pe = chain_mfma(xg[k].z, f16_hi(m0), pe);
        po = chain_mfma(xg[k].w, f16_hi(m1), po);
      }
#pragma unroll
      for (int r = 0; r < 16; r++) acc[r] = fmaf(sz.x * 0x1p24f, fmaf(po[r], 0.0625f, pe[r]), acc[r]);
    }
  }
}

// grid (row blocks, position blocks, splits): split z takes slots z * a.slots .. of the team.
template <int FMT>
__global__ __launch_bounds__(kBlock, 2) void k_chain_f32(ChainArgs a) {
  using F = ChainFmt<FMT>;
  __shared__ __attribute__((aligned(16))) ChainLds<FMT> lds[2];
  const int row0 = blockIdx.x * kChainN, pos0 = blockIdx.y * kChainM;
  const int wave = threadIdx.x / kWave, wp = wave >> 1, wr = wave & 1;
  const int n = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  const int first = blockIdx.z * a.slots, nc = a.m.nchunks;
  const int groups = a.slots / F::kS;
  // Slabs in the order they are summed: group by group, a lane's chunks (tl apart) within it.
  auto slabs_of = [&](int g) {
    const int c = first + g * F::kS;
    return c < nc ? (nc - 1 - c) / a.tl + 1 : 0;
  };
  const bool active = pos0 + 32 * wp < a.seq && row0 + 32 * wr < a.m.rows;  // wave-uniform

  f32x16 st[F::kLevels], root;
  ChainRegs<FMT> regs;
  int cur = 0;
  if (slabs_of(0) > 0) {
    chain_load<FMT>(a, row0, pos0, first, regs);
    chain_store<FMT>(regs, lds[0]);
    __syncthreads();
  }
  for (int g = 0; g < groups; g++) {
    f32x16 acc[F::kS];
#pragma unroll
    for (int i = 0; i < F::kS; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
    const int ns = slabs_of(g);
    for (int j = 0; j < ns; j++) {
      const int c0 = first + g * F::kS + j * a.tl;
      // The next slab's chunk: the group's next, else the next group's first, if it has any.
      const int cn = j + 1 < ns ? c0 + a.tl : first + (g + 1) * F::kS;
      const bool more = j + 1 < ns || (g + 1 < groups && slabs_of(g + 1) > 0);
      if (more) chain_load<FMT>(a, row0, pos0, cn, regs);
      if (active) {
#pragma unroll
        for (int i = 0; i < F::kS; i++)
          if (c0 + i < nc) chain_chunk<FMT>(lds[cur], i, wp, wr, acc[i]);
      }
      if (more) chain_store<FMT>(regs, lds[cur ^ 1]);
      __syncthreads();
      cur ^= 1;
    }
    // The butterfly over the team's lanes: a balanced tree in lane order.
#pragma unroll
    for (int w = 1; w < F::kS; w *= 2)
#pragma unroll
      for (int i = 0; i < F::kS; i += 2 * w) acc[i] += acc[i + w];
    root = acc[0];
    bool open = true;
#pragma unroll
    for (int lv = 0; lv < F::kLevels; lv++) {
      if (open) {
        if (g >> lv & 1) root = st[lv] + root;
        else {
          st[lv] = root;
          open = false;
        }
      }
    }
  }
  if (!active) return;
  const int row = row0 + 32 * wr + n;
  if (row >= a.m.rows) return;
  const bool whole = gridDim.z == 1;
  const float srow = FMT == QH_FMT_INT8 && whole ? a.m.scales[row] : 1.f;
  const float b = whole && a.bias ? a.bias[row] : 0.f;
  float* y = a.y + (size_t)blockIdx.z * a.seq * a.m.rows + row;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    const int p = pos0 + 32 * wp + 8 * (r / 4) + 4 * h + r % 4;
    if (p < a.seq) {
      float v = root[r];
      if (whole) {
        v = row_out_f32<FMT>(v, srow);
        if (a.bias) v = __fadd_rn(v, b);
      }
      y[(size_t)p * a.m.rows] = v;
    }
  }
}

// y[p][r] = the balanced tree over the splits' roots, then the row scale and the bias.
template <int FMT>
__global__ __launch_bounds__(kBlock) void k_chain_finish(const float* __restrict__ part, int splits, size_t plane,
                                                         int rows, const float* __restrict__ scales,
                                                         const float* __restrict__ bias, float* __restrict__ y) {
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= plane) return;
  const int r = (int)(i % rows);
  float v = split_tree(part + i, plane, splits);
  if constexpr (FMT == QH_FMT_INT8) v = row_out_f32<FMT>(v, scales[r]);
  y[i] = bias ? __fadd_rn(v, bias[r]) : v;
}

// Splits of the team's slots over blocks: enough that the chip holds about three blocks per CU.
// A split is a whole subtree of the butterfly, so the splits' roots meet in the same tree.
static int chain_splits(const DMat& m, int seq) {
  const int kS = kChainK / weights_per_chunk(m.format), tl = team_width(m.nchunks);
  const long blocks = (long)((m.rows + kChainN - 1) / kChainN) * ((seq + kChainM - 1) / kChainM);
  int splits = 1;
  while (splits < kChainMaxSplits && blocks * splits < 512 && tl / (2 * splits) >= 2 * kS &&
         m.nchunks > tl - tl / (2 * splits))
    splits *= 2;
  return splits;
}

size_t chain_partials_bytes(const DMat& m, int seq) {
  const int s = chain_splits(m, seq);
  return s > 1 ? (size_t)s * seq * m.rows * sizeof(float) : 0;
}

// Splitting stops at 512 blocks, so the roots stay below 1024 tiles.
size_t chain_partials_bound(const DMat& m, int P) {
  return sizeof(float) * std::min((size_t)kChainMaxSplits * P * m.rows, (size_t)1024 * kChainM * kChainN);
}

template <int FMT>
static hipError_t chain_fmt(hipStream_t s, const ChainArgs& a0, float* part, int splits) {
  ChainArgs a = a0;
  float* y = a.y;
  if (splits > 1) a.y = part;
  a.slots = a.tl / splits;
  const dim3 grid((a.m.rows + kChainN - 1) / kChainN, (a.seq + kChainM - 1) / kChainM, splits);
  hipLaunchKernelGGL(k_chain_f32<FMT>, grid, dim3(kBlock), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  const size_t plane = (size_t)a.seq * a.m.rows;
  hipLaunchKernelGGL(k_chain_finish<FMT>, dim3((unsigned)((plane + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, part,
                     splits, plane, a.m.rows, a.m.scales, a.bias, y);
  return hipGetLastError();
}

hipError_t launch_chain_f32(hipStream_t s, const DMat& m, const float* x, const float* bias, float* y, int seq,
                            float* part, size_t part_bytes) {
  if (chain_partials_bytes(m, seq) > part_bytes) return hipErrorInvalidValue;
  ChainArgs a{};
  a.m = m;
  a.x = x;
  a.bias = bias;
  a.y = y;
  a.seq = seq;
  a.tl = team_width(m.nchunks);
  const int splits = chain_splits(m, seq);
  switch (m.format) {
    case QH_FMT_F16: return chain_fmt<QH_FMT_F16>(s, a, part, splits);
    case QH_FMT_INT8: return chain_fmt<QH_FMT_INT8>(s, a, part, splits);
    default: return chain_fmt<QH_FMT_INT4>(s, a, part, splits);
  }
}

}  // namespace qh
