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
#include <type_traits>

#include "device_common.h"

namespace qh {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kChainM = 64;                 // positions per block
constexpr int kChainN = 64;                 // rows per block

template <int FMT>
struct ChainFmt {
  static constexpr int kW = Fmt<FMT>::kW;
  static constexpr int kS = FMT == QH_FMT_INT4 ? 2 : 4;    // slots (decode lanes) per slab
  static constexpr int kK = kS * kW;                       // columns per slab
  static constexpr int kXRow = kK + 4;                     // staged floats per position: the pad spreads rows over the banks
  static constexpr int kXPer = kChainM * kK / 4 / kBlock;  // float4 loads per thread
  static constexpr int kWBytes = 16 * kS;                  // weight bytes of a row in a slab
  static constexpr int kWRow = kWBytes + 16;               // staged, padded against bank conflicts
  static constexpr int kPieces = kChainN * kS;             // 16-byte pieces of a weight slab
  static constexpr int kPer = (kPieces + kBlock - 1) / kBlock;
  // log2 of the slot groups of one block: 16 at most (chain_splits cuts an int4 team of 64 lanes in
  // two at least), and fewer where lanes sum several chunks: in int8 and int4 those are rows of more
  // than 1024 or 2048 columns, a down projection's at most 1024 of them, cut in four at least.
  static constexpr int kLevels = 4;
  static constexpr int kMultiLevels = FMT == QH_FMT_F16 ? 4 : FMT == QH_FMT_INT8 ? 2 : 3;
};

struct ChainArgs {
  DMat m;
  const float* x;     // [seq][cols]
  const float* bias;  // [rows] or null
  float* y;           // [seq][rows]; with several splits [splits][seq][rows] roots without scale or bias
  int seq, tl;        // positions; decode team width
};

template <int FMT>
struct ChainLds {
  float x[kChainM * ChainFmt<FMT>::kXRow];
  float sx[ChainFmt<FMT>::kS][kChainM];
  float sz[FMT == QH_FMT_INT4 ? kChainN * 2 * ChainFmt<FMT>::kS : 4];
  __attribute__((aligned(16))) uint8_t w[kChainN * ChainFmt<FMT>::kWRow];
};

// A slab's loads, in flight in registers while the previous slab is contracted.
template <int FMT>
struct ChainRegs {
  v4f x[ChainFmt<FMT>::kXPer];
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
  for (int j = 0; j < F::kXPer; j++) {
    const int i = t + j * kBlock, p = min(pos0 + i / (F::kK / 4), a.seq - 1);
    const int col = min(c0 * F::kW + 4 * (i % (F::kK / 4)), a.m.cols - 4);
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
  for (int j = 0; j < F::kXPer; j++) {
    const int i = t + j * kBlock, p = i / (F::kK / 4), q = i % (F::kK / 4);
    const v4f v = r.x[j];
    float* d = l.x + p * F::kXRow + 8 * (q >> 1) + 2 * (q & 1);
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
      if ((q & (G - 1)) == 0) l.sx[q / G][p] = FMT == QH_FMT_INT8 ? -128.f * s4 : s4;  // exact
    }
  }
#pragma unroll
  for (int j = 0; j < F::kPer; j++) {
    const int i = t + j * kBlock;
    const uint32_t flip = FMT == QH_FMT_INT8 ? 0x80808080u : 0u;  // int8: q + 128 in every byte
    if (F::kPieces % kBlock == 0 || i < F::kPieces)
      *reinterpret_cast<v4u*>(l.w + (i / F::kS) * F::kWRow + 16 * (i % F::kS)) = r.w[j] ^ flip;
  }
  if constexpr (FMT == QH_FMT_INT4) {
    if (t < kChainN * F::kS) *reinterpret_cast<float2*>(l.sz + 2 * t) = float2{r.s, r.z};
  }
}

__device__ __forceinline__ f32x16 chain_mfma(float x, float w, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(x, w, c, 0, 0, 0);
}

// One staged chunk's operands in registers for this wave's 32 positions x 32 rows.
template <int FMT>
struct ChainOps {
  v4u w;
  v4f x[ChainFmt<FMT>::kW / 8];
  f32x16 sx;  // the chunk sums of the lane's accumulator positions (int8: times -128)
  float2 sz;  // int4: group scale and zero point of the lane's row
};
template <int FMT>
__device__ __forceinline__ void chain_ops(const ChainLds<FMT>& l, int ci, int wp, int wr, ChainOps<FMT>& o) {
  using F = ChainFmt<FMT>;
  const int n = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  o.w = *reinterpret_cast<const v4u*>(l.w + (32 * wr + n) * F::kWRow + 16 * ci);
  const float* xp = l.x + (32 * wp + n) * F::kXRow + ci * F::kW + 4 * h;
#pragma unroll
  for (int g = 0; g < F::kW / 8; g++) o.x[g] = *reinterpret_cast<const v4f*>(xp + 8 * g);
  if constexpr (FMT != QH_FMT_F16) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const v4f q = *reinterpret_cast<const v4f*>(&l.sx[ci][32 * wp + 8 * i + 4 * h]);
#pragma unroll
      for (int e = 0; e < 4; e++) o.sx[4 * i + e] = q[e];
    }
  }
  if constexpr (FMT == QH_FMT_INT4) o.sz = *reinterpret_cast<const float2*>(l.sz + 2 * ((32 * wr + n) * F::kS + ci));
}

// acc (+)= the chunk. Accumulator register r holds position 8 (r / 4) + 4 (lane / 32) + r % 4,
// row lane % 32. FIRST: the lane's first chunk, acc starting at 0 (an int8 chunk's sum is
// never -0: 0 + d is d).
template <int FMT, bool FIRST>
__device__ __forceinline__ void chain_chunk(ChainOps<FMT>& o, f32x16& acc) {
  const int h = (threadIdx.x >> 5) & 1;
  if constexpr (FIRST && FMT != QH_FMT_INT8) {
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = 0.f;
  }
  if constexpr (FMT == QH_FMT_F16) {
#pragma unroll
    for (int k = 0; k < 4; k++) acc = chain_mfma(o.x[0][k], f16_lo(o.w[k] >> (16 * h)), acc);
  } else if constexpr (FMT == QH_FMT_INT8) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t t = o.w[k] >> (8 * h);  // elements 4k + h and 4k + 2 + h in bytes 0 and 2
      o.sx = chain_mfma(o.x[k >> 1][2 * (k & 1)], ubyte<0>(t), o.sx);
      o.sx = chain_mfma(o.x[k >> 1][2 * (k & 1) + 1], ubyte<2>(t), o.sx);
    }
    if constexpr (FIRST) acc = o.sx;
    else acc += o.sx;
  } else {
    f32x16 pe, po;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      pe[r] = mul_rounded(-o.sz.y, o.sx[r]) * 0x1p-24f;
      po[r] = 0.f;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const uint32_t t = o.w[k] >> (8 * h);  // bytes 0 and 2: element pairs 8k + 2h and 8k + 4 + 2h
      const uint32_t m0 = t & 0x000F000Fu, m1 = t & 0x00F000F0u;
      pe = chain_mfma(o.x[k].x, f16_lo(m0), pe);
      po = chain_mfma(o.x[k].y, f16_lo(m1), po);
      pe = chain_mfma(o.x[k].z, f16_hi(m0), pe);
      po = chain_mfma(o.x[k].w, f16_hi(m1), po);
    }
    const float s = o.sz.x * 0x1p24f;
#pragma unroll
    for (int r = 0; r < 16; r++) acc[r] = fmaf(s, fmaf(po[r], 0.0625f, pe[r]), acc[r]);
  }
}

// The slab whose first chunk is c0 into the group's slot sums. A whole slab is straight-line
// code with each chunk's LDS reads issued before the previous chunk's products.
template <int FMT, bool FIRST>
__device__ __forceinline__ void chain_slab(const ChainLds<FMT>& l, int c0, int nc, int wp, int wr,
                                           f32x16 (&acc)[ChainFmt<FMT>::kS]) {
  constexpr int S = ChainFmt<FMT>::kS;
  ChainOps<FMT> o[2];
  if (c0 + S <= nc) {
    chain_ops<FMT>(l, 0, wp, wr, o[0]);
#pragma unroll
    for (int i = 0; i < S; i++) {
      if (i + 1 < S) chain_ops<FMT>(l, i + 1, wp, wr, o[(i + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      chain_chunk<FMT, FIRST>(o[i & 1], acc[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < S; i++) {
      if (c0 + i < nc) {
        chain_ops<FMT>(l, i, wp, wr, o[0]);
        chain_chunk<FMT, FIRST>(o[0], acc[i]);
      } else if constexpr (FIRST) {
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.f;
      }
    }
  }
}

// grid (row blocks, position blocks, splits): split z takes slots z * a.slots .. of the team,
// 2^LV groups of kS. MULTI: some lane of the team sums more than one chunk.
template <int FMT, int LV, bool MULTI>
__global__ __launch_bounds__(kBlock, 2) void k_chain_f32(ChainArgs a) {
  using F = ChainFmt<FMT>;
  __shared__ __attribute__((aligned(16))) ChainLds<FMT> lds[2];
  const int row0 = blockIdx.x * kChainN, pos0 = blockIdx.y * kChainM;
  const int wave = threadIdx.x / kWave, wp = wave >> 1, wr = wave & 1;
  const int n = threadIdx.x & 31, h = (threadIdx.x >> 5) & 1;
  constexpr int kGroups = 1 << LV;
  const int first = blockIdx.z * (F::kS * kGroups), nc = a.m.nchunks;
  // Slabs in the order they are summed: group by group, a lane's chunks (tl apart) within it.
  auto slabs_of = [&](int g) {
    const int c = first + g * F::kS;
    return c < nc ? (MULTI ? (nc - 1 - c) / a.tl + 1 : 1) : 0;
  };
  const bool active = pos0 + 32 * wp < a.seq && row0 + 32 * wr < a.m.rows;  // wave-uniform

  f32x16 st[LV > 0 ? LV : 1], root;
  ChainRegs<FMT> regs;
  int cur = 0;
  if (slabs_of(0) > 0) {
    chain_load<FMT>(a, row0, pos0, first, regs);
    chain_store<FMT>(regs, lds[0]);
    __syncthreads();
  }
#pragma unroll 1
  for (int g = 0; g < kGroups; g++) {
    f32x16 acc[F::kS];
    const int ns = slabs_of(g);
    if (ns == 0) {
#pragma unroll
      for (int r = 0; r < 16; r++) root[r] = 0.f;
    }
#pragma unroll 1
    for (int j = 0; j < ns; j++) {
      const int c0 = first + g * F::kS + j * a.tl;
      // The next slab's chunk: the group's next, else the next group's first, if it has any.
      const int cn = j + 1 < ns ? c0 + a.tl : first + (g + 1) * F::kS;
      const bool more = j + 1 < ns || (g + 1 < kGroups && slabs_of(g + 1) > 0);
      if (more) chain_load<FMT>(a, row0, pos0, cn, regs);
      if (active) {
        if (!MULTI || j == 0) chain_slab<FMT, true>(lds[cur], c0, nc, wp, wr, acc);
        else chain_slab<FMT, false>(lds[cur], c0, nc, wp, wr, acc);
      }
      if (more) chain_store<FMT>(regs, lds[cur ^ 1]);
      __syncthreads();
      cur ^= 1;
    }
    // The butterfly over the team's lanes: a balanced tree in lane order.
    if (ns > 0) {
#pragma unroll
      for (int w = 1; w < F::kS; w *= 2)
#pragma unroll
        for (int i = 0; i < F::kS; i += 2 * w) acc[i] += acc[i + w];
      root = acc[0];
    }
    bool open = true;
#pragma unroll
    for (int lv = 0; lv < LV; lv++) {
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
__global__ __launch_bounds__(kBlock) void k_chain_finish(ChainOut o, float* __restrict__ y) {
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < (size_t)o.seq * o.rows) y[i] = chain_value(o, i, (int)(i % o.rows));
}

// Splits of the team's slots over blocks: until there are two blocks per CU, which is what the
// registers of nearly every form allow.
// A split is a whole subtree of the butterfly, so the splits' roots meet in the same tree.
static int chain_splits(const DMat& m, int seq) {
  const int kS = m.format == QH_FMT_INT4 ? 2 : 4, tl = team_width(m.nchunks);
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

// A launch's latency and its blocks' slabs one after another, more of them where a CU holds
// several blocks, slower ones where few share the loads. Fitted with matvec_f32_us to prompts of 9 to 512 positions through models of 128
// to 1024 columns and 256 to 8192 ffn rows in every format, and to a head of 151936 rows.
float chain_f32_us(const DMat& m, int seq) {
  const int kS = m.format == QH_FMT_INT4 ? 2 : 4, tl = team_width(m.nchunks), splits = chain_splits(m, seq);
  const int groups = std::min(tl / splits / kS, (std::min(m.nchunks, tl) + kS - 1) / kS);
  const int slabs = groups * ((m.nchunks + tl - 1) / tl);
  const long blocks = (long)((m.rows + kChainN - 1) / kChainN) * ((seq + kChainM - 1) / kChainM) * splits;
  const float slab = m.format == QH_FMT_F16 ? 0.5f : m.format == QH_FMT_INT8 ? 0.9f : 1.3f;
  return 3.5f + slab * slabs * std::max(blocks < 16 ? 1.2f : 1.f, 1.2f * blocks / 256);
}

// False where no form sums that many levels.
template <int FMT, int LV = ChainFmt<FMT>::kLevels>
static bool chain_lv(hipStream_t s, const ChainArgs& a, dim3 grid, int lv) {
  if (lv < LV) {
    if constexpr (LV > 0) return chain_lv<FMT, LV - 1>(s, a, grid, lv);
  }
  if (lv > LV) return false;
  if (a.m.nchunks <= a.tl) {
    hipLaunchKernelGGL((k_chain_f32<FMT, LV, false>), grid, dim3(kBlock), 0, s, a);
    return true;
  }
  if constexpr (LV <= ChainFmt<FMT>::kMultiLevels) {
    hipLaunchKernelGGL((k_chain_f32<FMT, LV, true>), grid, dim3(kBlock), 0, s, a);
    return true;
  }
  return false;
}

hipError_t launch_chain_roots(hipStream_t s, const DMat& m, const float* x, const float* bias, float* y, int seq,
                              float* part, size_t part_bytes, ChainOut* out) {
  if (chain_partials_bytes(m, seq) > part_bytes) return hipErrorInvalidValue;
  const int splits = chain_splits(m, seq);
  ChainArgs a{};
  a.m = m;
  a.x = x;
  a.bias = bias;
  a.y = splits > 1 ? part : y;
  a.seq = seq;
  a.tl = team_width(m.nchunks);
  const dim3 grid((m.rows + kChainN - 1) / kChainN, (seq + kChainM - 1) / kChainM, splits);
  int lv = 0;
  while (((m.format == QH_FMT_INT4 ? 2 : 4) << lv) < a.tl / splits) lv++;
  const bool ok = m.format == QH_FMT_F16    ? chain_lv<QH_FMT_F16>(s, a, grid, lv)
                  : m.format == QH_FMT_INT8 ? chain_lv<QH_FMT_INT8>(s, a, grid, lv)
                                            : chain_lv<QH_FMT_INT4>(s, a, grid, lv);
  if (!ok) return hipErrorInvalidValue;
  *out = ChainOut{a.y, splits, m.rows, seq, splits > 1 && m.format == QH_FMT_INT8 ? m.scales : nullptr,
                  splits > 1 ? bias : nullptr};
  return hipGetLastError();
}

hipError_t launch_chain_f32(hipStream_t s, const DMat& m, const float* x, const float* bias, float* y, int seq,
                            float* part, size_t part_bytes) {
  ChainOut o;
  const hipError_t e = launch_chain_roots(s, m, x, bias, y, seq, part, part_bytes, &o);
  if (e != hipSuccess || o.splits == 1) return e;
  const size_t plane = (size_t)seq * m.rows;
  hipLaunchKernelGGL(k_chain_finish, dim3((unsigned)((plane + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, o, y);
  return hipGetLastError();
}

// --------------------------------------------------------------- f64 order --
// The exact matvec (k_matvec of ops.hip: the loader's f32 weights, f64 sums) over several
// positions on v_mfma_f64_16x16x4f64, whose four k are ascending fused multiply-adds as above:
// the accumulator runs through a lane's chunks, so every output has k_matvec's bits.
//
// Bound: the f64 matrix rate (70 TFLOP/s in a large product), which the vector unit's f64 shares
// with everything else it does; what the VALU form lost was one LDS read of x per two products
// and a dequantized weight per eight positions. A block takes T tiles of 16 positions x 16 rows,
// its four waves a quarter of the team's slots each (so 52 positions of a 4864-row matrix are 608
// blocks of two tiles), joined through LDS in tree order. A wave stages its own slabs of x, so no
// barrier runs in the loop; weights go to registers a chunk ahead. 4864 x 896 int8, 52 positions:
// 90 -> 23 us.
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <int FMT>
struct Chain64 {
  static constexpr int kW = Fmt<FMT>::kW;
  static constexpr int kS = FMT == QH_FMT_INT4 ? 2 : 4;  // slots per slab
  static constexpr int kK = kS * kW;
  static constexpr int kXRow = kK + 4;
  static constexpr int kLevels = FMT == QH_FMT_INT4 ? 3 : 2;  // log2 of a wave's groups, 16 slots at most
};
constexpr int kChain64M = 16, kChain64N = 16;  // a tile's positions and rows

// One chunk of one row as the loader's f32 weights: w(s) is the lane's element 4s + g.
template <int FMT>
struct RowChunk {
  v4u w;
  float s, z;
  int zi;
  bool zint;
  __device__ __forceinline__ void set(v4u w_, float s_, float z_) {
    w = w_;
    s = s_;
    z = z_;
    if constexpr (FMT == QH_FMT_INT4) {
      zi = (int)z_;
      zint = (float)zi == z_ && (unsigned)zi <= 15u;  // what the quantizer writes
    }
  }
  template <int STEP>
  __device__ __forceinline__ double at(int g) const {
    if constexpr (FMT == QH_FMT_F16) {
      const uint32_t d = g < 2 ? w[2 * STEP] : w[2 * STEP + 1];
      return (double)f16_lo(d >> (16 * (g & 1)));
    } else if constexpr (FMT == QH_FMT_INT8) {
      return (double)((float)(int8_t)(uint8_t)(w[STEP] >> (8 * g)) * s);  // q*s is exact before rounding
    } else {
      const int lv = (int)((w[STEP / 2] >> (16 * (STEP & 1) + 4 * g)) & 0xfu);
      if (zint) return (double)((float)(lv - zi) * s);  // exact before rounding
      return (double)(float)(((double)lv - (double)z) * (double)s);
    }
  }
};

// acc[tile] += one chunk for 16 rows x T tiles of 16 positions (`two`: the second has any).
// Accumulator register r holds position 4r + lane / 16, row lane % 16.
template <int FMT, int STEPS, int T, int K = 0>
__device__ __forceinline__ void chain64_steps(const RowChunk<FMT>& rc, const float (&xv)[T][STEPS], int g, bool two,
                                              f64x4 (&acc)[T]) {
  if constexpr (K < STEPS) {
    const double w = rc.template at<K>(g);
    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)xv[0][K], w, acc[0], 0, 0, 0);
    if constexpr (T == 2) {
      if (two) acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)xv[1][K], w, acc[1], 0, 0, 0);
    }
    chain64_steps<FMT, STEPS, T, K + 1>(rc, xv, g, two, acc);
  }
}

template <int FMT, bool MULTI, int T>
__global__ __launch_bounds__(kBlock, 2) void k_chain_f64(ChainArgs a) {
  using F = Chain64<FMT>;
  constexpr int S = F::kS, kLoads = T * kChain64M * F::kK / 4 / kWave;
  // A wave's slab of x (its LDS operations run in order, so the next slab is stored over it after
  // its reads), then its sums [tile][register][lane].
  __shared__ __attribute__((aligned(16))) float xs[kBlock / kWave][T * kChain64M * F::kXRow];
  static_assert(2 * 4 * kWave <= kChain64M * F::kXRow, "the sums fit the slab");
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, n = lane & 15, g4 = lane >> 4;
  const int row0 = blockIdx.x * kChain64N, pos0 = blockIdx.y * (T * kChain64M);
  const int nc = a.m.nchunks, slots = a.tl / (kBlock / kWave), first = wave * slots, groups = slots / S;
  const int row = min(row0 + n, a.m.rows - 1);
  const bool two = T == 2 && pos0 + 16 < a.seq;  // uniform: the second position tile has any
  const v4u* rp = reinterpret_cast<const v4u*>(a.m.data + (size_t)row * a.m.row_bytes);
  const float srow = FMT == QH_FMT_INT8 ? a.m.scales[row] : 0.f;
  auto slabs_of = [&](int g) {
    const int c = first + g * S;
    return c < nc ? (MULTI ? (nc - 1 - c) / a.tl + 1 : 1) : 0;
  };
  // x of a slab: 16 T positions x kK columns, one float4 per lane and load.
  v4f xr[kLoads];
  v4u wr[S];
  float sr[S], zr[S];
  auto load = [&](int c0) {
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
      const int i = lane + j * kWave, p = min(pos0 + i / (F::kK / 4), a.seq - 1);
      const int col = min(c0 * F::kW + 4 * (i % (F::kK / 4)), a.m.cols - 4);
      xr[j] = *reinterpret_cast<const v4f*>(a.x + (size_t)p * a.m.cols + col);
    }
#pragma unroll
    for (int i = 0; i < S; i++) {
      const int c = min(c0 + i, nc - 1);
      wr[i] = rp[c];
      if constexpr (FMT == QH_FMT_INT4) {
        sr[i] = a.m.scales[(size_t)row * a.m.gpr + c / a.m.cpg];
        zr[i] = a.m.zeros[(size_t)row * a.m.gpr + c / a.m.cpg];
      } else {
        sr[i] = srow;
        zr[i] = 0.f;
      }
    }
  };
  // Stored with each 16 columns as [k % 4][k / 4], so a lane's element of four instructions is
  // one ds_read_b128 (f16's 8-column chunks: halves of it).
  auto store = [&](float* dst) {
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
      const int i = lane + j * kWave, p = i / (F::kK / 4), q = i % (F::kK / 4);
      float* d = dst + p * F::kXRow + 16 * (q >> 2) + (q & 3);
      d[0] = xr[j].x;
      d[4] = xr[j].y;
      d[8] = xr[j].z;
      d[12] = xr[j].w;
    }
  };
  f64x4 st[F::kLevels][T], root[T];
  if (slabs_of(0) > 0) {
    load(first);
    store(xs[wave]);
  }
#pragma unroll 1
  for (int g = 0; g < groups; g++) {
    f64x4 acc[S][T];
#pragma unroll
    for (int i = 0; i < S; i++)
#pragma unroll
      for (int t = 0; t < T; t++) acc[i][t] = (f64x4){0.0, 0.0, 0.0, 0.0};
    const int ns = slabs_of(g);
#pragma unroll 1
    for (int j = 0; j < ns; j++) {
      const int c0 = first + g * S + j * a.tl;
      const int cn = j + 1 < ns ? c0 + a.tl : first + (g + 1) * S;
      const bool more = j + 1 < ns || (g + 1 < groups && slabs_of(g + 1) > 0);
      RowChunk<FMT> rc[S];
#pragma unroll
      for (int i = 0; i < S; i++) rc[i].set(wr[i], sr[i], zr[i]);
      if (more) load(cn);
      wave_lds_handoff();  // the wave's own stores of this slab precede its reads
      const float* xb = xs[wave];
#pragma unroll
      for (int i = 0; i < S; i++) {
        if (c0 + i < nc) {
          constexpr int kSteps = F::kW / 4;
          float xv[T][kSteps];
#pragma unroll
          for (int t = 0; t < T; t++) {
            const float* xp = xb + (16 * t + n) * F::kXRow + 4 * g4;
            if constexpr (FMT == QH_FMT_F16) {
              const float2 v = *reinterpret_cast<const float2*>(xp + 16 * (i >> 1) + 2 * (i & 1));
              xv[t][0] = v.x;
              xv[t][1] = v.y;
            } else {
#pragma unroll
              for (int q = 0; q < kSteps / 4; q++) {
                const v4f v = *reinterpret_cast<const v4f*>(xp + i * F::kW + 16 * q);
#pragma unroll
                for (int e = 0; e < 4; e++) xv[t][4 * q + e] = v[e];
              }
            }
          }
          chain64_steps<FMT, kSteps, T>(rc[i], xv, g4, two, acc[i]);
        }
      }
      wave_lds_handoff();
      if (more) store(xs[wave]);
    }
#pragma unroll
    for (int w = 1; w < S; w *= 2)
#pragma unroll
      for (int i = 0; i < S; i += 2 * w)
#pragma unroll
        for (int t = 0; t < T; t++) acc[i][t] += acc[i + w][t];
    bool open = true;
#pragma unroll
    for (int t = 0; t < T; t++) root[t] = acc[0][t];
#pragma unroll
    for (int lv = 0; lv < F::kLevels; lv++) {
      if (open) {
        if (g >> lv & 1) {
#pragma unroll
          for (int t = 0; t < T; t++) root[t] = st[lv][t] + root[t];
        } else {
#pragma unroll
          for (int t = 0; t < T; t++) st[lv][t] = root[t];
          open = false;
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < T; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) reinterpret_cast<double*>(xs[wave])[(t * 4 + r) * kWave + lane] = root[t][r];
  __syncthreads();
  // Wave w finishes register w of each tile: position 16t + 4r + lane / 16, row lane % 16.
  if (row0 + n >= a.m.rows) return;
#pragma unroll
  for (int t = 0; t < T; t++) {
    const int p = pos0 + 16 * t + 4 * wave + g4;
    if (p < a.seq) {
      double q[kBlock / kWave];
#pragma unroll
      for (int w = 0; w < kBlock / kWave; w++) q[w] = reinterpret_cast<const double*>(xs[w])[(t * 4 + wave) * kWave + lane];
      const double v = (q[0] + q[1]) + (q[2] + q[3]);
      a.y[(size_t)p * a.m.rows + row] = (float)(a.bias ? v + (double)a.bias[row] : v);
    }
  }
}

bool chain_f64_supported(const DMat& m, const float* x, int seq) {
  return seq >= kChain64MinSeq && m.cols % 4 == 0 && ((uintptr_t)x & 15) == 0;
}

hipError_t launch_chain_f64(hipStream_t s, const DMat& m, const float* x, const float* bias, float* y, int seq) {
  ChainArgs a{};
  a.m = m;
  a.x = x;
  a.bias = bias;
  a.y = y;
  a.seq = seq;
  a.tl = team_width(m.nchunks);
  const int rows = (m.rows + kChain64N - 1) / kChain64N, tiles = (seq + kChain64M - 1) / kChain64M;
  const bool multi = m.nchunks > a.tl;
  // A tile a block where each CU then has at most one: two a block would leave CUs idle and take a
  // third longer (24 positions, us, two | one: 128 x 896 f16 12.0 | 8.5, 30 x 4864 int4 54.8 | 35.0).
  const int t = tiles > 1 && rows * tiles > 256 ? 2 : 1;
  const dim3 grid(rows, (tiles + t - 1) / t);
  auto go = [&](auto one, auto many) {
    if (multi) hipLaunchKernelGGL(many, grid, dim3(kBlock), 0, s, a);
    else hipLaunchKernelGGL(one, grid, dim3(kBlock), 0, s, a);
  };
  auto fmt = [&](auto f) {
    constexpr int F = decltype(f)::value;
    if (t == 2) go(k_chain_f64<F, false, 2>, k_chain_f64<F, true, 2>);
    else go(k_chain_f64<F, false, 1>, k_chain_f64<F, true, 1>);
  };
  switch (m.format) {
    case QH_FMT_F16: fmt(std::integral_constant<int, QH_FMT_F16>()); break;
    case QH_FMT_INT8: fmt(std::integral_constant<int, QH_FMT_INT8>()); break;
    default: fmt(std::integral_constant<int, QH_FMT_INT4>()); break;
  }
  return hipGetLastError();
}

}  // namespace qh
