// The batched prefill forward: GpuModel.#forward (src/gpu/model.js:240-402) over
// `seq` positions at once, with the decode step's sums
// (QH_MATMUL_BATCHED: chain.hip; the reference's batchedMatvec, src/gpu/kernels.js:232-290,
// selected by src/gpu/model.js:297-306) or once per prefill on the matrix cores
// (QH_MATMUL_MFMA, prefill.hip).
//
// Per layer, over all positions: rmsnorm -> q|k|v matmul + bias -> rope (f64) with
// the f16 K/V append -> attention (QH_MATMUL_BATCHED: the decode step's algorithm
// for the model's numerics, one query per position; QH_MATMUL_MFMA: flash attention
// on the matrix cores) -> o matmul, residual add -> rmsnorm -> gate|up
// matmul -> swiglu -> down matmul, residual add. The last position's row then goes
// through the decode step's own output head and pick.
//
// QH_MATMUL_BATCHED sums every output exactly as the decode step does (same
// matvec summation order, same rope, attention and merge arithmetic, same f32
// residual adds), so a prefill and the same positions decoded one by one give
// the same bits -- the reference's prefill == incremental decode property
// (README.md:256-272, web/model.html:169-198). QH_MATMUL_MFMA is held to a stated
// tolerance instead.
#include <initializer_list>

#include "attention.h"
#include "device_common.h"
#include "model_dev.h"

namespace qh {

// Rows of q|k|v at positions past+t -- each the sum of `splits` partial rows (planes of
// seq rows apart, in k_gemm_finish's order) plus `bias` when given, else the row itself
// (bias included) -- with q and k heads rotated as the decode step's QKV epilogue does
// (rope_pair over f64 angles), q to `q`, k and v to the f16 caches.
// grid (ceil(items / 256), seq).
// Columns col[0..N) of a row summed over `splits` partial rows (`plane` floats apart) in split
// order, + bias. Every load is issued before any is used -- the splits four at a time from
// clamped indices, the bias (or the row itself where there is none) up front -- since a load
// inside a loop of run-time count, or behind a branch, makes the compiler wait for each in turn.
template <int N>
__device__ __forceinline__ void split_sum_cols(const float* row, size_t plane, int splits, const float* bias,
                                               const int (&col)[N], float (&v)[N]) {
  const float* bsrc = bias ? bias : row;
  float b[N];
#pragma unroll
  for (int k = 0; k < N; k++) {
    b[k] = bsrc[col[k]];
    v[k] = 0.f;
  }
  for (int sp0 = 0; sp0 < splits; sp0 += 4) {
    float x[4][N];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const float* src = row + (size_t)min(sp0 + u, splits - 1) * plane;
#pragma unroll
      for (int k = 0; k < N; k++) x[u][k] = src[col[k]];
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (sp0 + u < splits) {
#pragma unroll
        for (int k = 0; k < N; k++) v[k] += x[u][k];
      }
  }
  if (bias) {
#pragma unroll
    for (int k = 0; k < N; k++) v[k] += b[k];
  }
}

// CHAIN: the row comes from the f32 contraction `chain` (its splits' tree, scale and bias) instead.
template <bool CHAIN>
__global__ void k_rope_kv(const float* __restrict__ qkv, int splits, const float* __restrict__ bias, ChainOut chain,
                          float* __restrict__ q, uint16_t* __restrict__ kc, uint16_t* __restrict__ vt,
                          const double* __restrict__ rope_cos, const double* __restrict__ rope_sin, int past,
                          int heads, int kv_heads, int capacity, int vstride) {
  const int t = blockIdx.y, pos = past + t;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int hidden = heads * kHeadDim, kvd = kv_heads * kHeadDim;
  const int width = hidden + 2 * kvd;
  const size_t plane = (size_t)gridDim.y * width;
  const float* row = qkv + (size_t)t * width;
  const int rope_pairs = (heads + kv_heads) * 32;
  if (i < rope_pairs) {
    const int head = i / 32, j = i % 32;
    const int base = head < heads ? head * kHeadDim : hidden + (head - heads) * kHeadDim;
    const double cs = rope_cos[(size_t)pos * 32 + j], sn = rope_sin[(size_t)pos * 32 + j];
    const int col[2] = {base + j, base + j + 32};
    float x[2], lo, hi;
    if constexpr (CHAIN) {
#pragma unroll
      for (int k = 0; k < 2; k++) x[k] = chain_value(chain, (size_t)t * width + col[k], col[k]);
    } else {
      split_sum_cols<2>(row, plane, splits, bias, col, x);
    }
    rope_pair(x[0], x[1], cs, sn, &lo, &hi);
    if (head < heads) {
      q[(size_t)t * hidden + head * kHeadDim + j] = lo;
      q[(size_t)t * hidden + head * kHeadDim + j + 32] = hi;
    } else {
      uint16_t* k = kc + ((size_t)(head - heads) * capacity + pos) * kHeadDim;
      k[j] = __builtin_bit_cast(uint16_t, (_Float16)lo);
      k[j + 32] = __builtin_bit_cast(uint16_t, (_Float16)hi);
    }
  } else if (i < rope_pairs + kvd) {
    const int e = i - rope_pairs;  // kv head e/64, dimension e%64
    const int col[1] = {hidden + kvd + e};
    float x[1];
    if constexpr (CHAIN) x[0] = chain_value(chain, (size_t)t * width + col[0], col[0]);
    else split_sum_cols<1>(row, plane, splits, bias, col, x);
    vt[(size_t)e * vstride + pos] = __builtin_bit_cast(uint16_t, (_Float16)x[0]);
  }
}

// The decode step's slot merge for every query: out [seq][heads*64]. grid (seq).
__global__ __launch_bounds__(kBlock) void k_attn_merge_rows(const float* __restrict__ part, int heads,
                                                            float* __restrict__ out) {
  __shared__ float wl[kBlock];
  const int t = blockIdx.x;
  CombineIn in;
  in.load(part + (size_t)t * heads * kDecodeSlots * kPartStride, heads);
  const v4f acc = attn_combine_quad(in, wl);
  const int i = threadIdx.x;
  if (i < heads * kCombineLanes)
    *reinterpret_cast<v4f*>(out + (size_t)t * heads * kHeadDim + 4 * i) = acc;
}

// h[t][j] = silu(g) * u over interleaved gate|up rows (g = gu[t][2j], u = gu[t][2j+1]), as
// the decode step's SWIGLU epilogue evaluates it: in f64 (src/core/ops.js:81-91), or in
// f32 for fast numerics (F32).
template <bool F32>
__global__ void k_swiglu_pairs(const float* __restrict__ gu, float* __restrict__ h, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if constexpr (F32) {
    h[i] = swiglu_f32(gu[2 * i], gu[2 * i + 1]);
  } else {
    const double g = gu[2 * i], u = gu[2 * i + 1];
    h[i] = (float)(g / (1.0 + exp(-g)) * u);
  }
}

// The residual add of a contraction and the rmsnorm that follows it (gain null: the add alone), a
// row per block: x += y, xn = rmsnorm(x), as launch_add and k_rmsnorm_f32 evaluate them over a
// finished y. n % 4 == 0, n <= kStageMax.
__global__ __launch_bounds__(kBlock) void k_chain_add_norm(ChainOut y, float* __restrict__ x,
                                                           const float* __restrict__ gain, float eps,
                                                           float* __restrict__ xn) {
  __shared__ float red[kBlock / kWave];
  const int t = blockIdx.x, n = y.rows, n4 = n >> 2;
  v4f* x4 = reinterpret_cast<v4f*>(x + (size_t)t * n);
  StageIn in;
#pragma unroll
  for (int j = 0; j < kStageVec; j++) {
    const int i = threadIdx.x + j * kBlock;
    if (i < n4) {
      const v4f r = x4[i];
      if (gain) in.g[j] = reinterpret_cast<const v4f*>(gain)[i];
      in.v[j] = r + chain_value4(y, t, i);
      x4[i] = in.v[j];
    }
  }
  if (!gain) return;
  const float scale = rms_scale_f32(in, n, eps, red);
  v4f* y4 = reinterpret_cast<v4f*>(xn + (size_t)t * n);
#pragma unroll
  for (int j = 0; j < kStageVec; j++) {
    const int i = threadIdx.x + j * kBlock;
    if (i < n4) y4[i] = rms_apply_f32(in.v[j], scale, in.g[j]);
  }
}

// h[t][j] = silu(gate) * up over the interleaved gate|up outputs, four outputs a thread.
// grid (ceil(rows / 4 / 256), seq).
__global__ __launch_bounds__(kBlock) void k_chain_swiglu(ChainOut gu, float* __restrict__ h) {
  const int t = blockIdx.y, i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= gu.rows / 4) return;
  const v4f v = chain_value4(gu, t, i);
  *reinterpret_cast<float2*>(h + (size_t)t * (gu.rows / 2) + 2 * i) =
      float2{swiglu_f32(v.x, v.y), swiglu_f32(v.z, v.w)};
}

// rows [seq][hidden] = bf16 embedding rows of tokens[past .. past+seq-1], widened exactly.
__global__ void k_embed_rows(const uint16_t* __restrict__ embed, const int* __restrict__ tokens, int past,
                             int hidden, int vocab, float* __restrict__ rows) {
  const int t = blockIdx.x;
  int tok = tokens[past + t];
  tok = (tok < 0 || tok >= vocab) ? 0 : tok;  // ids are validated on the host
  const uint16_t* src = embed + (size_t)tok * hidden;
  for (int i = threadIdx.x; i < hidden; i += blockDim.x)
    rows[(size_t)t * hidden + i] = __builtin_bit_cast(float, (uint32_t)src[i] << 16);
}

// Whether the attention of `seq` prompt queries, the last over `total` positions, runs as the decode
// step's launch and a merge over its partials, 16 blocks a query and kv head, instead of in
// launch_attn_prompt's one block: its eight waves take the context's 16 slots two each, for every 256
// blocks once more, where the 16 blocks of few queries have the chip to themselves. What one block
// costs more than 16 and the merge was fitted to 2 to 64 queries over 0 to 8000 positions of 1 to 16
// kv heads; us a layer, 2 kv heads: 2 queries after 8000 positions +50, after 2000 +11, after 200
// -0.6; 32 after 8000 +39, after 1000 +1.4, after 500 -3; 64 after 3000 +3.7, after 2000 -1.3.
static bool attn_steps_pay(int seq, int kv_heads, int total) {
  const int rows = seq * kv_heads;
  const float k = 0.001f * total;
  return 6.6f * k * ((rows + 255) / 256) > 1.5f + rows * (0.07f + 0.0165f * k);
}
// The most queries that do; their partials are in the workspace.
static int step_queries(int kv_heads) { return std::max(64, 256 / kv_heads); }

// Whether batched contractions of `seq` positions run on the f32 matrix cores (launch_chain_f32, the
// same bits) or in launch_matvec_f32's tiles of 8 / 4 / 2 / 1 positions. A chain launch costs the
// same up to 64 positions, the tiles by pass: about 4 units a tile of 8, 5 a smaller one; int4
// chains pay more to convert their weights. Prompts of 24 layers of 896 columns and 4864 ffn rows,
// ms, tiles | chain: int8 10 positions 1.82 | 2.12, 11 2.23 | 2.14, 16 1.90 | 2.18, 20 2.36 | 2.24,
// 32 2.50 | 2.30, 64 3.82 | 2.42; int4 16 1.82 | 2.40, 23 3.08 | 2.47, 32 2.35 | 2.56, 48 2.89 | 2.64;
// f16 20 2.39 | 2.28, 24 2.16 | 2.29, 32 2.55 | 2.37. Narrower matrices leave CUs free for more
// tiles at once, so the chain also has to be estimated shorter over `matrices` (four layers, us: 512
// columns and 1536 rows int4 64 positions 315 | 572, 128 and 256 int8 64 209 | 274, 512 positions
// 334 | 372; the estimates err by a few per cent, and lean to the chain by three).
static bool chain_pays(std::initializer_list<const DMat*> matrices, int seq) {
  const int units = 4 * (seq / 8) + 5 * __builtin_popcount(seq & 7);
  if (seq <= 8 || units <= ((*matrices.begin())->format == QH_FMT_INT4 ? 16 : 12)) return false;
  float tiles = 0.f, chain = 0.f;
  for (const DMat* m : matrices) {
    tiles += matvec_f32_us(*m, seq);
    chain += chain_f32_us(*m, seq);
  }
  return 0.97f * chain < tiles;
}

int prefill_chunk(const ModelDev& m, const CacheDev& c) {
  int p = c.capacity < kPrefillChunk ? c.capacity : kPrefillChunk;
  if (m.numerics == QH_NUMERICS_EXACT && c.capacity > kPLds) {
    // exact attention past kPLds keeps every query's scores: bound them to 64M floats
    const size_t per = (size_t)m.heads * (c.score_stride + attn_spans(c.capacity));
    const size_t fit = ((size_t)64 << 20) / per;
    p = (int)std::max<size_t>(1, std::min<size_t>(p, fit));
  }
  return p;
}

// Every layer matrix contracts on the matrix cores (the fused layer loop below).
static bool all_mfma(const ModelDev& m) {
  for (int L = 0; L < m.layers; L++) {
    const LayerDev& l = m.layers_host[L];
    for (const DMat* w : {&l.qkv, &l.o, &l.gu, &l.down})
      if (!matmul_prefill_supported(*w)) return false;
  }
  return m.hidden <= 8192 && m.intermediate <= 8192;
}

// The fused layer loop's part of the scratch: digit planes of the widest row, row factors,
// then the largest split partials of any matrix at any length up to P.
static size_t mfma_digit_region(const ModelDev& m, size_t P) {
  return digits_bytes((int)P, std::max(m.hidden, m.intermediate)) + ((P * sizeof(double) + 255) & ~(size_t)255);
}

PrefillBytes prefill_bytes(const ModelDev& m, const CacheDev& c, int matmul) {
  const size_t P = prefill_chunk(m, c);
  const size_t d = m.hidden, kv = (size_t)m.kv_heads * m.head_dim, f = m.intermediate;
  PrefillBytes b{};
  b.floats = P * (5 * d + (d + 2 * kv) + 3 * f);
  if (m.numerics == QH_NUMERICS_FAST)
    b.floats += (decode_attn_long(c.capacity) ? P : std::min<size_t>(P, step_queries(m.kv_heads))) * m.heads * kDecodeSlots * kPartStride;
  else if (m.numerics == QH_NUMERICS_EXACT && c.capacity > kPLds) b.floats += P * m.heads * (c.score_stride + attn_spans(c.capacity));
  b.counters = m.numerics == QH_NUMERICS_EXACT ? P * m.heads : 0;
  const bool chain = m.numerics == QH_NUMERICS_FAST && !(matmul == QH_MATMUL_MFMA && all_mfma(m));
  size_t scratch = chain ? chain_partials_bound(m.lm_head, kHeadRows) : 0;  // enqueue_head_rows
  // exact contractions read an f64 copy of x only below the f64 matrix cores' positions
  const int x64 = std::min((int)P, kChain64MinSeq - 1);
  if (m.numerics == QH_NUMERICS_EXACT) scratch = matvec_x64_bytes(m.lm_head, x64);
  for (int L = 0; L < m.layers; L++) {
    const LayerDev& l = m.layers_host[L];
    for (const DMat* w : {&l.qkv, &l.o, &l.gu, &l.down}) {
      if (m.numerics == QH_NUMERICS_EXACT) scratch = std::max(scratch, matvec_x64_bytes(*w, x64));
      if (chain) scratch = std::max(scratch, chain_partials_bound(*w, (int)P));
      if (matmul == QH_MATMUL_MFMA && matmul_prefill_supported(*w))
        scratch = std::max(scratch, matmul_prefill_scratch_bytes(*w, (int)P));
    }
  }
  if (matmul == QH_MATMUL_MFMA && all_mfma(m)) {
    size_t parts = 0;
    for (int L = 0; L < m.layers; L++) {
      const LayerDev& l = m.layers_host[L];
      for (const DMat* w : {&l.qkv, &l.o, &l.gu, &l.down}) parts = std::max(parts, gemm_partials_bytes(*w, (int)P));
    }
    scratch = std::max(scratch, mfma_digit_region(m, P) + parts);
  }
  b.scratch = scratch;
  return b;
}

// The matrix-core layers. Each contraction reads the digit planes its producer wrote
// (launch_rows), and its split partials are summed by its consumer -- rope and the KV
// write for q|k|v, the residual add + next rmsnorm for o and down, swiglu for gate|up --
// so a layer is ten launches: 4 contractions, rope, attention, 4 row kernels.
static hipError_t prefill_layers_mfma(hipStream_t s, const ModelDev& m, const CacheDev& c, const PrefillDev& p,
                                      int past, int seq) {
  const int d = m.hidden, f = m.intermediate;
  const size_t P = p.positions;
  char* base = static_cast<char*>(p.scratch);
  int8_t* digits = reinterpret_cast<int8_t*>(base);
  double* rowf = reinterpret_cast<double*>(base + digits_bytes((int)P, std::max(d, f)));
  float* part = reinterpret_cast<float*>(base + mfma_digit_region(m, P));
  const size_t part_bytes = p.scratch_bytes - mfma_digit_region(m, P);
  struct Out {
    const float* p;
    int splits;
    const float* bias;
  };
  auto gemm = [&](const DMat& w, const float* bias, float* y, Out* o) {
    int splits = 1;
    const hipError_t e = launch_gemm_digits(s, w, digits, rowf, seq, bias, y, part, part_bytes, &splits);
    *o = Out{splits > 1 ? part : y, splits, splits > 1 ? bias : nullptr};
    return e;
  };
  auto rows = [&](int op, const Out& in, float* resid, const float* gain, int n, bool want_digits) {
    RowArgs r{};
    r.in = in.p;
    r.splits = in.splits;
    r.bias = in.bias;
    r.resid = resid;
    r.gain = gain;
    r.eps = (float)m.eps;
    r.M = seq;
    r.n = n;
    r.Kp = digits_width(n);
    r.digits = want_digits ? digits : nullptr;
    r.row_factor = rowf;
    return launch_rows(s, op, r);
  };
  hipError_t e;
  if ((e = rows(ROW_RMSNORM, Out{p.X, 1, nullptr}, nullptr, m.layers_host[0].in_norm, d, true)) != hipSuccess)
    return e;
  for (int L = 0; L < m.layers; L++) {
    const LayerDev& l = m.layers_host[L];
    uint16_t* kc = c.kv + (size_t)L * c.layer_elems;
    uint16_t* vt = kc + c.key_elems;
    Out o;
    if ((e = gemm(l.qkv, l.qkv_bias, p.QKV, &o)) != hipSuccess) return e;
    const int items = (m.heads + m.kv_heads) * 32 + m.kv_heads * m.head_dim;
    hipLaunchKernelGGL(k_rope_kv<false>, dim3((items + 255) / 256, seq), dim3(256), 0, s, o.p, o.splits, o.bias,
                       ChainOut{}, p.Q, kc, vt, m.rope_cos, m.rope_sin, past, m.heads, m.kv_heads, c.capacity, c.vstride);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    FlashArgs a{};
    a.q = p.Q;
    a.kc = kc;
    a.vt = vt;
    a.out = p.ATT;
    a.past = past;
    a.seq = seq;
    a.capacity = c.capacity;
    a.vstride = c.vstride;
    a.heads = m.heads;
    a.kv_heads = m.kv_heads;
    if ((e = launch_flash_prefill(s, a)) != hipSuccess) return e;
    if ((e = rows(ROW_PLAIN, Out{p.ATT, 1, nullptr}, nullptr, nullptr, d, true)) != hipSuccess) return e;
    if ((e = gemm(l.o, nullptr, p.Y, &o)) != hipSuccess) return e;
    if ((e = rows(ROW_RMSNORM, o, p.X, l.post_norm, d, true)) != hipSuccess) return e;
    if ((e = gemm(l.gu, nullptr, p.GU, &o)) != hipSuccess) return e;
    if ((e = rows(ROW_SWIGLU, o, nullptr, nullptr, f, true)) != hipSuccess) return e;
    if ((e = gemm(l.down, nullptr, p.Y, &o)) != hipSuccess) return e;
    if (L + 1 < m.layers) e = rows(ROW_RMSNORM, o, p.X, m.layers_host[L + 1].in_norm, d, true);
    else e = rows(ROW_PLAIN, o, p.X, nullptr, d, false);  // the last residual add; the head follows
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// The layer's matmul: MFMA (int8/int4 weights), or the batched matvec tiles summing as
// the decode step does for the model's numerics.
static hipError_t matmul(hipStream_t s, const ModelDev& m, int mode, const DMat& w, const float* x,
                         const float* bias, float* y, int seq, const PrefillDev& p) {
  if (mode == QH_MATMUL_MFMA && matmul_prefill_supported(w))
    return launch_matmul_prefill(s, w, x, bias, y, seq, p.scratch, p.scratch_bytes);
  if (m.numerics == QH_NUMERICS_FAST) {
    if (chain_pays({&w}, seq))
      return launch_chain_f32(s, w, x, bias, y, seq, static_cast<float*>(p.scratch), p.scratch_bytes);
    return launch_matvec_f32(s, w, x, bias, y, seq);
  }
  if (!chain_f64_supported(w, x, seq) && matvec_x64_bytes(w, seq) > p.scratch_bytes) return hipErrorInvalidValue;
  return launch_matvec(s, w, x, bias, y, seq, static_cast<double*>(p.scratch));
}

// ------------------------------------------- a prompt's queries, merged in place --
// The decode step's attention for each query of a prompt (caches of up to kLongCapacity
// positions), slots and merge in one block per (kv head, query): the step's launch gives a query
// 32 blocks, most of them empty at prompt lengths, and passes 16 slots of partials through memory
// to a merge launch. A wave takes slots w and w + 8; a slot's steps go to four states (two where
// no slot has more than one chunk), the step's four waves, merged in wave order, and the slots
// merge by the step's own combine: every output has the decode step's bits. An empty slot is the
// neutral partial and is never read. Bound: latency, a query's K/V from L2. 512 queries, 14 heads:
// 83 us (plus a 6 us merge) -> 20 us.
constexpr int kPromptWaves = 8;
template <int NS>
static __global__ __launch_bounds__(kPromptWaves * kWave) void k_attn_prompt(SlotArgs a) {
  __shared__ __attribute__((aligned(16))) float part[kDecodeSlots][8][kPartStride];
  __shared__ float wl[8 * kCombineLanes];
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, n = lane & 15, g = lane >> 4;
  const int group = a.heads / a.kv_heads, kvh = blockIdx.x;
  const int t = gridDim.y - 1 - blockIdx.y;  // the longest contexts first
  const int ctx = a.past + t + 1, nch = attn_chunks(ctx);
  const float* q = a.q + ((size_t)t * a.heads + kvh * group) * kHeadDim;
  f16x8 qh[2], ql[2];
  load_query_split(q + (n < group ? n : 0) * kHeadDim, g, qh, ql);
  const uint16_t* kb = a.kc + (size_t)kvh * a.capacity * kHeadDim;
  const uint16_t* vb = a.vt + (size_t)kvh * kHeadDim * a.vstride;
  for (int sl = w; sl < kDecodeSlots && sl < nch; sl += kPromptWaves) {
    const int chunks = (nch - 1 - sl) / kDecodeSlots + 1;
    const int last = sl + (chunks - 1) * kDecodeSlots;
    const int steps = 2 * chunks - (last * kChunk + 32 >= ctx ? 1 : 0);
    float m[NS], l[NS];
    f32x4 o[NS][4];
    KvStep d[2];
    kv_load(kb, vb, gqa_p0<kDecodeSlots>(sl, 0), a.capacity, a.vstride, n, g, d[0]);
#pragma unroll
    for (int v = 0; v < NS; v++) {
      m[v] = -INFINITY;
      l[v] = 0.f;
#pragma unroll
      for (int dt = 0; dt < 4; dt++) o[v][dt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    // Step i belongs to state i % 4, the next step's loads in flight.
#pragma unroll 1
    for (int i0 = 0; i0 < steps; i0 += NS) {
#pragma unroll
      for (int v = 0; v < NS; v++) {
        if (i0 + v < steps) {
          if (i0 + v + 1 < steps)
            kv_load(kb, vb, gqa_p0<kDecodeSlots>(sl, i0 + v + 1), a.capacity, a.vstride, n, g, d[(v + 1) & 1]);
          kv_step(qh, ql, d[v & 1], gqa_p0<kDecodeSlots>(sl, i0 + v), ctx, ctx, g, m[v], l[v], o[v]);
        }
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < NS; v++) mx = fmaxf(mx, m[v]);
    float wt[NS], lt = 0.f;
#pragma unroll
    for (int v = 0; v < NS; v++) {
      wt[v] = m[v] == -INFINITY ? 0.f : exp2_reduced(m[v] - mx);
      lt = fmaf(l[v], wt[v], lt);
    }
    if (n < group) {
#pragma unroll
      for (int dt = 0; dt < 4; dt++) {
        v4f ot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < NS; v++)
#pragma unroll
          for (int r = 0; r < 4; r++) ot[r] = fmaf(o[v][dt][r], wt[v], ot[r]);
        if (NS < kDecodeWaves) ot += (v4f){0.f, 0.f, 0.f, 0.f};  // the empty waves' + 0 (it turns a -0 around)
        *reinterpret_cast<v4f*>(&part[sl][n][4 + 16 * dt + 4 * g]) = ot;
      }
      if (g == 0) {
        part[sl][n][0] = mx;
        part[sl][n][1] = lt;
      }
    }
  }
  __syncthreads();
  const int i = threadIdx.x;
  if (i >= 8 * kCombineLanes) return;  // whole waves
  const int h = min(i / kCombineLanes, group - 1), k = i % kCombineLanes;
  CombineIn in;
#pragma unroll
  for (int s = 0; s < kDecodeSlots; s++)
    in.ov[s] = s < nch ? *reinterpret_cast<const v4f*>(&part[s][h][4 + 4 * k]) : (v4f){0.f, 0.f, 0.f, 0.f};
  in.mv = k < nch ? part[k][h][0] : -INFINITY;
  in.lv = k < nch ? part[k][h][1] : 0.f;
  const v4f acc = attn_combine_quad(in, wl);
  if (i < group * kCombineLanes)
    *reinterpret_cast<v4f*>(a.out + ((size_t)t * a.heads + kvh * group) * kHeadDim + 4 * i) = acc;
}

// The decode step's attention of `seq` prompt queries, merged into a.out [seq][heads*64]; for
// caches that decode_attn_long does not claim.
static hipError_t launch_attn_prompt(hipStream_t s, const SlotArgs& a, int seq) {
  const dim3 grid(a.kv_heads, seq), block(kPromptWaves * kWave);
  if (attn_chunks(a.past + seq) <= kDecodeSlots) hipLaunchKernelGGL(k_attn_prompt<2>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(k_attn_prompt<kDecodeWaves>, grid, block, 0, s, a);
  return hipGetLastError();
}

// The batched fast-numerics attention of a layer: the decode step's, merged, into p.ATT.
static hipError_t batched_attention(hipStream_t s, const ModelDev& m, const CacheDev& c, const PrefillDev& p,
                                    const uint16_t* kc, const uint16_t* vt, int past, int seq) {
  SlotArgs a{};
  a.q = p.Q;
  a.kc = kc;
  a.vt = vt;
  a.part = p.part;
  a.past = past;
  a.capacity = c.capacity;
  a.vstride = c.vstride;
  a.heads = m.heads;
  a.kv_heads = m.kv_heads;
  if (!decode_attn_long(c.capacity)) {
    if (seq <= step_queries(m.kv_heads) && attn_steps_pay(seq, m.kv_heads, past + seq)) {
      const hipError_t e = launch_attn_decode(s, a, seq, 1);
      if (e != hipSuccess) return e;
      hipLaunchKernelGGL(k_attn_merge_rows, dim3(seq), dim3(kBlock), 0, s, a.part, m.heads, p.ATT);
      return hipGetLastError();
    }
    a.out = p.ATT;
    return launch_attn_prompt(s, a, seq);
  }
  // a long cache's kLongSlots partials per query, a share of the rows at a time so that they fit
  // the workspace sized for kDecodeSlots (each query's result is its own)
  const int share = std::max(1, (int)p.positions * kDecodeSlots / kLongSlots);
  for (int t0 = 0; t0 < seq; t0 += share) {
    SlotArgs b = a;
    b.q = p.Q + (size_t)t0 * m.heads * kHeadDim;
    b.past = past + t0;
    const hipError_t e =
        launch_attn_decode(s, b, std::min(share, seq - t0), 1, p.ATT + (size_t)t0 * m.heads * kHeadDim);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// The batched fast-numerics layers with every contraction on the f32 matrix cores, its splits'
// tree, scale, residual add, rmsnorm or swiglu in its consumer: nine launches a layer against eleven
// and a finish per split contraction (scoring 127 positions of int4 layers 4.1 -> 3.7 ms). The same operations in the same order, so the
// same bits, as the launches of enqueue_prefill_layers.
static hipError_t prefill_layers_chain(hipStream_t s, const ModelDev& m, const CacheDev& c, const PrefillDev& p,
                                       int past, int seq) {
  hipError_t e;
  const int d = m.hidden, f = m.intermediate;
  float* part = static_cast<float*>(p.scratch);
  auto chain = [&](const DMat& w, const float* x, const float* bias, float* y, ChainOut* o) {
    return launch_chain_roots(s, w, x, bias, y, seq, part, p.scratch_bytes, o);
  };
  auto add_norm = [&](const ChainOut& o, const float* gain) {
    hipLaunchKernelGGL(k_chain_add_norm, dim3(seq), dim3(kBlock), 0, s, o, p.X, gain, (float)m.eps, p.XN);
    return hipGetLastError();
  };
  if ((e = launch_rmsnorm(s, p.X, m.layers_host[0].in_norm, p.XN, seq, d, m.eps, true)) != hipSuccess) return e;
  for (int L = 0; L < m.layers; L++) {
    const LayerDev& l = m.layers_host[L];
    uint16_t* kc = c.kv + (size_t)L * c.layer_elems;
    uint16_t* vt = kc + c.key_elems;
    ChainOut o;
    if ((e = chain(l.qkv, p.XN, l.qkv_bias, p.QKV, &o)) != hipSuccess) return e;
    const int items = (m.heads + m.kv_heads) * 32 + m.kv_heads * m.head_dim;
    hipLaunchKernelGGL(k_rope_kv<true>, dim3((items + 255) / 256, seq), dim3(256), 0, s, nullptr, 1, nullptr, o, p.Q,
                       kc, vt, m.rope_cos, m.rope_sin, past, m.heads, m.kv_heads, c.capacity, c.vstride);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = batched_attention(s, m, c, p, kc, vt, past, seq)) != hipSuccess) return e;
    if ((e = chain(l.o, p.ATT, nullptr, p.Y, &o)) != hipSuccess) return e;
    if ((e = add_norm(o, l.post_norm)) != hipSuccess) return e;
    if ((e = chain(l.gu, p.XN, nullptr, p.GU, &o)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_chain_swiglu, dim3((2 * f / 4 + kBlock - 1) / kBlock, seq), dim3(kBlock), 0, s, o, p.H);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = chain(l.down, p.H, nullptr, p.Y, &o)) != hipSuccess) return e;
    if ((e = add_norm(o, L + 1 < m.layers ? m.layers_host[L + 1].in_norm : nullptr)) != hipSuccess) return e;
  }
  return hipSuccess;
}

// Rows that prefill_layers_chain's consumers take as float4 groups.
static bool chain_layers_supported(const ModelDev& m) {
  return m.hidden % 4 == 0 && m.hidden <= kStageMax && m.intermediate % 2 == 0;
}

hipError_t enqueue_prefill_layers(hipStream_t s, const ModelDev& m, const CacheDev& c, const PrefillDev& p,
                                  int mode, int past, int seq) {
  if (mode == QH_MATMUL_MFMA && all_mfma(m)) return prefill_layers_mfma(s, m, c, p, past, seq);
  if (mode != QH_MATMUL_MFMA && m.numerics == QH_NUMERICS_FAST && chain_layers_supported(m)) {
    const LayerDev& l = m.layers_host[0];
    if (chain_pays({&l.gu, &l.qkv, &l.o, &l.down}, seq)) return prefill_layers_chain(s, m, c, p, past, seq);
  }
  hipError_t e;
  const int d = m.hidden, kvd = m.kv_heads * m.head_dim, f = m.intermediate;
  const size_t n = (size_t)seq * d;
  for (int L = 0; L < m.layers; L++) {
    const LayerDev& l = m.layers_host[L];
    uint16_t* kc = c.kv + (size_t)L * c.layer_elems;
    uint16_t* vt = kc + c.key_elems;
    if ((e = launch_rmsnorm(s, p.X, l.in_norm, p.XN, seq, d, m.eps, m.numerics == QH_NUMERICS_FAST)) != hipSuccess) return e;
    if ((e = matmul(s, m, mode, l.qkv, p.XN, l.qkv_bias, p.QKV, seq, p)) != hipSuccess) return e;
    const int items = (m.heads + m.kv_heads) * 32 + kvd;
    hipLaunchKernelGGL(k_rope_kv<false>, dim3((items + 255) / 256, seq), dim3(256), 0, s, p.QKV, 1, nullptr,
                       ChainOut{}, p.Q, kc, vt,
                       m.rope_cos, m.rope_sin, past, m.heads, m.kv_heads, c.capacity, c.vstride);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (mode == QH_MATMUL_MFMA) {
      // the matrix-core prefill: flash attention on MFMA (held to the MFMA tolerance)
      FlashArgs a{};
      a.q = p.Q;
      a.kc = kc;
      a.vt = vt;
      a.out = p.ATT;
      a.past = past;
      a.seq = seq;
      a.capacity = c.capacity;
      a.vstride = c.vstride;
      a.heads = m.heads;
      a.kv_heads = m.kv_heads;
      if ((e = launch_flash_prefill(s, a)) != hipSuccess) return e;
    } else if (m.numerics == QH_NUMERICS_FAST) {
      if ((e = batched_attention(s, m, c, p, kc, vt, past, seq)) != hipSuccess) return e;
    } else {
      ExactArgs a{};
      a.q = p.Q;
      a.kc = kc;
      a.vt = vt;
      a.scores = p.scores;
      a.score_stride = c.score_stride;
      a.max_stride = attn_spans(c.capacity);
      a.maxes = p.scores + (size_t)seq * m.heads * c.score_stride;
      a.counters = p.counters;
      a.out = p.ATT;
      a.past = past;
      a.capacity = c.capacity;
      a.vstride = c.vstride;
      a.heads = m.heads;
      a.kv_heads = m.kv_heads;
      // the arithmetic of the kernel the decode step picks for this cache
      if ((e = launch_attn_exact(s, a, seq, c.capacity, attn_spans(c.capacity))) != hipSuccess) return e;
    }
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = matmul(s, m, mode, l.o, p.ATT, nullptr, p.Y, seq, p)) != hipSuccess) return e;
    if ((e = launch_add(s, p.X, p.Y, (int)n)) != hipSuccess) return e;
    if ((e = launch_rmsnorm(s, p.X, l.post_norm, p.XN, seq, d, m.eps, m.numerics == QH_NUMERICS_FAST)) != hipSuccess) return e;
    if ((e = matmul(s, m, mode, l.gu, p.XN, nullptr, p.GU, seq, p)) != hipSuccess) return e;
    const size_t nh = (size_t)seq * f;
    if (m.numerics == QH_NUMERICS_FAST)
      hipLaunchKernelGGL(k_swiglu_pairs<true>, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, s, p.GU, p.H, nh);
    else
      hipLaunchKernelGGL(k_swiglu_pairs<false>, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, s, p.GU, p.H, nh);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if ((e = matmul(s, m, mode, l.down, p.H, nullptr, p.Y, seq, p)) != hipSuccess) return e;
    if ((e = launch_add(s, p.X, p.Y, (int)n)) != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t enqueue_head_rows(hipStream_t s, const ModelDev& m, const PrefillDev& p, int first, int n, float* logits) {
  const hipError_t e = launch_rmsnorm(s, p.X + (size_t)first * m.hidden, m.final_norm, p.XN, n, m.hidden, m.eps,
                                      m.numerics == QH_NUMERICS_FAST);
  if (e != hipSuccess) return e;
  return matmul(s, m, QH_MATMUL_BATCHED, m.lm_head, p.XN, nullptr, logits, n, p);
}

hipError_t enqueue_embed_rows(hipStream_t s, const ModelDev& m, const CacheDev& c, const PrefillDev& p, int past,
                              int seq) {
  hipLaunchKernelGGL(k_embed_rows, dim3(seq), dim3(256), 0, s, m.embed, c.tokens, past, m.hidden, m.vocab, p.X);
  return hipGetLastError();
}

}  // namespace qh
