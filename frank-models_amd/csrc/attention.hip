// The decode step's attention half: paged KV cache copies, the projection
// epilogue (bias + RoPE), and grouped-query attention of one new token per
// sequence against the paged cache.
//
// Paged cache (components/kvcache/kvcache.mlir, oracles/kvcache.py:51-185):
// a pool [n_blocks, block_size, n_head_kv, head_dim]; sequence b's position
// j lives in physical block block_tables[b, j / block_size] at row
// j % block_size.  The reference gathers max_context_len positions per
// sequence (zero rows at and past context_lens[b]), appends the new K/V and
// runs attention_gqa without a mask (attention_block_decode.mlir:202-216,
// attention_gqa.mlir:120-137).  The attention kernels here read the pool in
// place instead of gathering: the zero rows' contribution is exact in closed
// form (score 0, value 0), so they are counted, not read.
//
// Attention is split over the context: one block per (split of positions, KV
// head, sequence) computes, for the G query heads sharing the
// KV head, the split's max score, sum of exp and unnormalised output; a
// combine kernel merges the splits in order with the zero rows and the new
// token and, in the paged calls, writes the new K/V rows into the pools.
// Where the streaming GEMM does not apply its own epilogue (fp32
// activations, more rows than gemm_stream_fused_rows), the separate bias +
// RoPE and bias + cast kernels here finish the projections.
#include "common.h"
#include "launch.h"

namespace fmoe {
namespace {

constexpr int kCopyThreads = 256;

// ------------------------------------------------------------------ cache copies
// Rows are copied as 32-bit words (a row is n_head_kv * head_dim elements,
// head_dim even, so a bf16 row is a whole number of words).

__global__ __launch_bounds__(kCopyThreads) void kv_gather_kernel(const uint32_t* __restrict__ cache, int64_t n_blocks,
                                                                 int block_size, int row_words,
                                                                 const int* __restrict__ tables, int max_blocks,
                                                                 const int* __restrict__ ctx_lens, int max_ctx,
                                                                 uint32_t* __restrict__ out) {
  const int j = blockIdx.x, b = blockIdx.y;
  const int n = min(max(ctx_lens[b], 0), max_ctx);
  const uint32_t* src = nullptr;
  if (j < n) {
    const int lb = j / block_size;
    const int pb = lb < max_blocks ? tables[static_cast<int64_t>(b) * max_blocks + lb] : -1;
    if (pb >= 0 && pb < n_blocks) src = cache + (static_cast<int64_t>(pb) * block_size + j % block_size) * row_words;
  }
  uint32_t* dst = out + (static_cast<int64_t>(b) * max_ctx + j) * row_words;
  for (int w = threadIdx.x; w < row_words; w += kCopyThreads) dst[w] = src ? src[w] : 0u;
}

// Sequence b's new row into slot (block_idx[b], pos_idx[b]) of `cache`, by
// a whole block of NT threads.  When several sequences name the same slot
// the last one wins, as in the reference's sequential loop
// (oracles/kvcache.py:134-139); slots outside the pool are skipped.
template <int NT>
__device__ void scatter_decode_row(uint32_t* __restrict__ cache, int64_t n_blocks, int block_size, int row_words,
                                   const uint32_t* __restrict__ vals, const int* __restrict__ block_idx,
                                   const int* __restrict__ pos_idx, int batch, int b) {
  const int bi = block_idx[b], p = pos_idx[b];
  bool later = false;
  for (int b2 = b + 1 + static_cast<int>(threadIdx.x); b2 < batch; b2 += NT)
    later |= block_idx[b2] == bi && pos_idx[b2] == p;
  if (__syncthreads_or(later)) return;
  if (bi < 0 || bi >= n_blocks || p < 0 || p >= block_size) return;
  uint32_t* dst = cache + (static_cast<int64_t>(bi) * block_size + p) * row_words;
  const uint32_t* src = vals + static_cast<int64_t>(b) * row_words;
  for (int w = threadIdx.x; w < row_words; w += NT) dst[w] = src[w];
}

__global__ __launch_bounds__(kCopyThreads) void kv_scatter_decode_kernel(uint32_t* __restrict__ cache,
                                                                         int64_t n_blocks, int block_size,
                                                                         int row_words,
                                                                         const uint32_t* __restrict__ vals,
                                                                         const int* __restrict__ block_idx,
                                                                         const int* __restrict__ pos_idx, int batch) {
  scatter_decode_row<kCopyThreads>(cache, n_blocks, block_size, row_words, vals, block_idx, pos_idx, batch,
                                   blockIdx.x);
}

__global__ __launch_bounds__(kCopyThreads) void kv_scatter_prefill_kernel(
    uint32_t* __restrict__ cache, int64_t n_blocks, int block_size, int row_words, const uint32_t* __restrict__ vals,
    int seq_len, const int* __restrict__ tables, int max_blocks, const int* __restrict__ start) {
  const int s = blockIdx.x, b = blockIdx.y;
  const int64_t p = static_cast<int64_t>(start[b]) + s;
  if (p < 0) return;
  const int64_t lb = p / block_size;
  if (lb >= max_blocks) return;
  const int pb = tables[static_cast<int64_t>(b) * max_blocks + lb];
  if (pb < 0 || pb >= n_blocks) return;
  uint32_t* dst = cache + (static_cast<int64_t>(pb) * block_size + p % block_size) * row_words;
  const uint32_t* src = vals + (static_cast<int64_t>(b) * seq_len + s) * row_words;
  for (int w = threadIdx.x; w < row_words; w += kCopyThreads) dst[w] = src[w];
}

// ------------------------------------------------------------------ small helpers
__global__ void iota_kernel(int* __restrict__ v, int n, int* __restrict__ pair, int pair0, int pair1) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i;
  if (i == 0 && pair) {
    pair[0] = pair0;
    pair[1] = pair1;
  }
}

__global__ void fill_int_kernel(int* __restrict__ v, int n, int value) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = value;
}

__device__ __forceinline__ float load_act(const void* p, int dt, int64_t i) {
  return dt == DT_F32 ? static_cast<const float*>(p)[i] : bf16_to_f32(static_cast<const bf16_t*>(p)[i]);
}

__device__ __forceinline__ void store_act(void* p, int dt, int64_t i, float v) {
  if (dt == DT_F32)
    static_cast<float*>(p)[i] = v;
  else
    static_cast<bf16_t*>(p)[i] = f32_to_bf16(v);
}

// qkv [B, nq + 2 nkv] fp32 GEMM output -> + bias, RoPE on the q and k parts
// (pairs (2i, 2i+1), angle pos * freq_scale / freq_base^(2i/D), in double
// precision like the reference oracle), q_rot fp32 [B, nq], k_new / v_new
// [B, nkv] in act dtype (rope.mlir:38-104, oracles/position.py:6-50).
__device__ __forceinline__ float split_sum(const float* p, int nsplit, int64_t stride) {
  float v = p[0];
  for (int k = 1; k < nsplit; ++k) v += p[k * stride];
  return v;
}

__global__ __launch_bounds__(256) void qkv_rope_kernel(const float* __restrict__ qkv, int nsplit, int64_t split_stride,
                                                       const float* __restrict__ bq, const float* __restrict__ bk,
                                                       const float* __restrict__ bv,
                                                       const int64_t* __restrict__ positions, int nq, int nkv, int D,
                                                       double freq_base, double freq_scale, float* __restrict__ q_rot,
                                                       void* __restrict__ k_new, void* __restrict__ v_new, int act) {
  // grid (batch, items / 256): an item is a RoPE pair of the q or k part or
  // one element of the v part
  const int b = blockIdx.x;
  const int i = blockIdx.y * blockDim.x + threadIdx.x;
  const int pairs = (nq + nkv) / 2;
  if (i >= pairs + nkv) return;
  const int width = nq + 2 * nkv;
  const float* row = qkv + static_cast<int64_t>(b) * width;
  if (i >= pairs) {
    const int c = i - pairs;
    float v = split_sum(row + nq + nkv + c, nsplit, split_stride);
    if (bv) v += bv[c];
    store_act(v_new, act, static_cast<int64_t>(b) * nkv + c, v);
    return;
  }
  const int col = 2 * i;
  const bool is_q = col < nq;
  const int c = is_q ? col : col - nq;
  const float* bias = is_q ? bq : bk;
  float x0 = split_sum(row + col, nsplit, split_stride), x1 = split_sum(row + col + 1, nsplit, split_stride);
  if (bias) {
    x0 += bias[c];
    x1 += bias[c + 1];
  }
  float y0, y1;
  rope_pair(x0, x1, positions[b], (c % D) / 2, D, freq_base, freq_scale, y0, y1);
  if (is_q) {
    q_rot[static_cast<int64_t>(b) * nq + c] = y0;
    q_rot[static_cast<int64_t>(b) * nq + c + 1] = y1;
  } else {
    store_act(k_new, act, static_cast<int64_t>(b) * nkv + c, y0);
    store_act(k_new, act, static_cast<int64_t>(b) * nkv + c + 1, y1);
  }
}

// out[b, n] = y[b, n] (+ bias[n]) in act dtype.
// out may alias residual (element-wise, same index).
__global__ __launch_bounds__(256) void bias_cast_kernel(const float* __restrict__ y, int nsplit, int64_t split_stride,
                                                        const float* __restrict__ bias, const void* residual,
                                                        void* out, int64_t rows, int n, int act) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= rows * n) return;
  float v = split_sum(y + i, nsplit, split_stride);
  if (bias) v += bias[i % n];
  if (residual) {
    // the reference rounds the attention output, then adds
    // (transformer_layer_moe_decode.mlir:208-221)
    if (act == DT_BF16) v = bf16_to_f32(f32_to_bf16(v));
    v += load_act(residual, act, i);
  }
  store_act(out, act, i, v);
}

// ------------------------------------------------------------------ split attention
// Two bf16 (low element first) -> two floats.
__device__ __forceinline__ void unpack2(uint32_t w, float* v) {
  v[0] = __uint_as_float(w << 16);
  v[1] = __uint_as_float(w & 0xFFFF0000u);
}

__device__ __forceinline__ f32x4_t attn_mfma16(const u32x4_t a, const u32x4_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                0, 0, 0);
}

struct AttnArgs {
  const float* q;         // [B, n_head * D] fp32, RoPE applied
  const void* k_pool;     // [n_blocks, block_size, n_head_kv, D]
  const void* v_pool;
  const int* tables;      // [B, max_blocks] (this layer)
  const int* ctx_lens;    // [B] (this layer)
  int max_blocks;
  int max_ctx;
  int64_t n_blocks;
  int block_size;
  int n_head, n_head_kv;
  int n_split;
  int split_len;          // positions per split
  bool split_major;       // attn_ring_kernel: every sequence's split s before any split s + 1
  float scale;
  float* part;            // [B, n_head, n_split, D + 2]: o[D], m, l
};

constexpr int kSplitLen = 256;
constexpr int kAttnThreads = 256;  // one thread per position of a split (rows[] fill)
static_assert(kAttnThreads == kSplitLen, "the rows[] fill gives each thread one position");
constexpr int kAttnWaves = kAttnThreads / kWave;

// fp32 pools, and bf16 pools with head_dim 16 and 32 (attn_ring_kernel below
// takes the others).
// Block (split s of kSplitLen positions, KV head, sequence b); wave w owns the
// split's positions [64 w, 64 w + 64) in both phases, so a wave's memory traffic is two
// rounds of independent loads: all of its K rows, then (issued before the
// block-wide softmax, so that their latency overlaps it) all of its V rows.
// Scores: LP lanes per position, each lane holding DL = D/LP dimensions in
// chunks of up to 16 bytes spread so that the LP lanes of a position read
// each span of the row together; the G query heads of the KV head are
// scored from one read of K (query registers: G * DL per lane).  P.V: LPR
// lanes per row, 16 bytes each.
template <typename T, int D, int G, int LP>
__global__ __launch_bounds__(kAttnThreads) void attn_split_kernel(AttnArgs a) {
  constexpr int DL = D / LP;
  static_assert(G <= LP, "one lane per query head stores its score");
  constexpr int EPV = 16 / static_cast<int>(sizeof(T));  // elements per 16 bytes
  constexpr int CW = EPV < DL ? EPV : DL;                 // score chunk (elements)
  constexpr int NC = DL / CW;                             // score chunks per lane per position
  constexpr int kQ = kSplitLen / kAttnWaves;              // positions per wave
  constexpr int PPS = kWave / LP;                         // positions per score step
  constexpr int kSteps = kQ / PPS;                        // score steps
  constexpr int SR = 16 / NC < kSteps ? 16 / NC : kSteps;  // steps per load round (<= 16 loads)
  constexpr int VC = EPV;                                 // P.V elements per lane per row
  constexpr int LPR = D / VC;                             // lanes per row
  constexpr int PP = kWave / LPR;                         // rows per load instruction
  constexpr int NV = kQ / PP;                             // V load instructions per wave
  constexpr int VR = NV < 16 ? NV : 16;                   // per round
  static_assert(kSteps % SR == 0 && NV % VR == 0, "rounds must tile the wave's positions");
  __shared__ float sc[G][kSplitLen];
  __shared__ int rows[kSplitLen];
  __shared__ float red[kAttnWaves][G][D];
  __shared__ float stat[G][2];

  const int s = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
  const int n_b = min(max(a.ctx_lens[b], 0), a.max_ctx);
  const int j0 = s * kSplitLen;
  const int len = min(kSplitLen, n_b - j0);  // block-uniform; <= 0: no cached position here
  float* part = a.part + (static_cast<int64_t>(b) * a.n_head + kvh * G) * a.n_split * (D + 2);
  if (len <= 0) return;  // the combine reads only the splits with positions
  const int64_t row_elems = static_cast<int64_t>(a.n_head_kv) * D;
  {
    const int t = tid;  // kAttnThreads == kSplitLen: one position per thread
    int r = -2;         // -2: past the split's positions; -1: table entry outside the pool (a zero row)
    if (t < len) {
      const int j = j0 + t;
      const int lb = j / a.block_size;
      const int pb = lb < a.max_blocks ? a.tables[static_cast<int64_t>(b) * a.max_blocks + lb] : -1;
      r = (pb >= 0 && pb < a.n_blocks) ? pb * a.block_size + j % a.block_size : -1;
    }
    rows[t] = r;
  }
  const T* kp = static_cast<const T*>(a.k_pool) + static_cast<int64_t>(kvh) * D;
  const T* vp = static_cast<const T*>(a.v_pool) + static_cast<int64_t>(kvh) * D;
  const int tw = wave * kQ;  // this wave's first position
  const int pi = lane / LP, sub = lane % LP;
  float q[G][DL];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < CW; ++e)
        q[g][c * CW + e] =
            a.q[(static_cast<int64_t>(b) * a.n_head + kvh * G + g) * D + c * LP * CW + sub * CW + e] * a.scale;
  __syncthreads();

  // ---- scores, SR steps of 8 positions per round of loads; K stays in its
  // storage format (CWW 32-bit words per chunk) until it is used
  constexpr int CWW = CW * static_cast<int>(sizeof(T)) / 4;
#pragma unroll
  for (int r0 = 0; r0 < kSteps; r0 += SR) {
    uint32_t kr[SR][NC][CWW];
    int rr[SR];
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      rr[u] = rows[tw + (r0 + u) * PPS + pi];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const T* src = kp + rr[u] * row_elems + c * LP * CW + sub * CW;
        if (CWW == 4) {
          const u32x4_t w = rr[u] >= 0 ? *reinterpret_cast<const u32x4_t*>(src) : u32x4_t{0u, 0u, 0u, 0u};
          kr[u][c][0] = w[0], kr[u][c][1 % CWW] = w[1], kr[u][c][2 % CWW] = w[2], kr[u][c][3 % CWW] = w[3];
        } else if (CWW == 2) {
          const u32x2_t w = rr[u] >= 0 ? *reinterpret_cast<const u32x2_t*>(src) : u32x2_t{0u, 0u};
          kr[u][c][0] = w[0], kr[u][c][1 % CWW] = w[1];
        } else {
          kr[u][c][0] = rr[u] >= 0 ? *reinterpret_cast<const uint32_t*>(src) : 0u;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int t = tw + (r0 + u) * PPS + pi;
      float kv[DL];
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (sizeof(T) == 4) {
#pragma unroll
          for (int e = 0; e < CW; ++e) kv[c * CW + e] = __uint_as_float(kr[u][c][e % CWW]);
        } else {
#pragma unroll
          for (int e = 0; e < CWW; ++e) unpack2(kr[u][c][e], kv + c * CW + 2 * e);
        }
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < DL; ++i) acc = fmaf(q[g][i], kv[i], acc);
#pragma unroll
        for (int o = 1; o < LP; o <<= 1) acc += __shfl_xor(acc, o, kWave);
        if (sub == g) sc[g][t] = rr[u] == -2 ? -INFINITY : acc;  // a zero row scores 0
      }
    }
  }

  // ---- V rows of this wave, first round issued before the softmax
  const int pr = lane / LPR, dl = lane - pr * LPR;
  u32x4_t vraw[VR];
  auto load_v = [&](int i0) {
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      const int r = rows[tw + (i0 + i) * PP + pr];
      vraw[i] = r >= 0 ? *reinterpret_cast<const u32x4_t*>(vp + r * row_elems + dl * VC) : u32x4_t{0u, 0u, 0u, 0u};
    }
  };
  load_v(0);
  __syncthreads();

  // ---- per-head max and sum of exp over the split's len positions (only
  // those scores were written); probabilities in place
  for (int g = wave; g < G; g += kAttnWaves) {
    float m = -INFINITY;
    for (int t = lane; t < len; t += kWave) m = fmaxf(m, sc[g][t]);
    m = wave_max(m);
    float l = 0.f;
    for (int t = lane; t < len; t += kWave) {
      const float p = __expf(sc[g][t] - m);
      sc[g][t] = p;
      l += p;
    }
    l = wave_sum(l);
    if (lane == 0) {
      stat[g][0] = m;
      stat[g][1] = l;
    }
  }
  __syncthreads();

  // ---- P.V over this wave's positions
  float acc[G][VC];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int e = 0; e < VC; ++e) acc[g][e] = 0.f;
#pragma unroll
  for (int i0 = 0; i0 < NV; i0 += VR) {
    if (i0 > 0) load_v(i0);
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      const int t = tw + (i0 + i) * PP + pr;
      if (t < len) {
        float v[VC];
        if (sizeof(T) == 4) {
#pragma unroll
          for (int e = 0; e < VC; ++e) v[e] = __uint_as_float(vraw[i][e]);
        } else {
#pragma unroll
          for (int e = 0; e < VC / 2; ++e) unpack2(vraw[i][e], v + 2 * e);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float p = sc[g][t];
#pragma unroll
          for (int e = 0; e < VC; ++e) acc[g][e] = fmaf(p, v[e], acc[g][e]);
        }
      }
    }
  }
  // rows handled by different lane groups of the wave, then the waves in order
#pragma unroll
  for (int o = LPR; o < kWave; o <<= 1)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int e = 0; e < VC; ++e) acc[g][e] += __shfl_xor(acc[g][e], o, kWave);
  if (pr == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int e = 0; e < VC; ++e) red[wave][g][dl * VC + e] = acc[g][e];
  }
  __syncthreads();
  for (int i = tid; i < G * D; i += kAttnThreads) {
    const int g = i / D, d = i - g * D;
    float o = red[0][g][d];
#pragma unroll
    for (int w = 1; w < kAttnWaves; ++w) o += red[w][g][d];
    float* pg = part + (static_cast<int64_t>(g) * a.n_split + s) * (D + 2);
    pg[d] = o;
    if (d == 0) {
      pg[D] = stat[g][0];
      pg[D + 1] = stat[g][1];
    }
  }
}

// bf16 pools with head_dim 64 or 128, 16-byte aligned: the same block
// (split, KV head, sequence) and partial results, with no block barrier
// between its loads.  A block's positions (split_len of them, 256 to 1024) go
// to its W waves in chunks of 64, chunk i to wave i % W (ring_plan).  A chunk is
// four 16-position tiles of K, then four of V, which pass through a ring of
// kSlots tiles of the wave's own in LDS (global_load_lds): a slot is refilled
// as soon as its tile has been used, so loads stay in flight through the
// score, softmax and P.V arithmetic and across the chunks, and nothing keeps
// the waves of a CU in step.
// Bound: the K and V rows' HBM read.  Measured (8 KV heads x 128, 32 query
// heads, kernel trace; before: every load of a phase in registers, two block
// barriers around the softmax): 16 sequences x 4096 positions 61.4 -> 50.7 us
// (5.3 TB/s), 61 x about 750 positions 52.3 -> 42.2 us.
// Scores: v_mfma_f32_16x16x32_bf16, A = 16 positions x 32 dimensions of K, B
// column h = query head h (G <= 8), column 8 + h its remainder: q * scale as
// bf16 high and low parts, about 16 significant bits; K is exact in bf16 and
// the sums are fp32.  K tiles sit in LDS with 16-byte chunk c of row r at
// c ^ (r & 15) (head_dim 64: c ^ ((r >> 1) & 7)), so an operand read of 16
// rows hits all 64 banks.  Softmax per wave in fp32, with a running maximum
// over its chunks.  P.V: 16 bytes of a row per lane in the loads' own lane
// order, fp32; load i of a V tile holds positions kLoads * (lane's row) + i,
// so a lane's probabilities of a tile are neighbours in LDS.
// Rows past the context (-2) and zero rows (-1, table entries outside the
// pool) load some valid row instead; their scores are replaced and their
// values zeroed by selects, so what they loaded never enters the result.
constexpr int kTileRows = 16;
constexpr int kSlots = 4;
constexpr int kChunk = 64;      // positions of a wave per round of the ring
constexpr int kMaxSplitLen = 1024;

template <int D, int G, int W>
struct Ring {
  static constexpr int kRowB = D * 2;
  static constexpr int kRowsPerLoad = 1024 / kRowB;             // 4 or 8
  static constexpr int kLoads = kTileRows / kRowsPerLoad;       // per tile
  static constexpr int kTileB = kTileRows * kRowB;
  static constexpr int kTiles = kChunk / kTileRows;             // of K, and of V, per chunk
  static constexpr int kWaveB = kSlots * kTileB;
  static constexpr int kRowIds = kMaxSplitLen / kAttnWaves;     // per wave
  static constexpr int kP = kChunk * G;                         // probabilities per wave
  static constexpr int kLds = W * (kWaveB + kRowIds * 4 + kP * 4 + G * 8);
  // waves per SIMD the registers must allow: blocks of four waves per CU
  static constexpr int kPerSimd = (D == 64 ? 3 : 2) - (G == 8 ? 1 : 0);
  static_assert(kSlots == kTiles, "K tile i and V tile i share slot i");
  static_assert(kWaveB >= 2 * G * D * 4, "a wave's two partial outputs fit its ring");
};

// What the exponents of a chunk are taken against: its maximum, or 0 where every
// score so far is minus infinity (finite keys whose products overflow, as
// masking ones do), so that such positions weigh 0 and not NaN.
__device__ __forceinline__ float finite_base(float m) { return m == -INFINITY ? 0.f : m; }

// Non-temporal: a step reads each K and V byte once (with the default policy
// the kernel takes 55.5 us at 16 x 4096 positions and 44.9 at 61 x 750).
__device__ __forceinline__ void ring_load(const unsigned char* src, unsigned char* dst) {
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, kNonTemporal);
}

template <int D, int G, int W>
__global__ __launch_bounds__(W * kWave, (Ring<D, G, W>::kPerSimd)) void attn_ring_kernel(AttnArgs a) {
  using R = Ring<D, G, W>;
  constexpr int kL = R::kLoads, kT = R::kTiles, kChunks = R::kRowB / 16;
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  const int s = a.split_major ? blockIdx.z : blockIdx.x, kvh = a.split_major ? blockIdx.x : blockIdx.y;
  const int b = a.split_major ? blockIdx.y : blockIdx.z;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  unsigned char* ring = lds + wave * R::kWaveB;
  int* rows = reinterpret_cast<int*>(lds + W * R::kWaveB) + wave * R::kRowIds;
  float* pw = reinterpret_cast<float*>(lds + W * (R::kWaveB + R::kRowIds * 4)) + wave * R::kP;  // [G][64]
  float* stat = reinterpret_cast<float*>(lds + W * (R::kWaveB + R::kRowIds * 4 + R::kP * 4));  // [waves][G][m, l]

  // Query operand: lane (g = l / 16, column l % 16) holds 8 dimensions at
  // chunk 4 ks + g of head l % 8, the high part in columns 0-7, the remainder
  // in 8-15.  Loaded beside the table entries and the context length, and
  // converted before the first tile load is issued (a wait for it later
  // would wait for those loads too).
  const int q4 = lane >> 4, col = lane & 15, head = col & 7;
  const float* qg = a.q + (static_cast<int64_t>(b) * a.n_head + kvh * G + (head < G ? head : 0)) * D + q4 * 8;
  f32x4_t qx[D / 32][2];
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) {
    qx[ks][0] = *reinterpret_cast<const f32x4_t*>(qg + ks * 32);
    qx[ks][1] = *reinterpret_cast<const f32x4_t*>(qg + ks * 32 + 4);
  }
  // Pool rows of the wave's positions, chunk by chunk.
  const int j0 = s * a.split_len;
  const int n_b = min(max(a.ctx_lens[b], 0), a.max_ctx);
  if (n_b <= j0) return;  // block-uniform; the combine reads only the splits with positions
  const int len = min(a.split_len, n_b - j0);
  const int n_all = (len + kChunk - 1) / kChunk;
  const int n = n_all > wave ? (n_all - wave + W - 1) / W : 0;  // this wave's chunks
  for (int c = 0; c < n; ++c) {
    const int t = (c * W + wave) * kChunk + lane;
    const int j = j0 + t;
    const int lb = j / a.block_size;
    int r = -2;  // past the context
    if (t < len) {
      const int pb = lb < a.max_blocks ? a.tables[static_cast<int64_t>(b) * a.max_blocks + lb] : -1;
      r = pb >= 0 && pb < a.n_blocks ? pb * a.block_size + (j - lb * a.block_size) : -1;
    }
    rows[c * kChunk + lane] = r;
  }

  u32x4_t qv[D / 32];
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y0 = qx[ks][e / 2][2 * (e % 2)] * a.scale, y1 = qx[ks][e / 2][2 * (e % 2) + 1] * a.scale;
      const uint32_t h = pack_bf16x2(y0, y1);
      const uint32_t lo = pack_bf16x2(y0 - __uint_as_float(h << 16), y1 - __uint_as_float(h & 0xFFFF0000u));
      qv[ks][e] = head < G ? (col < 8 ? h : lo) : 0u;
    }
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) asm volatile("" : "+v"(qv[ks]));  // converted here
  float m = -INFINITY, l = 0.f;
  float acc[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;

  // this lane's row and 16-byte chunk of a load
  const int lr = lane / kChunks, lc = lane % kChunks;
  const int64_t row_b = static_cast<int64_t>(a.n_head_kv) * R::kRowB;
  const unsigned char* kp = static_cast<const unsigned char*>(a.k_pool) + kvh * R::kRowB;
  const unsigned char* vp = static_cast<const unsigned char*>(a.v_pool) + kvh * R::kRowB + lc * 16;
  int kc[kL];
#pragma unroll
  for (int i = 0; i < kL; ++i) {
    const int row = i * R::kRowsPerLoad + lr;
    kc[i] = (lc ^ (D == 128 ? row & 15 : (row >> 1) & 7)) * 16;
  }
  uint64_t valid = 0, zero = 0;            // of the chunk whose K tiles are issued last
  uint64_t valid_now = 0, zero_now = 0;    // of the chunk being computed
  // Masks of chunk c, and its unusable rows replaced by a usable one.
  auto chunk_rows = [&](int c) __attribute__((always_inline)) {
    const int r = rows[c * kChunk + lane];
    valid = __ballot(r >= 0);
    zero = __ballot(r == -1);
    if (valid != ~0ull) {
      const int first = valid ? __builtin_amdgcn_readlane(r, __builtin_ctzll(valid)) : 0;
      if (r < 0) rows[c * kChunk + lane] = first;
    }
  };
  if (n > 0) {
    chunk_rows(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < kT; ++it)
#pragma unroll
      for (int i = 0; i < kL; ++i)
        ring_load(kp + rows[it * kTileRows + i * R::kRowsPerLoad + lr] * row_b + kc[i],
                  ring + it * R::kTileB + i * 1024);
  }
  for (int c = 0; c < n; ++c) {
    const bool more = c + 1 < n;
    const int* rc = rows + c * kChunk;
    valid_now = valid;
    zero_now = zero;
    const bool all = valid_now == ~0ull;

    // ---- scores: lane (g, column): positions 16 tile + 4 g + i.  In flight
    // behind K tile `it`: the three tiles after it (K, then V)
    f32x4_t sc[kT];
#pragma unroll
    for (int it = 0; it < kT; ++it) {
      __builtin_amdgcn_s_waitcnt(wait_vm((kSlots - 1) * kL, false));
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      const unsigned char* tile = ring + it * R::kTileB + col * R::kRowB;
      const int sw = D == 128 ? col : col >> 1;
      u32x4_t kv[D / 32];
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks)
        kv[ks] = *reinterpret_cast<const u32x4_t*>(tile + (((4 * ks + q4) ^ sw) << 4));
      int vr[kL];  // the V tile's rows
#pragma unroll
      for (int i = 0; i < kL; ++i) vr[i] = rc[it * kTileRows + lr * kL + i];
      // the slot is refilled after its reads have returned
      __builtin_amdgcn_s_waitcnt(wait_vm(63, true));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kL; ++i) ring_load(vp + vr[i] * row_b, ring + it * R::kTileB + i * 1024);
      f32x4_t d{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks) d = attn_mfma16(kv[ks], qv[ks], d);
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] += __shfl_xor(d[i], 8, kWave);  // high + low part
      if (!all) {
        const uint64_t vm = valid_now >> (4 * q4), zm = zero_now >> (4 * q4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint64_t bit = 1ull << (16 * it + i);
          d[i] = vm & bit ? d[i] : zm & bit ? 0.f : -INFINITY;
        }
      }
      sc[it] = d;
    }
    if (more) chunk_rows(c + 1);

    // ---- softmax over the wave's positions so far; every column of a head
    // agrees
    const float m_old = m;
#pragma unroll
    for (int it = 0; it < kT; ++it)
#pragma unroll
      for (int i = 0; i < 4; ++i) m = fmaxf(m, sc[it][i]);
    m = fmaxf(m, __shfl_xor(m, 16, kWave));
    m = fmaxf(m, __shfl_xor(m, 32, kWave));
    const float base = finite_base(m);
    float sum = 0.f;
#pragma unroll
    for (int it = 0; it < kT; ++it) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sc[it][i] = __expf(sc[it][i] - base);
        sum += sc[it][i];
      }
      if (col < G) *reinterpret_cast<f32x4_t*>(pw + col * kChunk + 16 * it + 4 * q4) = sc[it];
    }
    sum += __shfl_xor(sum, 16, kWave);
    sum += __shfl_xor(sum, 32, kWave);
    if (c > 0) {
      const float f = __expf(m_old - base);
      l = fmaf(l, f, sum);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float fg = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f), g));
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] *= fg;
      }
    } else {
      l = sum;
    }

    // ---- P.V.  In flight behind V tile `it`: the V tiles after it and the
    // next chunk's K tiles
#pragma unroll
    for (int it = 0; it < kT; ++it) {
      if (more || it == 0)
        __builtin_amdgcn_s_waitcnt(wait_vm((kSlots - 1) * kL, false));
      else if (it == 1)
        __builtin_amdgcn_s_waitcnt(wait_vm(2 * kL, false));
      else if (it == 2)
        __builtin_amdgcn_s_waitcnt(wait_vm(kL, false));
      else
        __builtin_amdgcn_s_waitcnt(wait_vm(0, false));
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      const unsigned char* tile = ring + it * R::kTileB + lane * 16;
      u32x4_t v[kL];
      float p[G][kL];
#pragma unroll
      for (int i = 0; i < kL; ++i) v[i] = *reinterpret_cast<const u32x4_t*>(tile + i * 1024);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < kL; ++i) p[g][i] = pw[g * kChunk + it * kTileRows + lr * kL + i];
      int kr[kL];  // the next chunk's K tile rows
#pragma unroll
      for (int i = 0; i < kL; ++i)
        kr[i] = more ? rc[kChunk + it * kTileRows + i * R::kRowsPerLoad + lr] : 0;
      __builtin_amdgcn_s_waitcnt(wait_vm(63, true));
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
#pragma unroll
        for (int i = 0; i < kL; ++i) ring_load(kp + kr[i] * row_b + kc[i], ring + it * R::kTileB + i * 1024);
      }
      if (!all) {
        const uint64_t vm = valid_now >> (lr * kL);
#pragma unroll
        for (int i = 0; i < kL; ++i) v[i] = vm & (1ull << (16 * it + i)) ? v[i] : u32x4_t{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int i = 0; i < kL; ++i) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) unpack2(v[i][e], x + 2 * e);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[g][e] = fmaf(p[g][i], x[e], acc[g][e]);
      }
    }
  }

  // ---- the waves merged in order: each leaves two partial outputs in its
  // (drained) ring and its statistics
#pragma unroll
  for (int o = 2 * kChunks; o < kWave; o <<= 1)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][e] += __shfl_xor(acc[g][e], o, kWave);
  if (lane < 2 * kChunks) {
    float* dst = reinterpret_cast<float*>(ring) + (lane / kChunks) * G * D + (lane % kChunks) * 8;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      *reinterpret_cast<f32x4_t*>(dst + g * D) = f32x4_t{acc[g][0], acc[g][1], acc[g][2], acc[g][3]};
      *reinterpret_cast<f32x4_t*>(dst + g * D + 4) = f32x4_t{acc[g][4], acc[g][5], acc[g][6], acc[g][7]};
    }
  }
  if (lane < G) {
    stat[(wave * G + lane) * 2] = m;
    stat[(wave * G + lane) * 2 + 1] = l;
  }
  __syncthreads();
  float* part = a.part + (static_cast<int64_t>(b) * a.n_head + kvh * G) * a.n_split * (D + 2);
  for (int i = tid; i < G * D; i += W * kWave) {
    const int g = i / D, d = i - g * D;
    float M = stat[g * 2];
#pragma unroll
    for (int w = 1; w < W; ++w) M = fmaxf(M, stat[(w * G + g) * 2]);
    const float base = finite_base(M);
    float o = 0.f, L = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float* src = reinterpret_cast<const float*>(lds + w * R::kWaveB);
      const float f = __expf(stat[(w * G + g) * 2] - base);  // 0 for a wave without positions
      o = fmaf(f, src[i] + src[G * D + i], o);
      L = fmaf(f, stat[(w * G + g) * 2 + 1], L);
    }
    float* pg = part + (static_cast<int64_t>(g) * a.n_split + s) * (D + 2);
    pg[d] = o;
    if (d == 0) {
      pg[D] = M;
      pg[D + 1] = L;
    }
  }
}

// One block per (query head, sequence) merges the context splits with the
// zero rows of the gather (max_ctx - min(ctx_len, max_ctx) keys of score 0
// and value 0) and the new token, whose K/V (RoPE applied) are k_new/v_new.
// Wave 0 reduces the per-split statistics with one split per lane and
// leaves the split weights exp(m_s - M) in LDS; then thread d adds
// dimension d over the splits, kCombineUnroll loads at a time.
constexpr int kCombineThreads = 128;  // >= head_dim
constexpr int kCombineChunk = 1024;   // splits whose weights are held in LDS at once
constexpr int kCombineUnroll = 16;
constexpr int kCombinePre = 16;       // splits (4096 to 16384 positions) prefetched into registers

// Blocks x = n_head and n_head + 1 (launched only with a scatter) write
// k_new / v_new into the pools: the split kernel has read them by then.
__global__ __launch_bounds__(kCombineThreads) void attn_combine_kernel(AttnArgs a, int D,
                                                                       const void* __restrict__ k_new,
                                                                       const void* __restrict__ v_new, int act,
                                                                       void* __restrict__ out, KvScatterDecode sc) {
  __shared__ float wts[kCombineChunk];
  __shared__ float stat[3];  // M, 1 / l, exp(s_new - M) / l
  const int h = blockIdx.x, b = blockIdx.y;
  if (h >= a.n_head) {  // block-uniform
    const bool v = h > a.n_head;
    scatter_decode_row<kCombineThreads>(static_cast<uint32_t*>(v ? sc.v_cache : sc.k_cache), sc.n_blocks,
                                        sc.block_size, sc.row_bytes / 4,
                                        static_cast<const uint32_t*>(v ? v_new : k_new), sc.block_idx, sc.pos_idx,
                                        static_cast<int>(gridDim.y), b);
    return;
  }
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int kvh = h / (a.n_head / a.n_head_kv);
  const int n_b = min(max(a.ctx_lens[b], 0), a.max_ctx);
  const int n_zero = a.max_ctx - n_b;
  const int n_used = (n_b + a.split_len - 1) / a.split_len;
  const float* qh = a.q + (static_cast<int64_t>(b) * a.n_head + h) * D;
  const int64_t kv0 = (static_cast<int64_t>(b) * a.n_head_kv + kvh) * D;
  const float* part = a.part + (static_cast<int64_t>(b) * a.n_head + h) * a.n_split * (D + 2);
  // The first kCombinePre splits' outputs and v_new are loaded before the
  // statistics, so their latency overlaps wave 0's reductions.
  const int n_pre = min(n_used, kCombinePre);
  float pv[kCombinePre];
#pragma unroll
  for (int u = 0; u < kCombinePre; ++u)
    pv[u] = tid < D && u < n_pre ? part[static_cast<int64_t>(u) * (D + 2) + tid] : 0.f;
  const float vn = tid < D ? load_act(v_new, act, kv0 + tid) : 0.f;
  if (tid < kWave) {
    float dot = 0.f;
    for (int d = lane; d < D; d += kWave) dot = fmaf(qh[d] * a.scale, load_act(k_new, act, kv0 + d), dot);
    const float s_new = wave_sum(dot);
    const float m0 = lane < n_used ? part[static_cast<int64_t>(lane) * (D + 2) + D] : -INFINITY;
    float M = fmaxf(fmaxf(s_new, n_zero > 0 ? 0.f : -INFINITY), m0);
    for (int s = lane + kWave; s < n_used; s += kWave) M = fmaxf(M, part[static_cast<int64_t>(s) * (D + 2) + D]);
    M = wave_max(M);
    float l = 0.f;
    for (int s = lane; s < n_used; s += kWave) {
      const float* ps = part + static_cast<int64_t>(s) * (D + 2);
      l = fmaf(ps[D + 1], __expf(ps[D] - M), l);
    }
    l = wave_sum(l) + __expf(s_new - M) + (n_zero > 0 ? static_cast<float>(n_zero) * __expf(-M) : 0.f);
    const float inv = 1.f / l;
    // the first chunk's split weights exp(m_s - M) / l
    for (int s = lane; s < min(n_used, kCombineChunk); s += kWave)
      wts[s] = __expf((s == lane ? m0 : part[static_cast<int64_t>(s) * (D + 2) + D]) - M) * inv;
    if (lane == 0) {
      stat[0] = M;
      stat[1] = inv;
      stat[2] = __expf(s_new - M) / l;
    }
  }
  __syncthreads();
  const float M = stat[0], inv = stat[1];
  float o = stat[2] * vn;
  // splits in order: the prefetched ones, then the rest of each chunk
#pragma unroll
  for (int u = 0; u < kCombinePre; ++u)
    if (u < n_pre) o = fmaf(pv[u], wts[u], o);
  for (int c0 = 0; c0 < n_used; c0 += kCombineChunk) {
    const int cn = min(kCombineChunk, n_used - c0);
    if (c0 > 0) {
      __syncthreads();
      for (int s = tid; s < cn; s += kCombineThreads)
        wts[s] = __expf(part[static_cast<int64_t>(c0 + s) * (D + 2) + D] - M) * inv;
      __syncthreads();
    }
    if (tid < D) {
      for (int s0 = c0 == 0 ? n_pre : 0; s0 < cn; s0 += kCombineUnroll) {
        float v[kCombineUnroll];
#pragma unroll
        for (int u = 0; u < kCombineUnroll; ++u)
          v[u] = s0 + u < cn ? part[static_cast<int64_t>(c0 + s0 + u) * (D + 2) + tid] : 0.f;
#pragma unroll
        for (int u = 0; u < kCombineUnroll; ++u)
          if (s0 + u < cn) o = fmaf(v[u], wts[s0 + u], o);
      }
    }
  }
  if (tid < D) store_act(out, act, (static_cast<int64_t>(b) * a.n_head + h) * D + tid, o);
}

// Lanes per position in the score phase: 8 beat 16 at head_dim 128 (measured
// on bf16 pools, 4 query heads per KV head: 61.5 against 77.9 us at 16 x 4096
// positions), although 16 lanes halve the query registers.
constexpr int kLanesPerPos64 = 8;
constexpr int kLanesPerPos128 = 8;

// How attn_ring_kernel covers `heads` (sequence, KV head) pairs of contexts up
// to max_ctx.  Measured: time of the attention kernels, the split kernel of 256
// positions (one block per 256 positions, whatever the batch) against the choice.
struct RingPlan {
  int split_len, waves;
  bool split_major;
};

// Time of a launch in units of 256 positions of one block, of one unit of
// overhead per block, where `round` blocks are resident and the full splits come
// first.
int64_t ring_rounds(int max_ctx, int64_t heads, int len, int round) {
  const int64_t n = (max_ctx + len - 1) / len, full = heads * (n - 1);
  const int64_t rounds = (full + round - 1) / round, idle = rounds * round - full;
  const int64_t last = (max_ctx - (n - 1) * len + kSplitLen - 1) / kSplitLen + 1;
  return rounds * (len / kSplitLen + 1) + (heads > idle ? (heads - idle + round - 1) / round * last : 0);
}

RingPlan ring_plan(int max_ctx, int64_t heads, int head_dim, int group) {
  RingPlan p{kMaxSplitLen, kAttnWaves, false};
  // head_dim 128 with 8 query heads keeps one wave per SIMD, the others two
  const bool one = head_dim == 128 && group == 8;
  const int round = one ? 256 : 512;
  // Short contexts of many pairs: a block of four waves reserves LDS and SIMD
  // slots for waves that have no chunk, so the blocks get fewer waves, each with
  // a chunk (one wave per SIMD: with enough chunks to fill the SIMDs).  8 query
  // heads x 128, pairs x positions: 1024 x 64 39.6 -> 28.4 us (four waves: 46.8),
  // 1024 x 256 55.9 -> 44.5 (59.6), 512 x 256 33.4 -> 28.2 (33.1), 1024 x 512
  // 85.4 -> 73.6 (83.1).  1 query head x 128: 2048 x 16 26.9 -> 19.6 (30.8), 4096 x
  // 48 53.5 -> 34.9 (56.1), 4096 x 128 78.1 -> 61.1 (66.0); 4 query heads: 1024 x 64
  // 28.3 -> 21.8 (24.3).  Up to one round of four-wave blocks they are level or
  // ahead (256 pairs x 64: 13.1 us, with one wave 14.2).
  if (heads > round) {
    if (max_ctx <= kChunk || (one && max_ctx <= kSplitLen && heads >= 4 * round))
      p.waves = 1;
    else if (max_ctx <= (one ? 2 * kSplitLen : 2 * kChunk))
      p.waves = 2;
    if (p.waves < kAttnWaves) {
      p.split_len = p.waves * kSplitLen;
      return p;
    }
  }
  // Positions per split.  Two waves per SIMD: the most that still gives the GPU
  // two blocks per CU; longer splits spend fewer prologues and merges (whole
  // step at 16 x 4096 positions: 94.3 us with 256, 92.7 with 512, 91.4 with 1024;
  // 128 x 380: 126, 122, 122).  One wave per SIMD: nothing covers a block's
  // latencies, so the length whose rounds of blocks take least (8 query heads,
  // 64 pairs x 2048 positions: 25.8 us with the split kernel, 30.8 with 256, 24.7
  // with 512; 128 x 1250: 32.0, 39.8, 34.4, with 768 30.2).
  if (one) {
    for (int len = kMaxSplitLen - kSplitLen; len >= kSplitLen; len -= kSplitLen)
      if (ring_rounds(max_ctx, heads, len, round) < ring_rounds(max_ctx, heads, p.split_len, round)) p.split_len = len;
  } else {
    while (p.split_len > kSplitLen && heads * ((max_ctx + p.split_len - 1) / p.split_len) < round) p.split_len /= 2;
  }
  // A short last split goes behind every full one: dealt in turn with them, the
  // last full ones start late and the launch ends on a few blocks (4 query heads
  // x 128: 512 pairs x 1100 positions 76.7 us with the split kernel, 79.5 dealt in
  // turn, 64.9 split-major; 256 x 600: 27.8, 29.2, 24.6; 1 query head x 64: 1024 x 1100 65.7,
  // 84.1, 61.6).  Else a sequence's splits run side by side (128 x 2500: 40.7
  // against 42.8; 256 x 5000 positions of 1 query head x 64: 63.0 against 68.0).
  const int n_split = (max_ctx + p.split_len - 1) / p.split_len;
  const int last = max_ctx - (n_split - 1) * p.split_len;
  p.split_major = n_split > 1 && n_split <= 65535 && 4ll * last < 3ll * p.split_len;
  return p;
}

template <int D, int G, int W>
void launch_ring_w(const AttnArgs& a, int B, hipStream_t s) {
  constexpr int lds = Ring<D, G, W>::kLds;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(attn_ring_kernel<D, G, W>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)attr;
  const dim3 grid = a.split_major ? dim3(a.n_head_kv, B, a.n_split) : dim3(a.n_split, a.n_head_kv, B);
  hipLaunchKernelGGL((attn_ring_kernel<D, G, W>), grid, dim3(W * kWave), lds, s, a);
}

template <int D, int G>
void launch_ring_n(const AttnArgs& a, int waves, int B, hipStream_t s) {
  if (waves == 1)
    launch_ring_w<D, G, 1>(a, B, s);
  else if (waves == 2)
    launch_ring_w<D, G, 2>(a, B, s);
  else
    launch_ring_w<D, G, kAttnWaves>(a, B, s);
}

template <int D>
hipError_t launch_ring(const AttnArgs& a, int G, int waves, int B, hipStream_t s) {
  switch (G) {
    case 1: launch_ring_n<D, 1>(a, waves, B, s); break;
    case 2: launch_ring_n<D, 2>(a, waves, B, s); break;
    case 4: launch_ring_n<D, 4>(a, waves, B, s); break;
    case 8: launch_ring_n<D, 8>(a, waves, B, s); break;
    default: return hipErrorNotSupported;
  }
  return hipGetLastError();
}

template <typename T, int D, int LP>
hipError_t launch_split_g(const AttnArgs& a, int G, int B, hipStream_t s) {
  const dim3 grid(a.n_split, a.n_head_kv, B);
  switch (G) {
    case 1: hipLaunchKernelGGL((attn_split_kernel<T, D, 1, LP>), grid, dim3(kAttnThreads), 0, s, a); break;
    case 2: hipLaunchKernelGGL((attn_split_kernel<T, D, 2, LP>), grid, dim3(kAttnThreads), 0, s, a); break;
    case 4: hipLaunchKernelGGL((attn_split_kernel<T, D, 4, LP>), grid, dim3(kAttnThreads), 0, s, a); break;
    case 8: hipLaunchKernelGGL((attn_split_kernel<T, D, 8, LP>), grid, dim3(kAttnThreads), 0, s, a); break;
    default: return hipErrorNotSupported;
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_split_d(const AttnArgs& a, int D, int G, int B, hipStream_t s) {
  switch (D) {
    case 16: return launch_split_g<T, 16, 8>(a, G, B, s);
    case 32: return launch_split_g<T, 32, 8>(a, G, B, s);
    default: break;
  }
  if constexpr (sizeof(T) == 4) {  // bf16: attn_ring_kernel
    if (D == 64) return launch_split_g<T, 64, kLanesPerPos64>(a, G, B, s);
    if (D == 128) return launch_split_g<T, 128, kLanesPerPos128>(a, G, B, s);
  }
  return hipErrorNotSupported;
}

}  // namespace

bool attn_decode_supported(int head_dim, int group) {
  return (head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128) &&
         (group == 1 || group == 2 || group == 4 || group == 8);
}

int attn_decode_splits(int max_ctx) { return (max_ctx + kSplitLen - 1) / kSplitLen; }

hipError_t launch_attn_decode(const float* q_rot, const void* k_pool, const void* v_pool, int64_t n_blocks,
                              int block_size, const int* tables, int max_blocks, const int* ctx_lens, int max_ctx,
                              const void* k_new, const void* v_new, int batch, int n_head, int n_head_kv,
                              int head_dim, int dtype, float scale, float* part, void* out, hipStream_t s,
                              const KvScatterDecode* scatter) {
  if (!attn_decode_supported(head_dim, n_head / n_head_kv) || n_head % n_head_kv) return hipErrorNotSupported;
  if (scatter && (scatter->row_bytes % 4 || !scatter->k_cache || !scatter->v_cache || !scatter->block_idx ||
                  !scatter->pos_idx))
    return hipErrorInvalidValue;
  if (batch == 0) return hipSuccess;
  AttnArgs a;
  a.q = q_rot;
  a.k_pool = k_pool;
  a.v_pool = v_pool;
  a.tables = tables;
  a.ctx_lens = ctx_lens;
  a.max_blocks = max_blocks;
  a.max_ctx = max_ctx;
  a.n_blocks = n_blocks;
  a.block_size = block_size;
  a.n_head = n_head;
  a.n_head_kv = n_head_kv;
  a.scale = scale;
  a.part = part;
  const int G = n_head / n_head_kv;
  const bool ring = dtype == DT_BF16 && (head_dim == 64 || head_dim == 128);
  RingPlan plan{kSplitLen, kAttnWaves, false};
  if (ring) plan = ring_plan(max_ctx, static_cast<int64_t>(batch) * n_head_kv, head_dim, G);
  a.split_len = plan.split_len;
  a.split_major = plan.split_major;
  a.n_split = (max_ctx + a.split_len - 1) / a.split_len;  // at most attn_decode_splits(max_ctx)
  if (a.n_split > 0) {
    if (reinterpret_cast<uintptr_t>(k_pool) % 16 || reinterpret_cast<uintptr_t>(v_pool) % 16)
      return hipErrorInvalidValue;  // 16-byte loads (the entry points check this too)
    const hipError_t e = ring && head_dim == 64 ? launch_ring<64>(a, G, plan.waves, batch, s)
                         : ring                 ? launch_ring<128>(a, G, plan.waves, batch, s)
                         : dtype == DT_F32      ? launch_split_d<float>(a, head_dim, G, batch, s)
                                                : launch_split_d<bf16_t>(a, head_dim, G, batch, s);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(attn_combine_kernel, dim3(n_head + (scatter ? 2 : 0), batch), dim3(kCombineThreads), 0, s, a,
                     head_dim, k_new, v_new, dtype, out, scatter ? *scatter : KvScatterDecode{});
  return hipGetLastError();
}

hipError_t launch_qkv_rope(const float* qkv, int nsplit, int64_t split_stride, const float* bq, const float* bk,
                           const float* bv, const int64_t* positions, int batch, int nq, int nkv, int head_dim,
                           double freq_base, double freq_scale, float* q_rot, void* k_new, void* v_new, int act,
                           hipStream_t s) {
  if (batch == 0) return hipSuccess;
  const int items = (nq + nkv) / 2 + nkv;
  hipLaunchKernelGGL(qkv_rope_kernel, dim3(batch, (items + 255) / 256), dim3(256), 0, s, qkv, nsplit, split_stride, bq,
                     bk, bv, positions,
                     nq, nkv, head_dim, freq_base, freq_scale, q_rot, k_new, v_new, act);
  return hipGetLastError();
}

hipError_t launch_bias_cast(const float* y, int nsplit, int64_t split_stride, const float* bias, const void* residual,
                            void* out, int64_t rows, int n, int act, hipStream_t s) {
  const int64_t total = rows * n;
  if (total == 0) return hipSuccess;
  hipLaunchKernelGGL(bias_cast_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, s, y, nsplit,
                     split_stride, bias, residual, out, rows, n, act);
  return hipGetLastError();
}

hipError_t launch_iota(int* v, int n, int* pair, int pair0, int pair1, hipStream_t s) {
  const int blocks = n > 0 ? (n + 255) / 256 : 1;
  hipLaunchKernelGGL(iota_kernel, dim3(blocks), dim3(256), 0, s, v, n, pair, pair0, pair1);
  return hipGetLastError();
}

hipError_t launch_fill_int(int* v, int n, int value, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(fill_int_kernel, dim3((n + 255) / 256), dim3(256), 0, s, v, n, value);
  return hipGetLastError();
}

hipError_t launch_kv_gather(const void* cache, int64_t n_blocks, int block_size, int row_bytes, const int* tables,
                            int max_blocks, const int* ctx_lens, int max_ctx, int batch, void* out, hipStream_t s) {
  if (batch == 0 || max_ctx == 0 || row_bytes == 0) return hipSuccess;
  hipLaunchKernelGGL(kv_gather_kernel, dim3(max_ctx, batch), dim3(kCopyThreads), 0, s,
                     static_cast<const uint32_t*>(cache), n_blocks, block_size, row_bytes / 4, tables, max_blocks,
                     ctx_lens, max_ctx, static_cast<uint32_t*>(out));
  return hipGetLastError();
}

hipError_t launch_kv_scatter_decode(void* cache, int64_t n_blocks, int block_size, int row_bytes, const void* vals,
                                    const int* block_idx, const int* pos_idx, int batch, hipStream_t s) {
  if (batch == 0 || row_bytes == 0) return hipSuccess;
  hipLaunchKernelGGL(kv_scatter_decode_kernel, dim3(batch), dim3(kCopyThreads), 0, s, static_cast<uint32_t*>(cache),
                     n_blocks, block_size, row_bytes / 4, static_cast<const uint32_t*>(vals), block_idx, pos_idx,
                     batch);
  return hipGetLastError();
}

hipError_t launch_kv_scatter_prefill(void* cache, int64_t n_blocks, int block_size, int row_bytes, const void* vals,
                                     int seq_len, const int* tables, int max_blocks, const int* start, int batch,
                                     hipStream_t s) {
  if (batch == 0 || seq_len == 0 || row_bytes == 0) return hipSuccess;
  hipLaunchKernelGGL(kv_scatter_prefill_kernel, dim3(seq_len, batch), dim3(kCopyThreads), 0, s,
                     static_cast<uint32_t*>(cache), n_blocks, block_size, row_bytes / 4,
                     static_cast<const uint32_t*>(vals), seq_len, tables, max_blocks, start);
  return hipGetLastError();
}

}  // namespace fmoe
