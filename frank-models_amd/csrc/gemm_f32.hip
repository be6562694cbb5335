// Grouped GEMM for fp32 activations x fp32 row-major expert weights
// [E][N][K] on the fp32 matrix instruction (v_mfma_f32_16x16x4_f32: fp32
// products and sums).  The same sums as gemm_generic_kernel (mul_mat_id's
// per-assignment mat-vec, components/moe/mul_mat_id.mlir:55-94, batched per
// expert), for the shapes whose rows are 16-byte aligned with K a multiple
// of 32; the generic kernel keeps the others.
//
// Bound: at few rows per expert the weights' HBM read (each weight byte is
// used by one block per 64 rows), above about 40 rows per expert the fp32
// matrix rate (157 TFLOP/s dense, 1/16 of bf16).  The SIMT kernel reached
// neither: 4-byte loads, a transposing LDS store per value and a barrier
// pair per 16 inputs with no load in flight across them.  Measured
// (DeepSeek-V2-Lite in fp32, 64 experts x 2048 x 1408, top-6): 500 tokens
// gate/up 1607 -> 405-440 us (86 TFLOP/s, 3.6 TB/s) and down 1059 -> 202-224
// us; 64 tokens, whole block, 378 us (5.9 TB/s of weights).  Other shapes, whole
// block, SIMT kernel -> this one (hidden x ff, experts, top-k): 512 x 1792, 8, 2
// with 1 / 40 / 2000 tokens 300 / 347 / 857 -> 40 / 51 / 270 us; 2048 x 768, 128, 8
// with 1 / 100 / 500 tokens 619 / 3171 / 4439 -> 60 / 217 / 600; 4096 x 14336, 8, 2
// with 1 / 64 tokens 2842 / 6066 -> 328 / 1033.  Counters at 500 tokens: the
// matrix cores are busy 66% (gate/up) and 60% (down) of the time, 15% of it on
// padding rows, beside 3.7 TB/s from HBM: neither bound is reached alone.
//
// Block: 256 threads, a tile of BM assignment rows x 32 * WN weight rows,
// stages of KS inputs through a ring in LDS filled by global_load_lds (16
// bytes per lane), one barrier per stage, kRing - 1 stages in flight.  The
// four waves are WN column slices x 4 / WN slices of a stage's 16-input
// steps (summed through LDS at the end), so narrow tiles keep all four
// matrix cores fed.  A wave holds two 16-row weight fragments (gate and up
// of the same columns, or two neighbouring column groups of a single set)
// against all the tile's 16-row groups, and skips groups past the expert's
// rows: the K loop is compiled for each count of them.
//
// Operands: lane l of a fragment reads the 16 bytes of row l % 16 at inputs
// 4 (l / 16) of a 16-input step, and MFMA j takes element j, so its four
// inputs are j, 4 + j, 8 + j, 12 + j of the step for both operands.  LDS
// rows are KS * 4 bytes with their 16-byte chunks at chunk ^ swizzle(row),
// which spreads the 16 rows of a read over all 64 banks.
#include "common.h"
#include "launch.h"

namespace fmoe {
namespace {

constexpr int kThreads = 256;

// WN column slices, BM assignment rows per tile (32 or 64).  Ring depth: as
// many blocks per CU as the stages leave room for beat a deeper ring at 32
// rows (DeepSeek-V2-Lite in fp32, 16 tokens: 365 us with 2 stages and four
// blocks per CU, 375 with 3 and two; 1 token: 70 us with 3 stages of a
// 32-column tile, 88 with 4) and lose to it at 64 (500 tokens: 622 us with 3
// stages, 640 with 2).
template <int WN, int BM>
struct Cfg {
  static constexpr int kRing = BM == 32 && WN == 4 ? 2 : 3;  // LDS stages
  static constexpr int kWK = 4 / WN;             // waves over a stage's steps
  static constexpr int kKS = WN == 1 ? 64 : 32;  // inputs per stage
  static constexpr int kRowB = kKS * 4;          // bytes per LDS row
  static constexpr int kRB = 32 * WN;            // weight rows per tile
  static constexpr int kRowsPerLoad = 1024 / kRowB;
  static constexpr int kABytes = BM * kRowB;
  static constexpr int kStage = kABytes + kRB * kRowB;
  static constexpr int kLB = kRB / kRowsPerLoad / 4;  // weight loads per wave per stage
  static constexpr int kSteps = kKS / 16 / kWK;       // 16-input steps per wave per stage
  static constexpr int kLds = kRing * kStage;
  static constexpr int kBlocks = 160 * 1024 / kLds < 5 ? 160 * 1024 / kLds : 5;  // per CU
  static_assert(kLB >= 1 && kSteps >= 1, "every wave loads and computes");
  static_assert(kABytes >= 4096, "one load per wave fits the A part");
};

// Chunk position of logical 16-byte chunk c of a row: 128-byte rows pair up
// to the 256 bytes of a bank cycle, 256-byte rows fill one.
template <int KS>
__device__ __forceinline__ int swz(int row, int c) {
  return KS == 64 ? c ^ (row & 15) : c ^ ((row >> 1) & 7);
}

struct F32Tile {
  int expert, row0, rows, col;
};

// Number of bm-row tiles of the grouping (every lane gets the count).
__device__ __forceinline__ int count_tiles(const int* __restrict__ offsets, int n_expert, int bm) {
  const int lane = threadIdx.x & (kWave - 1);
  int n = 0;
  for (int c = 0; c < n_expert; c += kWave) {
    const int e = c + lane;
    n += e < n_expert ? (offsets[e + 1] - offsets[e] + bm - 1) / bm : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, kWave);
  return n;
}

// The block's tile: hardware block b runs on XCD b % 8, and each XCD takes a
// contiguous range of the (row tile, column tile) list in row-tile-major
// order of groups of 4 column tiles, so the row tiles of one expert that
// share weight rows run side by side on one L2.
__device__ __forceinline__ bool find_block(const GroupedGemmArgs& g, int bm, int n_col, F32Tile* t) {
  const int n_row = g.offsets ? count_tiles(g.offsets, g.n_expert, bm) : (g.n_assign + bm - 1) / bm;
  const int total = n_row * n_col;
  const int per = (total + 7) / 8;
  const int b = blockIdx.x;
  if (b / 8 >= per) return false;
  const int logical = (b % 8) * per + b / 8;
  if (logical >= total) return false;
  const int span = 4 * n_row;
  const int group = logical / span;
  const int within = logical - group * span;
  const int cols = min(4, n_col - 4 * group);
  const int row = within / cols;
  t->col = 4 * group + within - row * cols;
  if (!g.offsets) {
    t->expert = 0;
    t->row0 = row * bm;
    t->rows = min(bm, g.n_assign - row * bm);
    return true;
  }
  TileInfo ti;
  if (!find_tile(g.offsets, g.n_expert, bm, row, &ti)) return false;
  t->expert = ti.expert;
  t->row0 = ti.row0;
  t->rows = ti.rows;
  return true;
}

// One wave's loads of stage st into its ring buffer.
template <int WN, int BM, int LA, bool NT>
__device__ __forceinline__ void issue_stage(const float* const* a_src, const float* const* b_src, int st,
                                            unsigned char* lds, int wave) {
  using C = Cfg<WN, BM>;
  // plain variables: the builtin's operands must not depend on the template
  unsigned char* a_dst = lds + (st % C::kRing) * C::kStage + wave * 1024;
  unsigned char* b_dst = a_dst + C::kABytes;
  const int ofs = st * C::kKS;
#pragma unroll
  for (int i = 0; i < LA; ++i) __builtin_amdgcn_global_load_lds(a_src[i] + ofs, a_dst + i * 4096, 16, 0, 0);
#pragma unroll
  for (int i = 0; i < C::kLB; ++i) {
    if (NT)
      __builtin_amdgcn_global_load_lds(b_src[i] + ofs, b_dst + i * 4096, 16, 0, kNonTemporal);
    else
      __builtin_amdgcn_global_load_lds(b_src[i] + ofs, b_dst + i * 4096, 16, 0, 0);
  }
}

// The K loop over stages [0, n_st) for MG 16-row groups.  a_src / b_src:
// this lane's source of each of its wave's loads at stage 0; load i of the
// wave covers LDS rows (wave + 4 i) * kRowsPerLoad of the A or weight part.
template <int WN, int BM, bool NT, int MG>
__device__ __forceinline__ void k_loop(const float* const* a_src, const float* const* b_src,
                                       int n_st, unsigned char* lds, f32x4_t (*acc)[BM / 16]) {
  using C = Cfg<WN, BM>;
  // Loads that cover the MG groups' rows, rounded up to whole rounds of the
  // four waves (rows past the tile re-read a valid row).
  constexpr int kLA = (16 * MG / C::kRowsPerLoad + 3) / 4;
  constexpr int kL = kLA + C::kLB;
  static_assert((C::kRing - 2) * kL <= 63, "loads in flight within the vmcnt range");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave % WN, wk = wave / WN;
  const int r = lane & 15, q = lane >> 4;

  // Stage st is visible to the block after each wave has waited for its own
  // loads of it and the barrier; the barrier also means every wave has
  // finished stage st - 1, whose buffer stage st + kRing - 1 then refills.
  for (int st = 0; st < C::kRing - 1 && st < n_st; ++st) issue_stage<WN, BM, kLA, NT>(a_src, b_src, st, lds, wave);
  for (int st = 0; st < n_st; ++st) {
    if (st + C::kRing - 1 <= n_st)
      __builtin_amdgcn_s_waitcnt(wait_vm((C::kRing - 2) * kL, true));
    else
      __builtin_amdgcn_s_waitcnt(wait_vm(0, true));
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (st + C::kRing - 1 < n_st) issue_stage<WN, BM, kLA, NT>(a_src, b_src, st + C::kRing - 1, lds, wave);
    const unsigned char* as = lds + (st % C::kRing) * C::kStage;
    const unsigned char* bs = as + C::kABytes;
#pragma unroll
    for (int s = 0; s < C::kSteps; ++s) {
      const int c = 4 * (wk + s * C::kWK) + q;
      const int pos = swz<C::kKS>(r, c) * 16;  // the same for rows 16 apart
      f32x4_t w[2], a[MG];
#pragma unroll
      for (int f = 0; f < 2; ++f)
        w[f] = *reinterpret_cast<const f32x4_t*>(bs + (wn * 32 + f * 16 + r) * C::kRowB + pos);
#pragma unroll
      for (int m = 0; m < MG; ++m) a[m] = *reinterpret_cast<const f32x4_t*>(as + (m * 16 + r) * C::kRowB + pos);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < MG; ++m)
#pragma unroll
          for (int f = 0; f < 2; ++f)
            acc[f][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[f][j], a[m][j], acc[f][m], 0, 0, 0);
    }
  }
}

template <int WN, int BM, int EPI, bool NT>
__global__ __launch_bounds__(kThreads, (Cfg<WN, BM>::kBlocks)) void gemm_f32_kernel(GroupedGemmArgs g, int n_col) {
  using C = Cfg<WN, BM>;
  constexpr bool kTwo = EPI == EPI_SWIGLU;              // two weight sets
  constexpr int kLAmax = C::kABytes / 4096;             // token row loads per wave per stage, at most
  constexpr int kMG = BM / 16;                          // 16-row groups per tile
  constexpr int kCols = kTwo ? C::kRB / 2 : C::kRB;     // output columns per tile
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  F32Tile t;
  if (!find_block(g, BM, n_col, &t)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t N = g.N, K = g.K;
  const int64_t n0 = static_cast<int64_t>(t.col) * kCols;

  // Weight row w of the tile: slice w / 32, fragment (w % 32) / 16, row
  // w % 16.  Columns past N read the last row (never stored).
  const int lrow = lane / (64 / C::kRowsPerLoad);   // row within a load
  const int lpos = lane % (64 / C::kRowsPerLoad);   // chunk position within the row
  const int n_st_all = static_cast<int>(K / C::kKS);
  const int kz = blockIdx.y, nz = gridDim.y;
  const int st0 = static_cast<int>(static_cast<int64_t>(kz) * n_st_all / nz);
  const int n_st = static_cast<int>(static_cast<int64_t>(kz + 1) * n_st_all / nz) - st0;
  const float* b_src[C::kLB];
#pragma unroll
  for (int i = 0; i < C::kLB; ++i) {
    const int w = (wave + 4 * i) * C::kRowsPerLoad + lrow;
    const int f = (w >> 4) & 1;
    const int64_t n = n0 + (kTwo ? (w >> 5) * 16 : (w >> 5) * 32 + f * 16) + (w & 15);
    const float* base = static_cast<const float*>(kTwo && f ? g.w1 : g.w0);
    b_src[i] = base + (static_cast<int64_t>(t.expert) * N + (n < N ? n : N - 1)) * K +
               static_cast<int64_t>(st0) * C::kKS + swz<C::kKS>(w, lpos) * 4;
  }
  const float* a_src[kLAmax];
#pragma unroll
  for (int i = 0; i < kLAmax; ++i) {
    const int ar = (wave + 4 * i) * C::kRowsPerLoad + lrow;
    const int p = t.row0 + (ar < t.rows ? ar : 0);
    int64_t row = p;
    if (g.a_mode == A_GATHER_TOKEN)
      row = g.order[p] % g.n_tokens;
    else if (g.a_mode == A_GATHER_FLAT)
      row = g.order[p];
    a_src[i] = static_cast<const float*>(g.a) + row * g.lda + static_cast<int64_t>(st0) * C::kKS +
               swz<C::kKS>(ar, lpos) * 4;
  }

  f32x4_t acc[2][kMG];
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int m = 0; m < kMG; ++m) acc[f][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int mg = (t.rows + 15) / 16;
  if (mg == 1)
    k_loop<WN, BM, NT, 1>(a_src, b_src, n_st, lds, acc);
  else if (BM == 32 || mg == 2)
    k_loop<WN, BM, NT, 2>(a_src, b_src, n_st, lds, acc);
  else if (mg == 3)
    k_loop<WN, BM, NT, BM == 32 ? 2 : 3>(a_src, b_src, n_st, lds, acc);
  else
    k_loop<WN, BM, NT, BM == 32 ? 2 : 4>(a_src, b_src, n_st, lds, acc);

  const int wn = wave % WN, wk = wave / WN;
  if (C::kWK > 1) {
    // Partial sums of the step slices, added in slice order.
    f32x4_t* part = reinterpret_cast<f32x4_t*>(lds);
    __syncthreads();
    if (wk > 0) {
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int m = 0; m < kMG; ++m)
          if (m < mg) part[((((wk - 1) * WN + wn) * 2 + f) * kMG + m) * kWave + lane] = acc[f][m];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int w = 1; w < C::kWK; ++w)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int m = 0; m < kMG; ++m)
          if (m < mg) acc[f][m] += part[((((w - 1) * WN + wn) * 2 + f) * kMG + m) * kWave + lane];
  }

  // Lane l holds row l % 16 of each group, columns 4 (l / 16) .. +4 of each
  // fragment.
  float* out = static_cast<float*>(g.out) + kz * g.split_stride;
#pragma unroll
  for (int m = 0; m < kMG; ++m) {
    const int r = m * 16 + (lane & 15);
    if (r >= t.rows) continue;
    const int p = t.row0 + r;
    const int c4 = 4 * (lane >> 4);
    if (EPI == EPI_SWIGLU) {
      const int64_t n = n0 + wn * 16 + c4;
      if (n >= N) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float u = acc[1][m][i];
        // gate * silu(up), silu(u) = u / (1 + exp(-u))  (swiglu.mlir:37-47)
        v[i] = acc[0][m][i] * (u / (1.f + expf(-u)));
      }
      *reinterpret_cast<float4*>(out + p * g.ldo + n) = float4{v[0], v[1], v[2], v[3]};
    } else {
      const int64_t orow = g.order ? g.order[p] : p;
      const float w = EPI == EPI_SCATTER_WEIGHTED ? g.route_w[orow] : 1.f;
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int64_t n = n0 + wn * 32 + f * 16 + c4;
        if (n >= N) continue;
        const f32x4_t v = acc[f][m];
        *reinterpret_cast<float4*>(out + orow * g.ldo + n) = float4{v[0] * w, v[1] * w, v[2] * w, v[3] * w};
      }
    }
  }
}

// Column tiles of a tile width: 16 columns per slice and set with two sets,
// 32 with one.
int col_tiles(const GroupedGemmArgs& g, int wn) {
  const int64_t cols = (g.epi == EPI_SWIGLU ? 16 : 32) * wn;
  return static_cast<int>((g.N + cols - 1) / cols);
}

// (The lines of pick_bm, pick_wn and launch_tile are DeepSeek-V2-Lite's.)
// Rows per tile: 32 up to 20 rows per expert on average, where a narrower
// token part leaves LDS for more blocks, else 64, which streams the weights
// once for more rows.  Measured (DeepSeek-V2-Lite in fp32, whole block,
// 32-row against 64-row tiles): 19 rows 447 against 452 us, 28 rows 503
// against 494, 47 rows 715 against 622.
int pick_bm(const GroupedGemmArgs& g) {
  const int64_t n = g.n_assign;
  return g.offsets ? (n <= 20ll * g.n_expert ? 32 : 64) : (n <= 32 ? 32 : 64);
}

// Row tiles that hold rows, about: every expert of a small batch, and one
// more tile per bm rows.
int64_t busy_tiles(const GroupedGemmArgs& g, int bm) {
  const int64_t n = g.n_assign;
  return g.offsets ? (n < g.n_expert ? n : g.n_expert) + n / bm : (n + bm - 1) / bm;
}

// Tile width: the widest that still gives the GPU two blocks per CU.
int pick_wn(const GroupedGemmArgs& g, int bm) {
  for (int wn = 4; wn > 1; wn /= 2)
    if (busy_tiles(g, bm) * col_tiles(g, wn) * g.ksplit >= 512) return wn;
  return g.K % 64 == 0 ? 1 : 2;
}

template <int WN, int BM, int EPI, bool NT>
hipError_t launch_policy(const GroupedGemmArgs& g, hipStream_t s) {
  using C = Cfg<WN, BM>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_f32_kernel<WN, BM, EPI, NT>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds);
  (void)attr;
  const int n_col = col_tiles(g, WN);
  const int64_t rows = g.offsets ? max_row_tiles(g.n_assign, g.n_expert, BM) : (g.n_assign + BM - 1) / BM;
  const int64_t blocks = (rows * n_col + 7) / 8 * 8;  // whole rounds of the 8 XCDs
  hipLaunchKernelGGL((gemm_f32_kernel<WN, BM, EPI, NT>),
                     dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(g.ksplit)), dim3(kThreads), C::kLds, s,
                     g, n_col);
  return hipGetLastError();
}

// The weights go non-temporally up to 64 rows per expert on average, where an
// expert is mostly one row tile; beyond, its row tiles share them in L2.
// Measured (DeepSeek-V2-Lite in fp32, whole block, default -> non-temporal):
// 6 rows 422 -> 378 us, 19 rows 451 -> 408, 47 rows 616 -> 608, 94 rows 1165 ->
// 1185, 188 rows 1916 -> 1997.
template <int WN, int BM, int EPI>
hipError_t launch_tile(const GroupedGemmArgs& g, hipStream_t s) {
  if (g.n_assign <= 64ll * g.n_expert) return launch_policy<WN, BM, EPI, true>(g, s);
  return launch_policy<WN, BM, EPI, false>(g, s);
}

template <int EPI>
hipError_t launch_epi(const GroupedGemmArgs& g, hipStream_t s) {
  const int bm = pick_bm(g);
  switch (pick_wn(g, bm)) {
    case 4: return bm == 32 ? launch_tile<4, 32, EPI>(g, s) : launch_tile<4, 64, EPI>(g, s);
    case 2: return bm == 32 ? launch_tile<2, 32, EPI>(g, s) : launch_tile<2, 64, EPI>(g, s);
    default: return bm == 32 ? launch_tile<1, 32, EPI>(g, s) : launch_tile<1, 64, EPI>(g, s);
  }
}

}  // namespace

bool gemm_f32_supported(const GroupedGemmArgs& g) {
  if (g.act_dtype != DT_F32 || g.w_dtype != DT_F32 || g.out_dtype != DT_F32 || g.epi < 0 ||
      g.epi > EPI_SCATTER_WEIGHTED || g.a_kb_rows || g.out_kb_rows)
    return false;
  if (g.K <= 0 || g.K % 32 || g.N % 4 || g.lda % 4 || g.ldo % 4) return false;
  // no grouping arrays: one expert's rows in order
  if (!g.offsets != !g.order) return false;
  if (!g.offsets && (g.n_expert != 1 || g.a_mode != A_DIRECT || g.epi != EPI_SCATTER)) return false;
  if (g.ksplit > 1 && (g.epi != EPI_SCATTER || g.split_stride <= 0 || g.split_stride % 4 || g.ksplit > 64)) return false;
  auto al16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (!al16(g.a) || !al16(g.w0) || !al16(g.out) || (g.epi == EPI_SWIGLU && !al16(g.w1))) return false;
  // the grid's block count
  const int64_t rows = g.offsets ? max_row_tiles(g.n_assign, g.n_expert, 32) : (g.n_assign + 31) / 32;
  return rows * ((g.N + 15) / 16) < (1ll << 31) - 8;
}

hipError_t launch_gemm_f32(const GroupedGemmArgs& g, hipStream_t s) {
  if (!gemm_f32_supported(g)) return hipErrorNotSupported;
  if (g.n_assign == 0 || g.N == 0) return hipSuccess;
  if (g.epi == EPI_SWIGLU) return launch_epi<EPI_SWIGLU>(g, s);
  if (g.epi == EPI_SCATTER) return launch_epi<EPI_SCATTER>(g, s);
  return launch_epi<EPI_SCATTER_WEIGHTED>(g, s);
}

}  // namespace fmoe
