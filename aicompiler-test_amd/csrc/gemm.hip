// Prompt GEMMs for gfx950: y[m, n] = x[m, k] w[n, k]^T with fp16 operands and
// fp32 accumulation, the linear layers of a chunked-prefill stage
// (emitTiledGEMM, DecodeGEMVMetalEmitter.cpp:134-169; prefillChunked,
// DecoderLLMExecutor.cpp:982-1034).
#include "tmc_abi.hpp"
#include "tmc_device.hpp"

#include <algorithm>
#include <cmath>

namespace tmc {
namespace {

// ------------------------------------------------------------ prompt GEMM
// y[m, n] = x[m, k] w[n, k]^T with fp16 operands and fp32 accumulation on
// v_mfma_f32_16x16x32_f16.  Both operands are k-contiguous rows, which is the
// MFMA operand order: lane (i, g) of a 16 x 32 fragment holds row i, k
// 8g ... 8g + 7.  w is the first operand, so a lane ends up with four
// consecutive outputs of one row of y and stores them together.
//
// Block: WM x WN waves over a BM x BN output tile, FA x FB fragments of 16 x
// 16 per wave.  k advances in stages of 64: a tile row's 64 halves are one
// LDS row of eight 16-byte chunks, chunk c at slot c ^ ((row / 2) % 8), so
// the 16 rows of an operand read fall on 16 distinct bank groups.  Stages
// move from memory to LDS by buffer loads with the LDS flag (no staging
// registers; a lane fetches the chunk that belongs into its slot, a row's
// 128 bytes staying one line); an offset past the operand's bytes writes
// zeros, so ragged m, n and k need no branches.
//
// Pipeline, NS stages in LDS, two fragment sets in registers: the MFMAs of
// half a stage run while the other half's fragments are read.  One barrier
// per stage, between its halves: there every wave has read all of stage st,
// whose buffer takes stage st + NS, and stage st + 1 has landed.  The wait
// counts loads, so later stages stay in flight across it (__syncthreads()
// would wait for all of them).  LDS reads and stage loads are spread over
// the MFMAs (1131 -> 1190 TFLOP/s on the 1024 x 4096 x 32000 LM head).
//
// What bounds the large tiles is the LDS: a 256 x 256 x 64 stage reads 192 KiB
// of fragments and writes 64 KiB at 128 bytes a clock, as long as its MFMAs
// take.  MI355X, m 2048, k 4096: 256 x 256 tiles in whole rounds of 256
// reach 1235 TFLOP/s (register-staged loads and __syncthreads(): 1016).
//
// Split K (SPLIT): block (tile, split s) multiplies k in [s * k_chunk,
// (s + 1) * k_chunk) and writes fp32 partials y[s][m][n]; gemm_reduce_kernel
// adds them in split order.
//
// Tiles are dealt XCD by XCD: blocks b, b + 8, b + 16, ... run on one XCD
// and take consecutive tiles, which walk the m tiles of one n tile first, so
// a weight slice is fetched from HBM once into that XCD's L2.
constexpr int kStageK = 64;  // k per stage: LDS rows of 64 halves (128 bytes)

template <typename OutT, bool SPLIT, int WM, int WN, int FA, int FB, int EU, int NS>
__global__ __launch_bounds__(WM * WN * kWave) __attribute__((amdgpu_waves_per_eu(EU, EU))) void gemm_tile_kernel(
    const half_t* __restrict__ x, const half_t* __restrict__ w, OutT* __restrict__ y, int m,
    int n, int k, int m_tiles, int tiles, int k_chunk, unsigned x_bytes, unsigned w_bytes) {
  constexpr int W = WM * WN, BM = WM * FA * 16, BN = WN * FB * 16;
  constexpr int QA = (BM / 8 + W - 1) / W, QB = (BN / 8 + W - 1) / W;  // 1 KiB loads per wave
  static_assert(W % 2 == 0, "a wave's loads share their swizzle");
  __shared__ __attribute__((aligned(16))) half_t lds[NS][(BM + BN) * kStageK];
  const int per_xcd = (int)(gridDim.x / 8u);
  const int unit = (int)(blockIdx.x % 8u) * per_xcd + (int)(blockIdx.x / 8u);
  const int splits = SPLIT ? (k + k_chunk - 1) / k_chunk : 1;
  if (unit >= tiles * splits) return;
  const int t = unit % tiles;
  const int k_begin = SPLIT ? (unit / tiles) * k_chunk : 0;
  const int k_end = SPLIT ? min(k, k_begin + k_chunk) : k;
  const int m0 = (t % m_tiles) * BM;
  const int n0 = (t / m_tiles) * BN;
  const int lane = (int)threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWave);
  const int i = lane & 15, g = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  const __amdgpu_buffer_rsrc_t rx = buffer_resource(x, x_bytes);
  const __amdgpu_buffer_rsrc_t rw = buffer_resource(w, w_bytes);

  // load q of this wave: tile rows 8 (q W + wave) .. + 7; lane l moves the
  // chunk that belongs into slot l % 8 of row l / 8
  const int chunk = (lane & 7) ^ ((4 * (wave & 1) + (lane >> 4)) & 7);
  const int row = 8 * wave + (lane >> 3);
  const unsigned step = (unsigned)(8 * W) * (unsigned)k * 2u;
  unsigned at_x = (((unsigned)(m0 + row)) * (unsigned)k + (unsigned)(k_begin + 8 * chunk)) * 2u;
  unsigned at_w = (((unsigned)(n0 + row)) * (unsigned)k + (unsigned)(k_begin + 8 * chunk)) * 2u;
  const int stages = (k_end - k_begin + kStageK - 1) / kStageK;
  int kk = k_begin + 8 * chunk;
  auto load_stage = [&](half_t* buf) {
    const bool in = kk < k_end;
    typedef __attribute__((address_space(3))) void lds_void;
#pragma unroll
    for (int q = 0; q < QA; ++q)
      if (BM % (8 * W) == 0 || q * W + wave < BM / 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rx, (lds_void*)(buf + (q * W + wave) * 8 * kStageK), 16,
          in ? (int)(at_x + (unsigned)q * step) : (int)kBufferAbsent, 0, 0, 0);
#pragma unroll
    for (int q = 0; q < QB; ++q)
      if (BN % (8 * W) == 0 || q * W + wave < BN / 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rw, (lds_void*)(buf + BM * kStageK + (q * W + wave) * 8 * kStageK), 16,
          in ? (int)(at_w + (unsigned)q * step) : (int)kBufferAbsent, 0, 0, 0);
    kk += kStageK;
    at_x += 2 * kStageK;
    at_w += 2 * kStageK;
  };

  const int swz = (i >> 1) & 7;
  const int off_x = (wm * FA * 16 + i) * kStageK, off_w = (BM + wn * FB * 16 + i) * kStageK;
  const int slot[2] = {8 * (g ^ swz), 8 * ((4 + g) ^ swz)};
  struct Frags {
    h8 a[FA], b[FB];
  };
  auto read = [&](Frags& f, const half_t* buf, int s) {
#pragma unroll
    for (int a = 0; a < FA; ++a)
      f.a[a] = *reinterpret_cast<const h8*>(buf + off_x + a * 16 * kStageK + slot[s]);
#pragma unroll
    for (int b = 0; b < FB; ++b)
      f.b[b] = *reinterpret_cast<const h8*>(buf + off_w + b * 16 * kStageK + slot[s]);
  };
  f4 acc[FA][FB];
#pragma unroll
  for (int a = 0; a < FA; ++a)
#pragma unroll
    for (int b = 0; b < FB; ++b) acc[a][b] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int a = 0; a < FA; ++a)
#pragma unroll
      for (int b = 0; b < FB; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[b], f.a[a], acc[a][b], 0, 0, 0);
  };
  // every wave's outstanding LDS reads are done, and the oldest stage in flight
  auto stage_barrier = [&]() {
    constexpr int N = (NS - 2) * (QA + QB);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4 << 14));  // vmcnt(N) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
  };
  static_assert(NS == 2 || (BM % (8 * W) == 0 && BN % (8 * W) == 0), "waves issue the same loads");

  Frags even, odd;
#pragma unroll
  for (int q = 0; q < NS - 1; ++q) load_stage(lds[q]);
  stage_barrier();
  load_stage(lds[NS - 1]);
  read(even, lds[0], 0);
  // schedule: one LDS read (and one stage load) before every few MFMAs
  auto interleave = [&](bool loads) {
    constexpr int R = FA + FB, M = FA * FB;
#pragma unroll
    for (int q = 0; q < R; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, M / R, 0);
      if (loads && q < QA + QB) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
    }
  };
  auto body = [&](half_t* cur, half_t* next) {
    read(odd, cur, 1);
    multiply(even);
    interleave(false);
    stage_barrier();
    load_stage(cur);
    read(even, next, 0);
    multiply(odd);
    interleave(true);
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int st = 0; st < stages; st += NS) {
#pragma unroll
    for (int q = 0; q < NS; ++q) body(lds[q], lds[(q + 1) % NS]);
  }
  // LDS loads still in flight must land before the block's LDS is reused
  __builtin_amdgcn_s_waitcnt(0x0070);

  // acc[a][b][r] = y[m0 + 16 (wm FA + a) + i][n0 + 16 (wn FB + b) + 4g + r]
  typedef OutT o4 __attribute__((ext_vector_type(4)));
  const bool whole = n % 4 == 0 && reinterpret_cast<uintptr_t>(y) % sizeof(o4) == 0;
#pragma unroll
  for (int a = 0; a < FA; ++a) {
    const int r = m0 + 16 * (wm * FA + a) + i;
    if (r >= m) continue;
#pragma unroll
    for (int b = 0; b < FB; ++b) {
      const int c = n0 + 16 * (wn * FB + b) + 4 * g;
      OutT* out = y + ((SPLIT ? (size_t)(unit / tiles) * m : 0) + (size_t)r) * n + c;
      if (whole) {
        o4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = from_float<OutT>(acc[a][b][e]);
        if (c < n) *reinterpret_cast<o4*>(out) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < n) out[e] = from_float<OutT>(acc[a][b][e]);
      }
    }
  }
}

// Partials summed in split order, V consecutive outputs per thread.
template <typename OutT, int V>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const float* __restrict__ partial,
                                                         OutT* __restrict__ y, size_t count,
                                                         int splits) {
  typedef float fv __attribute__((ext_vector_type(V)));
  typedef OutT ov __attribute__((ext_vector_type(V)));
  for (size_t e = ((size_t)blockIdx.x * 256 + threadIdx.x) * V; e < count;
       e += (size_t)gridDim.x * 256 * V) {
    fv sum = *reinterpret_cast<const fv*>(partial + e);
#pragma unroll 4
    for (int s = 1; s < splits; ++s)
      sum += *reinterpret_cast<const fv*>(partial + (size_t)s * count + e);
    ov out;
#pragma unroll
    for (int v = 0; v < V; ++v) out[v] = from_float<OutT>(sum[v]);
    *reinterpret_cast<ov*>(y + e) = out;
  }
}

template <typename OutT>
int launch_reduce(const float* partial, OutT* y, size_t count, int splits, hipStream_t stream) {
  if (count % 4 == 0 && aligned16(y))
    hipLaunchKernelGGL((gemm_reduce_kernel<OutT, 4>),
                       dim3((unsigned)std::min<size_t>((count + 1023) / 1024, 8192)), dim3(256), 0,
                       stream, partial, y, count, splits);
  else
    hipLaunchKernelGGL((gemm_reduce_kernel<OutT, 1>),
                       dim3((unsigned)std::min<size_t>((count + 255) / 256, 8192)), dim3(256), 0,
                       stream, partial, y, count, splits);
  return check_launch("gemm_reduce_kernel");
}

struct TilePlan {
  int bm, bn, stages, splits;
};

template <typename OutT, bool SPLIT, int WM, int WN, int FA, int FB, int EU, int NS>
int launch_tile(const half_t* x, const half_t* w, OutT* y, int64_t m, int64_t k, int64_t n,
                int64_t tiles, int m_tiles, int k_chunk, hipStream_t stream) {
  const int64_t units = tiles * (SPLIT ? (k + k_chunk - 1) / k_chunk : 1);
  const unsigned blocks = (unsigned)((units + 7) / 8 * 8);
  hipLaunchKernelGGL((gemm_tile_kernel<OutT, SPLIT, WM, WN, FA, FB, EU, NS>), dim3(blocks),
                     dim3(WM * WN * kWave), 0, stream, x, w, y, (int)m, (int)n, (int)k, m_tiles,
                     (int)tiles, k_chunk, (unsigned)(m * k * 2), (unsigned)(n * k * 2));
  return check_launch("gemm_tile_kernel");
}

template <typename OutT, bool SPLIT>
int launch_plan(const TilePlan& plan, const half_t* x, const half_t* w, OutT* y, int64_t m,
                int64_t k, int64_t n, int k_chunk, hipStream_t stream) {
  const int m_tiles = (int)((m + plan.bm - 1) / plan.bm);
  const int64_t tiles = (int64_t)m_tiles * ((n + plan.bn - 1) / plan.bn);
  TMC_REQUIRE(tiles < (1LL << 26), "Prompt GEMM: too many tiles.");
#define TMC_TILE(WM, WN, FA, FB, EU, NS) \
  return launch_tile<OutT, SPLIT, WM, WN, FA, FB, EU, NS>(x, w, y, m, k, n, tiles, m_tiles, k_chunk, stream)
  if (plan.bm == 64) TMC_TILE(2, 2, 2, 4, 1, 4);
  if (plan.bm == 128) {
    if (plan.stages == 2) TMC_TILE(2, 2, 4, 4, 2, 2);
    TMC_TILE(2, 2, 4, 4, 1, 4);
  }
  switch (plan.bn) {
  case 160: TMC_TILE(4, 2, 4, 5, 2, 2);
  case 192: TMC_TILE(4, 2, 4, 6, 2, 2);
  default: TMC_TILE(2, 4, 8, 4, 2, 2);
  }
#undef TMC_TILE
}

// Tile and split of a launch: the least estimated time over the tiles and
// splits below.  A block's time is 2.6 us plus its stages times the tile's
// time per stage, measured on MI355X with one block on a CU and, for the
// tile of which two fit, with two; blocks beyond one (or two) per CU run in
// further rounds.  A split adds the reduction: 3.9 us and 2.8 us per million
// partials.  The figures are a fit to 2000 launches (40 shapes, m 16-2048, k
// 1000-11008, n 2048-12288, every tile and split); its choices are within 1%
// of the best in the middle and 24% at worst (a 256 x 128 tile takes what two
// 128 x 128 tiles on one CU take, 1.024 us, and is never chosen: not built),
// and 1.02 to 1.75 times as fast
// as 128 x 128 and 256 x 256 tiles chosen by their count (1.31 in the mean):
// 2048 x 4096 x 12288 240 -> 184 us (256 x 192: two whole rounds where 256 x
// 256 leaves half of the second idle), 1024 x 4096 x 4096 57 -> 40 (four
// stages in flight), 200 x 4096 x 12288 53 -> 39.
TilePlan tile_plan(int64_t m, int64_t k, int64_t n, size_t workspace_bytes) {
  struct Tile {
    int bm, bn, stages;
    double one, two;  // us per stage: one block per CU, two (0: only one fits)
  };
  static constexpr Tile kTiles[] = {
      {64, 128, 4, 0.405, 0},  {128, 128, 2, 0.787, 1.024}, {128, 128, 4, 0.571, 0},
      {256, 160, 2, 1.108, 0}, {256, 192, 2, 1.236, 0},     {256, 256, 2, 1.497, 0}};
  static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8};
  TilePlan best{256, 256, 2, 1};
  double least = 1e30;
  for (const Tile& t : kTiles)
    for (const int splits : kSplits) {
      if (splits > 1 && (k / splits < 256 || (uint64_t)splits * m * n * 4 > workspace_bytes)) break;
      const double blocks =
          (double)((m + t.bm - 1) / t.bm) * (double)((n + t.bn - 1) / t.bn) * splits;
      const double stages = (double)(((k + splits - 1) / splits + kStageK - 1) / kStageK);
      const double per_cu = std::ceil(blocks / 256.0);
      const double alone = stages * t.one + 2.6;
      double time = per_cu * alone;
      if (t.two > 0.0) {
        const double pairs = std::floor(per_cu / 2.0);
        time = pairs * (stages * t.two + 2.6) + (per_cu - 2.0 * pairs) * alone;
      }
      if (splits > 1) time += 3.9 + 2.8e-6 * (splits + 0.5) * (double)m * (double)n;
      if (time < least) {
        least = time;
        best = {t.bm, t.bn, t.stages, splits};
      }
    }
  return best;
}

// k per split, in whole stages
int64_t split_length(int64_t k, int splits) {
  return ((k + splits - 1) / splits + kStageK - 1) / kStageK * kStageK;
}

int launch_gemm(const half_t* x, const half_t* w, void* y, int out_dtype, int64_t m, int64_t k,
                int64_t n, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  const uint64_t xb = (uint64_t)m * k * 2, wb = (uint64_t)n * k * 2;
  TMC_REQUIRE(xb < kBufferAbsent && wb < kBufferAbsent,
              "Prompt GEMM: each operand must stay below 4 GiB.");
  TMC_REQUIRE(k % 8 == 0, "Prompt GEMM: k must be a multiple of 8.");
  TMC_REQUIRE(aligned16(x) && aligned16(w), "Prompt GEMM: x and w must be 16-byte aligned.");
  const TilePlan plan = tile_plan(m, k, n, workspace ? workspace_bytes : 0);
  const int k_chunk = (int)split_length(k, plan.splits);
  const int used = (int)((k + k_chunk - 1) / k_chunk);
  if (used > 1) {
    float* partial = static_cast<float*>(workspace);
    if (launch_plan<float, true>(plan, x, w, partial, m, k, n, k_chunk, stream)) return 1;
    const size_t count = (size_t)m * n;
    if (out_dtype == TMC_F32)
      return launch_reduce(partial, static_cast<float*>(y), count, used, stream);
    return launch_reduce(partial, static_cast<half_t*>(y), count, used, stream);
  }
  if (out_dtype == TMC_F32)
    return launch_plan<float, false>(plan, x, w, static_cast<float*>(y), m, k, n, (int)k, stream);
  return launch_plan<half_t, false>(plan, x, w, static_cast<half_t*>(y), m, k, n, (int)k, stream);
}

}  // namespace
}  // namespace tmc

using namespace tmc;

extern "C" int tmc_gemm_mfma_f16(const void* x, const void* weight, void* y, int out_dtype,
                                 int64_t m, int64_t k, int64_t n, void* stream) {
  TMC_REQUIRE(x && weight && y, "Prompt GEMM: null device pointer.");
  TMC_REQUIRE(out_dtype == TMC_F16 || out_dtype == TMC_F32, "Prompt GEMM: output must be f16 or f32.");
  TMC_REQUIRE(m > 0 && k > 0 && n > 0 && m < (1LL << 31) && k < (1LL << 31) && n < (1LL << 31),
              "Prompt GEMM: invalid shape.");
  return launch_gemm(static_cast<const half_t*>(x), static_cast<const half_t*>(weight), y,
                        out_dtype, m, k, n, nullptr, 0, as_stream(stream));
}

extern "C" int tmc_gemm_rows_plan(int64_t m, int64_t k, int64_t n, size_t workspace_bytes,
                                  int32_t out[4]) {
  TMC_REQUIRE(out, "Prompt GEMM: null plan.");
  TMC_REQUIRE(m > 0 && k > 0 && n > 0 && m < (1LL << 31) && k < (1LL << 31) && n < (1LL << 31),
              "Prompt GEMM: invalid shape.");
  const TilePlan plan = tile_plan(m, k, n, workspace_bytes);
  const int64_t length = split_length(k, plan.splits);
  out[0] = plan.bm;
  out[1] = plan.bn;
  out[2] = plan.stages;
  out[3] = (int32_t)((k + length - 1) / length);
  return 0;
}

extern "C" size_t tmc_gemm_rows_workspace_bytes(void) { return (size_t)32 << 20; }

extern "C" int tmc_gemm_rows_f16(const void* x, const void* weight, void* y, int out_dtype,
                                 int64_t m, int64_t k, int64_t n, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  TMC_REQUIRE(x && weight && y, "Prompt GEMM: null device pointer.");
  TMC_REQUIRE(out_dtype == TMC_F16 || out_dtype == TMC_F32, "Prompt GEMM: output must be f16 or f32.");
  TMC_REQUIRE(m > 0 && k > 0 && n > 0 && m < (1LL << 31) && k < (1LL << 31) && n < (1LL << 31),
              "Prompt GEMM: invalid shape.");
  TMC_REQUIRE(workspace || workspace_bytes == 0, "Prompt GEMM: null workspace with a nonzero size.");
  TMC_REQUIRE(!workspace || aligned16(workspace), "Prompt GEMM: the workspace must be 16-byte aligned.");
  return launch_gemm(static_cast<const half_t*>(x), static_cast<const half_t*>(weight), y,
                        out_dtype, m, k, n, workspace, workspace_bytes, as_stream(stream));
}

