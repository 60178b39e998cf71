// Deterministic, batch-invariant bf16 GEMM for gfx950:  C[M,N] = X[M,K] * W[N,K]^T.
//
// Replaces the kernels behind rl_engine._C.det_gemm_* (reference
// csrc/cuda/gemm/det_gemm_kernel.cu:92-101, 250-402) and the Triton MFMA kernels of
// rl_engine/backends/rocm/gemm/mfma_gemm.py:135-274. No split-K, no atomics, no
// stream-K: one workgroup owns an output tile for the whole K range.
#include "det_gemm_solo_body.h"
#include "rlk_host.h"

namespace rlk {

template <class S, int LOOP, bool OUT_F32, int KS = 1, int NS = 2>
__global__ __launch_bounds__(S::kThreads + (has_prefetch_wave<LOOP, KS>() ? kWave : 0)) void det_gemm_kernel(MatView W, MatView X, void* __restrict__ C,
                                                                int64_t ldc, int M, int N, int K,
                                                                int tiles_m, int tiles_n, int group_m) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  det_gemm_tile<S, LOOP, OUT_F32, KS, NS>(W, X, C, ldc, M, N, K, tiles_m, tiles_n, group_m, blockIdx.x, lds);
}

// 256 x 256 tiles, one workgroup per CU that goes through its share of them (det_gemm_solo.h).
template <class Layout>
__global__ __launch_bounds__(SoloShape::kThreads) void det_gemm_solo_kernel(SoloProblem p) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  solo_product<Layout>(p, blockIdx.x, gridDim.x, p.tiles_m * p.tiles_n, lds);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

template <class Layout>
static hipError_t launch_solo(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                              hipStream_t stream) {
  auto kernel = det_gemm_solo_kernel<Layout>;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), Layout::kLds, once);
  if (err != hipSuccess) return err;
  const SoloProblem p = solo_problem<typename Layout::Shape>(W, X, C, ldc, M, N, K);
  const int cus = device_cu_count(), tiles = p.tiles_m * p.tiles_n;
  hipLaunchKernelGGL(kernel, dim3(tiles < cus ? tiles : cus), dim3(SoloShape::kThreads), Layout::kLds, stream, p);
  return hipGetLastError();
}

// A smaller shape on four waves, native operands.
template <int BN, int BM>
static hipError_t launch_solo_shape(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K, hipStream_t stream) {
  return launch_solo<SoloLayout<false, false, TileShape<BN, BM, 2, 2>>>(W, X, C, ldc, M, N, K, stream);
}

template <class S, int LOOP, bool OUT_F32, int KS = 1, int NS = 2>
static hipError_t launch_tile(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                              hipStream_t stream) {
  auto kernel = det_gemm_kernel<S, LOOP, OUT_F32, KS, NS>;
  constexpr int kLds = NS * KS * S::kStageBytes + (has_prefetch_wave<LOOP, KS>() ? kPrefetchDumpBytes : 0);
  static_assert(kLds <= 160 * 1024, "stages exceed the LDS");
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  const int tiles_m = (M + S::BM - 1) / S::BM;
  const int tiles_n = (N + S::BN - 1) / S::BN;
  if constexpr (LOOP == kLoopPingPong && S::BM <= 128 && !OUT_F32) {
    if (streamed_weight(N, K, M, S::BM))
      return launch_tile<S, kLoopPingPongWStream, OUT_F32, KS, NS>(W, X, C, ldc, M, N, K, stream);
  }
  int group_m = tiles_m < 8 ? tiles_m : 8;
  // Two readers, one of them with a few tokens only (whose loads are mostly repeats of its last row), drift apart, and the
  // wave then costs up to 10 % (67 tokens on 64-token tiles, K = 24576: 105 -> 116 us) instead of gaining 18 % (128).
  // A weight that the forward has just left in the memory-side cache costs 3 to 9 % with the wave (dX of 6144 outputs, 4096
  // inputs at 333 tokens 33.3 -> 35.1 us, of 14336 outputs 71.9 -> 76.7), where it saves 10 to 20 % from HBM (42.6 -> 38.1,
  // 94.3 -> 79.8): it runs where the weight is too large to still be there, from 128 MiB, or from 96 MiB with many tokens,
  // whose activations displace it. Right behind the forward / from HBM, in % of the time at 300 / 500 / 700 / 1000 tokens,
  // 4096 inputs: 48 MiB of weight +6 / +2 / +2 / -2 and -14 / -13 / -23 / -17, 96 MiB +1 / -3 / -2 / +1 and -16 / -13 / -25 /
  // -15, 112 MiB +3 / 0 / -8 / -14 and -19 / -15 / -25 / -16, 128 MiB -13 / -11 / -21 / -17 and -19 / -14 / -25 / -16.
  const bool shared_panel = tiles_m > 2 || M > S::BM + S::BM / 2;
  const int64_t weight_bytes = (int64_t)N * K * 2;
  const bool from_hbm = weight_bytes >= ((int64_t)128 << 20) || (weight_bytes >= ((int64_t)96 << 20) && M > 512);
  const bool prefetch = LOOP == kLoopQuadPrefetch || (has_prefetch_wave<LOOP, KS>() && shared_panel && from_hbm);
  const int threads = S::kThreads + (prefetch ? kWave : 0);
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n), dim3(threads), kLds, stream, W, X, C, ldc, M, N, K,
                     tiles_m, tiles_n, group_m);
  return hipGetLastError();
}

template <class S, int LOOP, int NS = 2>
static hipError_t launch_loop(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                              bool out_f32, hipStream_t stream) {
  return out_f32 ? launch_tile<S, LOOP, true, 1, NS>(W, X, C, ldc, M, N, K, stream)
                 : launch_tile<S, LOOP, false, 1, NS>(W, X, C, ldc, M, N, K, stream);
}

// LDS stages of the native ping-pong loop: 256 x 128 and 256 x 64 run three (144 / 120 KiB). With
// weights that come from HBM the extra K tile of lead is worth 8 % (gate_up at 256 tokens:
// 73 -> 68 us); on cache-resident operands it changes nothing. The smaller shapes have their
// deep-stage variants; the K-major loops measured no gain from a third stage and keep two.
template <class S>
constexpr int pingpong_stages() {
  return (S::BN >= 192 && S::BM <= 128) ? 3 : 2;
}

// `loop`: the K-major ping-pong variant the operand layouts call for.
template <class S>
static hipError_t launch_kmajor(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K, int loop,
                                bool out_f32, hipStream_t stream) {
  static_assert(pingpong_supported<S>() && S::TN == 4, "64-feature wave columns");
  if (loop == kLoopPingPongKMajor) return launch_loop<S, kLoopPingPongKMajor>(W, X, C, ldc, M, N, K, out_f32, stream);
  if constexpr (S::BM % 128 == 0) {
    if (loop == kLoopPingPongXKMajor) return launch_loop<S, kLoopPingPongXKMajor>(W, X, C, ldc, M, N, K, out_f32, stream);
    if (loop == kLoopPingPongBothKMajor)
      return launch_loop<S, kLoopPingPongBothKMajor>(W, X, C, ldc, M, N, K, out_f32, stream);
  }
  return hipErrorInvalidValue;
}

// ELEMENTS: whether operands that are not 16-byte aligned come here (`vec` is true otherwise).
template <class S, bool ELEMENTS = true>
static hipError_t launch_shape(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                               bool vec, bool allow_pingpong, bool out_f32, hipStream_t stream) {
  if constexpr (pingpong_supported<S>()) {
    if (vec && allow_pingpong && K % kTileK == 0) {
      return launch_loop<S, kLoopPingPong, pingpong_stages<S>()>(W, X, C, ldc, M, N, K, out_f32, stream);
    }
  }
  if constexpr (ELEMENTS) {
    if (!vec) return launch_loop<S, kLoopGeneric>(W, X, C, ldc, M, N, K, out_f32, stream);
  }
  return vec ? launch_loop<S, kLoopStaged>(W, X, C, ldc, M, N, K, out_f32, stream) : hipErrorInvalidValue;
}

// Deep-stage variant (KS K tiles per barrier pair) of a small tile; native layout only. Two stages of 64 KiB, three of 48
// for 128x64 (8 % faster; deeper rings did not pay for the square ones).
constexpr int kDeep64 = 4;   // 64x32 / 64x64: K tiles per stage
constexpr int kDeep128 = 2;  // 64x96 / 128x64 / 128x128
template <class S, int KS, int NS = 2>
static hipError_t launch_deep(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                              bool out_f32, hipStream_t stream) {
  return out_f32 ? launch_tile<S, kLoopPingPong, true, KS, NS>(W, X, C, ldc, M, N, K, stream)
                 : launch_tile<S, kLoopPingPong, false, KS, NS>(W, X, C, ldc, M, N, K, stream);
}

// The quad loop, with the prefetch wave where several workgroups read a weight panel: from HBM all of them wait for the
// same lines, and whole token tiles keep them in step (a nearly empty one runs ahead and is the others' prefetch). Weights
// from HBM / from the memory-side cache, eight waves in two groups -> four -> four and the prefetch wave, 4096 outputs,
// K = 12288:
//   64 x 96, 384 tokens:  66.6 / 58.3 -> 68.5 / 51.0 -> 59.2 / 50.9 us      333 tokens:  64.0 / 60.7 -> 60.1 / 52.9 -> 58.0 / 50.5
//   128 x 64, 512 tokens: 78.1 / 65.6 -> 86.9 / 63.9 -> 69.8 / 62.2 (six stages of one K tile)
//   32 x 64, 128 tokens:  45.2 / 29.6 -> 42.0 / 32.8 with the wave            80 tokens:  33.4 / 28.7 -> 36.1 / 30.8
// (64 x 64, 256 tokens: 49.2 / 41.4 -> 59.2 / 39.3 -> 50.2 / 41.2, 128 x 128: 99 / 93 -> 117 / 107: they stay with eight
// waves.) A panel that several workgroups read always has the wave on 64 x 96 and 64 x 160 tiles (and on 128 x 64, which
// are launched without this rule), on the smaller ones where the weight is larger than what the memory-side cache holds
// beside others (96 MiB) and the last token tile is more than half full, on 32 x 32 never (two readers at most: 64 tokens
// 33.2 -> 35.1).
template <class S, int KS, int NS, bool PREFETCH = true>
static hipError_t launch_quad(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K, bool out_f32,
                              hipStream_t stream) {
  if constexpr (PREFETCH) {
    const bool shared_panel = M > S::BM + S::BM / 2;  // (see launch_tile)
    const bool in_step = (M - 1) % S::BM >= S::BM / 2 && (int64_t)N * K * 2 >= ((int64_t)96 << 20);
    if (shared_panel && (S::BN + S::BM >= 160 || in_step))
      return out_f32 ? launch_tile<S, kLoopQuadPrefetch, true, KS, NS>(W, X, C, ldc, M, N, K, stream)
                     : launch_tile<S, kLoopQuadPrefetch, false, KS, NS>(W, X, C, ldc, M, N, K, stream);
  }
  if (out_f32) return launch_tile<S, kLoopQuad, true, KS, NS>(W, X, C, ldc, M, N, K, stream);
  if (M <= S::BM && streamed_weight(N, K, M, S::BM))
    return launch_tile<S, kLoopQuadWStream, false, KS, NS>(W, X, C, ldc, M, N, K, stream);
  return launch_tile<S, kLoopQuad, false, KS, NS>(W, X, C, ldc, M, N, K, stream);
}

// The loops of a small tile for a K-major weight: from one ring on (512 / 384 / 256 values of K for 64 x 64 / 128 x 64 /
// 128 x 128) the direct-to-LDS ping-pong loop, with the rest that its stages do not divide behind it (LogP grad_hidden,
// 1024 tokens, V = 18992, whose rest is 48 values: 154 us, register-staged 250); below that the register-staged loop, whose
// two stages hold all or most of so short a reduction.
template <class S>
static hipError_t launch_small_kmajor(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                                       bool out_f32, hipStream_t stream) {
  // Stages of two K tiles, as many of them as 128 KiB (144 for the 128 x 64 tile) hold.
  constexpr int kDmaKs = 2;
  constexpr int kDmaNs = S::kStageBytes <= 16 * 1024 ? 4 : S::kStageBytes <= 24 * 1024 ? 3 : 2;
  if (K >= kTileK * kDmaKs * kDmaNs)
    return out_f32 ? launch_tile<S, kLoopPingPongKMajor, true, kDmaKs, kDmaNs>(W, X, C, ldc, M, N, K, stream)
                   : launch_tile<S, kLoopPingPongKMajor, false, kDmaKs, kDmaNs>(W, X, C, ldc, M, N, K, stream);
  constexpr int kKs = 128 * 1024 / (2 * S::kStageBytes) >= 4 ? 4 : 2;
  if (K % kTileK != 0)
    return out_f32 ? launch_tile<S, kLoopStagedKMajorTail, true, kKs, 2>(W, X, C, ldc, M, N, K, stream)
                   : launch_tile<S, kLoopStagedKMajorTail, false, kKs, 2>(W, X, C, ldc, M, N, K, stream);
  return out_f32 ? launch_tile<S, kLoopStagedKMajor, true, kKs, 2>(W, X, C, ldc, M, N, K, stream)
                 : launch_tile<S, kLoopStagedKMajor, false, kKs, 2>(W, X, C, ldc, M, N, K, stream);
}

// Tile shapes. Which one runs is a pure performance choice (see det_gemm_tile.h).
using Shape256x256 = TileShape<256, 256, 4, 2>;
using Shape192x256 = TileShape<192, 256, 4, 2>;  // 192 features x 256 tokens: three MFMA tiles per wave along N
using Shape256x192 = TileShape<256, 192, 4, 2>;
using Shape192x192 = TileShape<192, 192, 4, 2>;  // 192 features x 192 tokens
using Shape192x128 = TileShape<192, 128, 4, 2>;  // 192 features x 128 tokens
using Shape256x128 = TileShape<256, 128, 4, 2>;
using Shape256x64 = TileShape<256, 64, 4, 2>;
using Shape128x128 = TileShape<128, 128, 4, 2>;
using Shape128x64 = TileShape<128, 64, 4, 2>;
using Shape64x64 = TileShape<64, 64, 4, 2>;
using Shape64x16 = TileShape<64, 16, 4, 1>;
using Quad128x64 = TileShape<128, 64, 2, 2>;
using Quad64x160 = TileShape<64, 160, 2, 2>;
using Quad96x64 = TileShape<96, 64, 2, 2>;
using Quad64x96 = TileShape<64, 96, 2, 2>;
using Quad64x32 = TileShape<64, 32, 2, 2>;
using Quad32x64 = TileShape<32, 64, 2, 2>;
using Quad32x32 = TileShape<32, 32, 2, 2>;
using Shape16x16 = TileShape<16, 16, 1, 1>;

static bool view_is_vectorizable(const MatView& v) {
  return v.k_stride == 1 && (v.row_stride % kChunkElems) == 0 && pitch_fits_lane_offsets(v.row_stride) &&
         (reinterpret_cast<uintptr_t>(v.ptr) & 15) == 0;
}

static int64_t tile_count(int M, int N, int bm, int bn) {
  return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

int device_cu_count() {
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return 256;
  }
  const bool tracked = dev >= 0 && dev < kMaxDevices;
  if (tracked) {
    const int have = cached[dev].load(std::memory_order_relaxed);
    if (have > 0) return have;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess || prop.multiProcessorCount <= 0) {
    (void)hipGetLastError();
    return 256;
  }
  if (tracked) cached[dev].store(prop.multiProcessorCount, std::memory_order_relaxed);
  return prop.multiProcessorCount;
}

// Every tile shape the automatic choice weighs, in one table. `native` is the relative throughput of the shape on a
// full chip with both operands in the native (reduction-contiguous) layout, `w_kmajor` the same with a K-major weight
// (0: the shape has no such loop); `x_kmajor` says whether the shape also takes a K-major activation operand. The
// estimated time of a launch is rounds_of_workgroups(tiles) x tile area / quality; larger tiles win ties.
//
// Native column, fitted to sweeps over the Qwen3-8B projection shapes at 384 ... 6144 tokens: 192 x 256 (three
// quarters of the large tile at 0.89 of its throughput) fills the rounds that N / 256 leaves half empty - gate_up at
// 1024 tokens is 512 tiles = two full rounds instead of 384 = one and a half (169 -> 152 us), qkv at 3072 tokens
// 150 -> 128 us. Where 192 does not divide N its last feature tile is partly empty and the shape counts as
// `ragged192`: it still wins where it turns a round and a fraction into less (N = 5120 at 4096 tokens 293 -> 256 us,
// N = 10240 at 2048 tokens 190 -> 162 us) and loses the tie against 256 x 128 at N = 4096, 2048 tokens. 192 x 128
// (three stages) does the same one size down (weights from HBM: gate_up at 256 tokens 65.0 -> 62.2 us, N = 6144 at 768
// tokens 55.1 -> 49.1 us).
// 192-token tiles where two of them, or three, hold what 128- and 256-token tiles do not divide well; they read 144 and
// 160 rows per wave and K tile from LDS for 36 and 48 matrix instructions a step, between 256 x 128 (128 for 32) and 256 x
// 256. Weights of three layers in turn, before -> with them: gate_up at 360 / 700 / 900 tokens 89.9 / 156 / 169 -> 72.0 / 134 /
// 157 us, 12288 outputs at 700 / 1500 tokens 78.8 / 153 -> 65.2 / 133, 14336 at 540 / 1300 tokens 81.3 / 158 -> 65.1 / 144,
// qkv at 1300 tokens 67.4 -> 58.3, down at 2600 tokens 224 -> 206.
// K-major-weight column (`dY @ W`, `a @ b`, prepared weights): the 64- and 128-feature tiles give a long reduction
// against few output tiles - grad_hidden of the LogP backward up to about a thousand tokens (N = 4096, K = 151936) - a
// workgroup per CU, each streaming a narrow slice of the weight instead of a 256-column one (1.9 -> 0.8 ms at 256
// tokens, 1.8 -> 1.03 ms at 512, 1.65 -> 1.45 ms at 1024); their qualities are those of the direct-to-LDS loop. 256 x 192:
// dX of 14336 inputs, 4096 outputs at 540 / 1300 tokens 106 / 169 -> 68 / 142 us, of 4096, 6144 at 2300 tokens 108 -> 95.
//
// The `four` column is the relative throughput of a shape's four-wave form (det_gemm_solo.h, 0: none), which native operands with
// whole K tiles and bf16 results have. Waves of half a tile by half read every row of a K tile from LDS twice, where eight of a
// quarter by half read token rows four times; those reads and what arrives are 1856 cycles of LDS a K tile beside 1536 of MFMAs in 192
// x 256, 1344 with four waves, 1536 / 1152 beside 1152 in 192 x 192. With them a round that fills part of the chip costs less, the more
// so behind others (kPartialFirst, kPartialLast). Shapes without such a form are weighed beside them at their `native` quality, 256 x
// 128 in one full round at a better one. 560 shapes of 33 to 16000 tokens, 128 to 24576 outputs, K = 64 to 14336, weights in turn: where 128 does
// not divide K, which shuts out the deep tiles of few tokens, 0.983 of the eight waves' time, 0.6 % above the best shape of each, where
// it does 0.935 and 1.2 %. Eight waves -> these, us: 4096 outputs, K = 4096 at 1400 / 2047 / 3000 tokens 53.9 / 62.8 / 79.1 -> 49.7 /
// 57.8 / 73.8, 6144 at 1024 / 2048 / 3072 56.9 / 83.6 / 124.8 -> 51.7 / 78.4 / 117.9, K = 12288 at 2047 176 -> 164, 24576 outputs at 700 /
// 1024 129.9 / 167.4 -> 120.2 / 156.6. What the small shapes and 256 x 128 are there for (the best without them / with): K = 2880, 2880
// outputs at 65 / 200 tokens 31.9 / 32.9 -> 22.6 / 22.5, 5760 at 100 34.6 -> 23.1, K = 1600, 1536 outputs at 300 16.6 -> 11.2; K = 12288,
// 8192 outputs at 1009 191 -> 169 (but K = 4096, 14336 outputs at 487, 7 / 8 of a round, 58.9 / 62.7). (256 x 128 and 128 x 128 on four
// waves were never the best shape by more than the noise.)
struct TileCandidate {
  int config, bn, bm;
  double native, ragged192, w_kmajor;
  bool x_kmajor;
  double four;
};
static const TileCandidate kTileCandidates[] = {
    {RLK_GEMM_CFG_256x256, 256, 256, 1.00, 0.00, 1.00, true, 1.00},  {RLK_GEMM_CFG_192x256, 192, 256, 0.89, 0.85, 0.00, false, 0.95},
    {RLK_GEMM_CFG_256x192, 256, 192, 0.87, 0.00, 0.87, false, 0.94}, {RLK_GEMM_CFG_192x192, 192, 192, 0.75, 0.68, 0.00, false, 0.93},
    {RLK_GEMM_CFG_256x128, 256, 128, 0.65, 0.00, 0.70, true, 0.00},  {RLK_GEMM_CFG_192x128, 192, 128, 0.56, 0.53, 0.00, false, 0.80},
    {RLK_GEMM_CFG_256x64, 256, 64, 0.50, 0.00, 0.56, false, 0.00},   {RLK_GEMM_CFG_128x128, 128, 128, 0.65, 0.00, 0.62, false, 0.00},
    {RLK_GEMM_CFG_128x64, 128, 64, 0.45, 0.00, 0.40, false, 0.00},   {RLK_GEMM_CFG_64x64, 64, 64, 0.42, 0.00, 0.25, false, 0.00},
};
constexpr double kPartialFirst = 0.82, kPartialLast = 0.6, kFourRagged192 = 0.92, kPartialEight = 0.9, kFullRound256x128 = 0.80;

// The cheapest shape for operands that the four-wave forms take.
static int pick_four_wave_shape(int M, int N) {
  const int cus = device_cu_count();
  int best = RLK_GEMM_CFG_256x256;
  double best_time = 1e300;
  for (const TileCandidate& c : kTileCandidates) {
    const int64_t tiles = tile_count(M, N, c.bm, c.bn);
    const bool one_round = tiles <= cus;
    double quality = c.four, partial = one_round ? kPartialFirst : kPartialLast;
    if (c.four == 0.0) {
      quality = one_round && 16 * tiles >= 15 * cus && c.config == RLK_GEMM_CFG_256x128 ? kFullRound256x128 : c.native;
      partial = kPartialEight;
    } else if (c.bn == 192 && N % 192 != 0) {
      quality *= kFourRagged192;
    }
    const double t = rounds_of_workgroups(tiles, cus, partial) * (double)(c.bn * c.bm) / quality;
    if (t < best_time * 0.999) {
      best_time = t;
      best = c.config;
    }
  }
  return best;
}

// The cheapest candidate by the estimate above. `w_kmajor` / `x_kmajor`: the operand layouts of the call.
static const TileCandidate& best_tile_candidate(int M, int N, int K, bool w_kmajor, bool x_kmajor, double partial_floor,
                                                double* estimate) {
  const int cus = device_cu_count();
  const TileCandidate* best = kTileCandidates;
  double best_time = 1e300;
  for (const TileCandidate& c : kTileCandidates) {
    double quality;
    if (w_kmajor || x_kmajor) {
      if (c.w_kmajor == 0.0 || (x_kmajor && !c.x_kmajor)) continue;
      if (c.bn <= 128 && !w_kmajor) continue;  // the small K-major tiles exist for a K-major weight only
      quality = c.w_kmajor;
    } else {
      const bool wide192 = c.ragged192 != 0.0;
      if ((wide192 || c.bm == 192) && K % kTileK != 0) continue;  // the direct-to-LDS loop only
      quality = (wide192 && N % 192 != 0) ? c.ragged192 : c.native;
    }
    const double t = rounds_of_workgroups(tile_count(M, N, c.bm, c.bn), cus, partial_floor) * (double)(c.bn * c.bm) / quality;
    if (t < best_time * 0.999) {
      best_time = t;
      best = &c;
    }
  }
  *estimate = best_time;
  return *best;
}

static int pick_tile_candidate(int M, int N, int K, bool w_kmajor, bool x_kmajor) {
  double estimate;
  return best_tile_candidate(M, N, K, w_kmajor, x_kmajor, kPartialEight, &estimate).config;
}

// Not where a single K tile is one round of the shape that eight waves would have: four have nothing in front of its loads (eight /
// four waves, us, K = 64: 1822 x 5760 10.6 / 12.3, 1590 x 4096 8.6 / 11.6; of more rounds 6000 x 5760 28.6 / 20.9).
static bool four_waves_pay(int M, int N, int K) {
  if (K > kTileK) return true;
  double estimate;
  const TileCandidate& c = best_tile_candidate(M, N, K, false, false, kPartialEight, &estimate);
  return tile_count(M, N, c.bm, c.bn) > device_cu_count();
}

double det_gemm_kmajor_us(int M, int N, int K, bool w_kmajor, bool x_kmajor, double partial_floor, int* tile_outputs) {
  // Of 256 x 256 tiles at the native rate, 11 + 21 K / 1024 us each (see remainder_launch_pays): the eight-wave loops. On the four waves
  // that det_gemm_launch() gives most of them the products take 2 to 10 % less, which the estimates of linear_backward_plan(), fitted
  // beside this one, do not have.
  double outputs;
  const TileCandidate& tile = best_tile_candidate(M, N, K, w_kmajor, x_kmajor, partial_floor, &outputs);
  if (tile_outputs) *tile_outputs = tile.bn * tile.bm;
  return (11.0 + 21.0 * K / 1024.0) * outputs / 65536.0;
}

int pick_det_gemm_config(int M, int N, int K, bool four_waves) {
  const int cus = device_cu_count();
  // Decode (weights fitted while they rotate through 1.3 GB, i.e. come from HBM as in a model with
  // many layers, not from the 256 MB memory-side cache): up to 16 tokens the streaming kernel with
  // two workgroups per CU is the fastest or equal for every Qwen3-8B projection (gate_up 52 -> 38 us,
  // qkv 14 -> 12 us against the one-wave tile kernel, which wins only when the weight is cache
  // resident). Up to 32 tokens it holds while there is at most a panel per CU; for a K that the 32 x 32 tiles below do not
  // take, up to 32 / 64 tokens with 1.5 / 1 panels per CU.
  if (M <= 16) return (K >= 1024 && K % kTileK == 0) ? RLK_GEMM_CFG_STREAM16 : RLK_GEMM_CFG_16x16;
  const bool deep = K % (kTileK * kDeep128) == 0;
  if (K >= 1024 && K % kTileK == 0 &&
      ((M <= 32 && N <= (deep ? 16 : 24) * cus) || (M <= 64 && !deep && N <= 16 * cus)))
    return RLK_GEMM_CFG_STREAM64;
  // Problems that give the chip at most one small tile per CU: one workgroup per CU with several K tiles in flight beats
  // the same tile run several workgroups per CU. A CU's time goes with the rows (features + tokens) that its workgroup
  // brings in and reads back from LDS per K tile, so the tile with the fewest that still fits one round is taken. Weights
  // from HBM / from the memory-side cache, before each tile was there -> with it:
  //   32 x 32: down at 33 / 64 tokens 28.0 / 25.0, 36.7 / 28.0 (streaming kernel) -> 24.4 / 20.6, 33.2 / 20.4 us; N = 6144 at
  //            17 / 32 tokens 15.8 / 13.5, 17.8 / 14.3 -> 12.0 / 10.3, 13.5 / 10.5; N = 1536 at 128 tokens 16.0 / 11.3 -> 11.1 / 8.1
  //   32 x 64: down at 80 tokens 45.8 / 36.4 (64 x 64, on half the CUs) -> 33.4 / 28.7, at 128 tokens 50.4 / 37.0 -> 42.0 / 32.8
  //   64 x 32: N = 12288 at 17 tokens 22.1 / 17.0 -> 21.6 / 16.9
  //   64 x 96: down at 288 / 384 tokens 74.6 / 60.2, 76.7 / 60.5 (128 x 64) -> 59.0 / 49.1, 59.4 / 51.4; N = 6144 at 192 tokens
  //            29.1 / 23.6 -> 23.3 / 20.2
  //   96 x 64: N = 24576 at 64 tokens 42.4 / 39.0 (128 x 64) -> 40.3 / 36.1, 12288 at 100 tokens 32.6 / 24.0 -> 29.0 / 23.0, 6144
  //            at 200 tokens 30.2 / 23.0 -> 24.7 / 19.0, K = 12288 at 256 tokens 92.6 / 62.2 -> 77.0 / 52.0
  //   128 x 64 with the prefetch: down at 512 tokens 76.6 / 65.0 -> 70.1 / 60.7, N = K = 4096 at 512 tokens 27.6 / 24.8 -> 25.0 / 22.6
  //   64 x 160: down at 600 tokens 90.6 / 75.1 (128 x 128) -> 80.2 / 74.1, N = K = 4096 at 600 tokens 32.0 / 28.1 -> 29.3 / 27.6
  if (deep && tile_count(M, N, 32, 32) <= cus) return RLK_GEMM_CFG_32x32_DEEP;
  if (K % (kTileK * kDeep64) == 0) {
    if (tile_count(M, N, 64, 32) <= cus) return RLK_GEMM_CFG_32x64_DEEP;
    if (tile_count(M, N, 32, 64) <= cus) return RLK_GEMM_CFG_64x32_DEEP;
    if (tile_count(M, N, 64, 64) <= cus) return RLK_GEMM_CFG_64x64_DEEP;
  }
  if (deep) {
    // 160 rows both. 96 x 64 first where its three token tiles hold what two of 96 leave partly empty (N = 6144 at 160 tokens 27.0
    // / 20.3 as 64 x 96, 24.5 / 18.1 as 96 x 64; with K = 12288 77.9 / 51.6, 70.1 / 46.8).
    const bool fits96x64 = tile_count(M, N, 64, 96) <= cus;
    if (fits96x64 && M > 128 && M <= 192) return RLK_GEMM_CFG_96x64_DEEP;
    if (tile_count(M, N, 96, 64) <= cus) return RLK_GEMM_CFG_64x96_DEEP;
    if (fits96x64) return RLK_GEMM_CFG_96x64_DEEP;
    if (tile_count(M, N, 64, 128) <= cus) return RLK_GEMM_CFG_128x64_DEEP;
    if (tile_count(M, N, 160, 64) <= cus) return RLK_GEMM_CFG_64x160_DEEP;
    if (tile_count(M, N, 128, 128) <= cus) return RLK_GEMM_CFG_128x128_DEEP;
  }
  return four_waves && four_waves_pay(M, N, K) ? pick_four_wave_shape(M, N) : pick_tile_candidate(M, N, K, false, false);
}

// A K-major view (element [row, k] at ptr[k * k_stride + row], rows contiguous: B[K,N] as the
// weight operand, or the transposed operands of a weight gradient) that the transposing
// ping-pong loop can take.
static bool view_is_kmajor_fast(const MatView& v) {
  return v.row_stride == 1 && v.k_stride >= v.rows && (v.k_stride % kChunkElems) == 0 && pitch_fits_lane_offsets(v.k_stride) &&
         (reinterpret_cast<uintptr_t>(v.ptr) & 15) == 0 && (v.rows % kChunkElems) == 0;
}

// A reduction length that 64 does not divide (the token count of a weight gradient) runs its whole K tiles in
// the same loops and the rest in a register-staged step behind them; a native operand of the pair then
// needs whole 16-byte chunks (K % 8 == 0, or rows that go on to the end of the chunk).
bool det_gemm_takes_kmajor(const MatView& W, const MatView& X, int K) {
  const bool w_native = view_is_vectorizable(W), x_native = view_is_vectorizable(X);
  const bool w_kmajor = !w_native && view_is_kmajor_fast(W), x_kmajor = !x_native && view_is_kmajor_fast(X);
  const bool k_fits = K >= 1 && ((K % kChunkElems) == 0 || (w_kmajor && x_kmajor) || (w_kmajor && X.k_padded));
  return k_fits && (w_kmajor || x_kmajor) && (w_native || w_kmajor) && (x_native || x_kmajor);
}

// A token count just above a multiple of 256 (4097, 8200 ...) gives the large tiles a last row of token tiles that
// is nearly empty; when that row is what opens another round of workgroups, the few tokens cost a whole tile
// time (down at 4097 tokens: 272 tiles = two rounds instead of one, 0.54 against 0.27 ms). Rows are independent,
// so the remainder can run as a launch of its own on the few-token kernels without changing a bit. Returns
// whether that pays: the round the remainder opens, priced at 11 + 21 K / 1024 us for a 256 x 256 tile
// (measured on gate_up across K), against the few-token launch, which streams the weight once.
static bool remainder_launch_pays(int M, int N, int K, int rest, bool fast_few_tokens, bool w_kmajor) {
  const int64_t cus = device_cu_count();
  const int64_t feature_tiles = (N + 255) / 256;
  const int64_t rounds_all = (feature_tiles * ((M + 255) / 256) + cus - 1) / cus;
  const int64_t rounds_main = (feature_tiles * (M / 256) + cus - 1) / cus;
  if (rounds_all == rounds_main) return false;  // the remainder's tiles fit beside the last round
  const double round_us = 11.0 + 21.0 * K / 1024.0;
  double rest_us;
  if (w_kmajor) {
    // A chain of K tiles on the small tiles, an upper estimate: 0.27 to 0.41 us each at 1 to 64 tokens from HBM (4096
    // inputs, K = 4096 / 12288 / 24576: 20 to 26, 53 to 71, 103 to 142 us), 0.2 from the cache. Either way it pays from two
    // K tiles on.
    rest_us = 10.0 + 0.4 * (K / 64.0);
  } else if (fast_few_tokens) {
    rest_us = 8.0 + 2.0 * N * (double)K / 4.5e6 * (rest <= 16 ? 1.0 : 1.5);  // the weight once at 4.5 TB/s
  } else {
    return false;
  }
  return rest_us < 0.8 * round_us;
}

// Native operands (16-byte rows) that the four-wave forms take.
static bool four_waves_take(const MatView& W, const MatView& X, int K, bool out_f32) {
  return K % kTileK == 0 && !out_f32 && solo_offsets_fit(W) && solo_offsets_fit(X);
}

// K rows of a K-major weight a multiple of 4 KiB apart that is no power of two: the columns that four waves load each for itself take
// longer there than the rows that eight load side by side. Eight / four, us, 256 x 128, K = 2880 at 200 tokens, by outputs: 4096 40.2 /
// 38.4, 5120 45.1 / 41.7, 6144 42.1 / 43.9, 7680 44.1 / 41.9, 8192 40.4 / 38.2, 10240 44.4 / 45.7, 11264 43.1 / 43.6, 12288 43.1 / 47.4, 13312
// 43.6 / 43.6, 14336 43.0 / 45.3, 16384 42.2 / 40.4, 18432 44.3 / 46.8, 20480 45.5 / 56.5; 256 x 192, K = 4096 at 700, 12288 69.7 / 77.5,
// 14336 77.2 / 78.2, in two rounds, 2047 tokens, 214.6 / 199.8, 217.6 / 208.4. (256 x 256: four at every pitch.)
static bool kmajor_rows_clash(const MatView& v) {
  const int64_t pitch = v.k_stride * 2;
  return pitch % 4096 == 0 && (pitch & (pitch - 1)) != 0;
}

hipError_t det_gemm_launch(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                           bool out_f32, int config, hipStream_t stream) {
  if (config == RLK_GEMM_CFG_AUTO && M > 256 && M % 256 >= 1 && M % 256 <= 64) {
    const int rest = M % 256;
    const bool natives = view_is_vectorizable(W) && view_is_vectorizable(X) && K % kTileK == 0 && K >= 1024;
    const bool kmajor_w = !view_is_vectorizable(W) && view_is_kmajor_fast(W) && view_is_vectorizable(X) &&
                          (K % kChunkElems == 0 || X.k_padded);
    if ((natives || kmajor_w) && remainder_launch_pays(M, N, K, rest, natives, kmajor_w)) {
      MatView head = X, tail = X;
      head.rows = M - rest;
      tail.rows = rest;
      tail.ptr = X.ptr + (int64_t)(M - rest) * X.row_stride;
      hipError_t err = det_gemm_launch(W, head, C, ldc, M - rest, N, K, out_f32, config, stream);
      if (err != hipSuccess) return err;
      char* c_tail = reinterpret_cast<char*>(C) + (int64_t)(M - rest) * ldc * (out_f32 ? 4 : 2);
      return det_gemm_launch(W, tail, c_tail, ldc, rest, N, K, out_f32, config, stream);
    }
  }
  if ((config & ~RLK_GEMM_CFG_FORCE_STAGED) == RLK_GEMM_CFG_SHORTK) {
    // Serves a K-major token operand with K <= 256 only (and has no register-staged form); anything else runs
    // the picked tile kernel (same bits).
    if (config == RLK_GEMM_CFG_SHORTK && det_gemm_shortk_supported(W, X, M, N, K))
      return det_gemm_shortk_launch(W, X, C, ldc, M, N, K, out_f32, stream);
    config = RLK_GEMM_CFG_AUTO | (config & RLK_GEMM_CFG_FORCE_STAGED);
  }
  // A weight gradient of up to 256 tokens with many output rows: the feature operand stays in registers.
  if (config == RLK_GEMM_CFG_AUTO && det_gemm_shortk_supported(W, X, M, N, K) && det_gemm_shortk_pays(M, N))
    return det_gemm_shortk_launch(W, X, C, ldc, M, N, K, out_f32, stream);
  const bool w_native = view_is_vectorizable(W), x_native = view_is_vectorizable(X);
  const bool vec = w_native && x_native && (K % kChunkElems) == 0;
  const bool allow_pingpong = (config & RLK_GEMM_CFG_FORCE_STAGED) == 0;
  bool four_waves = (config & RLK_GEMM_CFG_FOUR_WAVES) != 0;
  const bool automatic = (config & ~RLK_GEMM_CFG_FORCE_STAGED) == RLK_GEMM_CFG_AUTO;
  config &= ~(RLK_GEMM_CFG_FORCE_STAGED | RLK_GEMM_CFG_FOUR_WAVES);
  const bool w_kmajor = !w_native && view_is_kmajor_fast(W), x_kmajor = !x_native && view_is_kmajor_fast(X);
  if (allow_pingpong && det_gemm_takes_kmajor(W, X, K)) {
    const int loop = w_kmajor ? (x_kmajor ? kLoopPingPongBothKMajor : kLoopPingPongKMajor) : kLoopPingPongXKMajor;
    // Only the shapes with 64-feature wave columns have the transposing loop, and a K-major
    // activation needs at least 128 tokens per tile.
    // With few token tiles against a long reduction (grad_hidden of the LogP backward at 1024 tokens: N = 4096,
    // K = 151936) a smaller token tile doubles the workgroups, every one of which still streams its whole weight panel.
    if (config == RLK_GEMM_CFG_AUTO) {
      config = pick_tile_candidate(M, N, K, w_kmajor, x_kmajor);
      // 256 x 128 where the weight can still be in the memory-side cache, from HBM the eight waves are faster (12288 outputs, K = 4096 at
      // 324 / 483 tokens 58.9 / 61.1 us, four 65.4 / 68.7), 256 x 192 wherever its rows do not clash in one round. Eight -> four: 4096
      // outputs at 1400 / 2047 tokens 59.5 / 66.7 -> 54.3 / 59.1, 256 x 192: 2300 tokens, K = 6144 104 -> 98, K = 14336 at 5969 495 -> 467.
      const bool clash = kmajor_rows_clash(W);
      four_waves = config == RLK_GEMM_CFG_256x192 ? !clash || tile_count(M, N, 192, 256) > device_cu_count()
                                                  : !clash && (int64_t)N * K * 2 < ((int64_t)96 << 20);
      if (config == RLK_GEMM_CFG_256x256 && solo_kmajor_pays(tile_count(M, N, 256, 256), device_cu_count(), w_kmajor && x_kmajor))
        config = RLK_GEMM_CFG_256x256_SOLO;
    }
    if (config == RLK_GEMM_CFG_256x256_SOLO) {
      if (!out_f32 && solo_kmajor_fits(W) && solo_kmajor_fits(X))
        return !x_kmajor   ? launch_solo<SoloLayout<true, false>>(W, X, C, ldc, M, N, K, stream)
               : w_kmajor ? launch_solo<SoloLayout<true, true>>(W, X, C, ldc, M, N, K, stream)
                          : launch_solo<SoloLayout<false, true>>(W, X, C, ldc, M, N, K, stream);
      config = RLK_GEMM_CFG_256x256;
    }
    switch (config) {
      case RLK_GEMM_CFG_256x256:
        return launch_kmajor<Shape256x256>(W, X, C, ldc, M, N, K, loop, out_f32, stream);
      case RLK_GEMM_CFG_256x192:
        if (four_waves && w_kmajor && !x_kmajor && !out_f32 && solo_kmajor_fits(W) && solo_kmajor_fits(X))
          return launch_solo<SoloLayout<true, false, TileShape<256, 192, 2, 2>>>(W, X, C, ldc, M, N, K, stream);
        if (!x_kmajor) return launch_kmajor<Shape256x192>(W, X, C, ldc, M, N, K, loop, out_f32, stream);
        break;
      case RLK_GEMM_CFG_256x128:
        if (four_waves && w_kmajor && !x_kmajor && !out_f32 && solo_kmajor_fits(W) && solo_kmajor_fits(X))
          return launch_solo<SoloLayout<true, false, TileShape<256, 128, 2, 2>>>(W, X, C, ldc, M, N, K, stream);
        return launch_kmajor<Shape256x128>(W, X, C, ldc, M, N, K, loop, out_f32, stream);
      case RLK_GEMM_CFG_256x64:
        if (!x_kmajor) return launch_kmajor<Shape256x64>(W, X, C, ldc, M, N, K, loop, out_f32, stream);
        break;
      case RLK_GEMM_CFG_64x64:
        if (w_kmajor && x_native) return launch_small_kmajor<Shape64x64>(W, X, C, ldc, M, N, K, out_f32, stream);
        break;
      case RLK_GEMM_CFG_128x64:
        if (w_kmajor && x_native) return launch_small_kmajor<Shape128x64>(W, X, C, ldc, M, N, K, out_f32, stream);
        break;
      case RLK_GEMM_CFG_128x128:
        if (w_kmajor && x_native) return launch_small_kmajor<Shape128x128>(W, X, C, ldc, M, N, K, out_f32, stream);
        break;
      default:
        break;  // an explicitly requested other shape runs the element-wise loader below
    }
  }
  if (config == RLK_GEMM_CFG_AUTO) {
    four_waves = vec && allow_pingpong && four_waves_take(W, X, K, out_f32) && four_waves_pay(M, N, K);
    config = pick_det_gemm_config(M, N, K, four_waves);
    // the picked shape with one wave per SIMD (which a call can ask for, and which is 256 x 256 again for what it does not take)
    if (config == RLK_GEMM_CFG_256x256 && four_waves && solo_tiles_pay(tile_count(M, N, 256, 256), device_cu_count()))
      config = RLK_GEMM_CFG_256x256_SOLO;
  }
  if (config == RLK_GEMM_CFG_STREAM16_DEEP || config == RLK_GEMM_CFG_STREAM16 || config == RLK_GEMM_CFG_STREAM64) {
    // The streaming kernel serves up to 16 (STREAM16*) or 64 tokens and needs the fast layout;
    // otherwise a tile kernel computes the same bits.
    const int max_m = config == RLK_GEMM_CFG_STREAM64 ? 64 : 16;
    if (M <= max_m && vec && allow_pingpong && K % kTileK == 0)
      return det_gemm_stream_launch(W, X, C, ldc, M, N, K, out_f32, config == RLK_GEMM_CFG_STREAM16, stream);
    config = M <= 16 ? RLK_GEMM_CFG_16x16 : M <= 64 ? RLK_GEMM_CFG_64x64 : pick_det_gemm_config(M, N, K, false);
    if (config == RLK_GEMM_CFG_STREAM64) config = RLK_GEMM_CFG_64x64;
  }
  // Deep-stage variants need the fast layout and whole stages; otherwise the plain shape
  // computes the same bits.
  if (config == RLK_GEMM_CFG_32x32_DEEP || config == RLK_GEMM_CFG_32x64_DEEP || config == RLK_GEMM_CFG_64x32_DEEP ||
      config == RLK_GEMM_CFG_64x64_DEEP || config == RLK_GEMM_CFG_64x96_DEEP || config == RLK_GEMM_CFG_96x64_DEEP || config == RLK_GEMM_CFG_64x160_DEEP ||
      config == RLK_GEMM_CFG_128x64_DEEP || config == RLK_GEMM_CFG_128x128_DEEP) {
    const int ks = config == RLK_GEMM_CFG_32x64_DEEP || config == RLK_GEMM_CFG_64x32_DEEP || config == RLK_GEMM_CFG_64x64_DEEP
                       ? kDeep64
                       : kDeep128;
    if (vec && allow_pingpong && K % (kTileK * ks) == 0) {
      if (config == RLK_GEMM_CFG_32x32_DEEP)
        return launch_quad<Quad32x32, kDeep128, 8, false>(W, X, C, ldc, M, N, K, out_f32, stream);
      if (config == RLK_GEMM_CFG_32x64_DEEP) return launch_quad<Quad32x64, kDeep64, 3>(W, X, C, ldc, M, N, K, out_f32, stream);
      if (config == RLK_GEMM_CFG_64x32_DEEP) return launch_quad<Quad64x32, kDeep64, 3>(W, X, C, ldc, M, N, K, out_f32, stream);
      if (config == RLK_GEMM_CFG_64x96_DEEP) return launch_quad<Quad64x96, kDeep128, 3>(W, X, C, ldc, M, N, K, out_f32, stream);
      // (the prefetching wave loses here: four readers at most)
      if (config == RLK_GEMM_CFG_96x64_DEEP) return launch_quad<Quad96x64, 1, 7, false>(W, X, C, ldc, M, N, K, out_f32, stream);
      if (config == RLK_GEMM_CFG_64x160_DEEP) return launch_quad<Quad64x160, 1, 5>(W, X, C, ldc, M, N, K, out_f32, stream);
      if (config == RLK_GEMM_CFG_128x64_DEEP) {
        // Four waves gain nothing from HBM with two token tiles and lose from the cache (12288 outputs, K = 4096, 100 tokens:
        // 31.7 / 23.7 us with eight waves, 32.0 / 26.5 with four and the prefetch).
        if (M <= 2 * Shape128x64::BM) return launch_deep<Shape128x64, kDeep128, 3>(W, X, C, ldc, M, N, K, out_f32, stream);
        return out_f32 ? launch_tile<Quad128x64, kLoopQuadPrefetch, true, 1, 6>(W, X, C, ldc, M, N, K, stream)
                       : launch_tile<Quad128x64, kLoopQuadPrefetch, false, 1, 6>(W, X, C, ldc, M, N, K, stream);
      }
      if (config == RLK_GEMM_CFG_64x64_DEEP) return launch_deep<Shape64x64, kDeep64>(W, X, C, ldc, M, N, K, out_f32, stream);
      return launch_deep<Shape128x128, kDeep128>(W, X, C, ldc, M, N, K, out_f32, stream);
    }
    config = config == RLK_GEMM_CFG_128x128_DEEP || config == RLK_GEMM_CFG_64x160_DEEP     ? RLK_GEMM_CFG_128x128
             : config == RLK_GEMM_CFG_128x64_DEEP || config == RLK_GEMM_CFG_64x96_DEEP || config == RLK_GEMM_CFG_96x64_DEEP ? RLK_GEMM_CFG_128x64
                                                                                       : RLK_GEMM_CFG_64x64;
  }
  if (config == RLK_GEMM_CFG_256x256_SOLO) {
    if (vec && allow_pingpong && four_waves_take(W, X, K, out_f32))
      return launch_solo<SoloLayout<false, false>>(W, X, C, ldc, M, N, K, stream);
    config = RLK_GEMM_CFG_256x256;
  }
  if (four_waves && vec && allow_pingpong && four_waves_take(W, X, K, out_f32)) {
    switch (config) {  // (weights read past the caches are the eight waves')
      case RLK_GEMM_CFG_256x192:
        return launch_solo_shape<256, 192>(W, X, C, ldc, M, N, K, stream);
      case RLK_GEMM_CFG_192x256:
        return launch_solo_shape<192, 256>(W, X, C, ldc, M, N, K, stream);
      case RLK_GEMM_CFG_192x192:
        return launch_solo_shape<192, 192>(W, X, C, ldc, M, N, K, stream);
      case RLK_GEMM_CFG_192x128:
        if (!streamed_weight(N, K, M, 128)) return launch_solo_shape<192, 128>(W, X, C, ldc, M, N, K, stream);
        break;
      default:
        break;
    }
  }
  // The element-wise loader keeps eight values per chunk in flight, and a picked 256-feature tile gives way to 128 x 128, which
  // holds them without spilling. The 192-feature and 192-token tiles, which have no such loader, become 256-feature tiles
  // behind this line and keep them: spilled registers (98 of 256 x 256) cost less there than twice the loads. Odd pitch, as
  // the large tile / as 128 x 128, us: 4096 outputs at 2817 tokens, K = 4096 604 / 829, 14336 at 3456 2459 / 3285, 24576 at 300
  // 565 / 779, 6144 at 768 (192 x 128) 295 / 567; K = 128: 36.5 / 35.4, 64: 26.5 / 25.2.
  if (!vec && (config == RLK_GEMM_CFG_256x256 || config == RLK_GEMM_CFG_256x128 || config == RLK_GEMM_CFG_256x64))
    config = RLK_GEMM_CFG_128x128;
  // A round of 256 x 128 takes 5.5 us a K tile, one of 128 x 128 4.8, full or not, so the first where it saves a round: odd pitch, as
  // 128 x 128 / 256 x 128, K = 4992, 4096 outputs at 1452 tokens (384 / 192 tiles) 775 / 429, K = 2048, 8695 outputs at 1830 (1020 / 510) 661 /
  // 393, but K = 2880, 4096 at 830 (224 / 112) 215 / 244. Not of short reductions, whose tiles are their stores: K = 200, 6141 outputs, K-major
  // tokens at 1733 62 / 73 (K = 320, a K-major weight, 2875 at 2206 60.0 / 47.6).
  if (!vec && automatic && config == RLK_GEMM_CFG_128x128 && K >= 256) {
    const int64_t cus = device_cu_count();
    const int64_t rounds128 = (tile_count(M, N, 128, 128) + cus - 1) / cus, rounds256 = (tile_count(M, N, 128, 256) + cus - 1) / cus;
    if (25 * rounds128 > 28 * rounds256) config = RLK_GEMM_CFG_256x128;
  }
  if (config == RLK_GEMM_CFG_192x128) {
    if (vec && allow_pingpong && K % kTileK == 0)
      return launch_loop<Shape192x128, kLoopPingPong, pingpong_stages<Shape192x128>()>(W, X, C, ldc, M, N, K, out_f32, stream);
    config = RLK_GEMM_CFG_256x128;
  }
  if (config == RLK_GEMM_CFG_256x192) {
    if (vec && allow_pingpong && K % kTileK == 0)
      return launch_loop<Shape256x192, kLoopPingPong>(W, X, C, ldc, M, N, K, out_f32, stream);
    config = RLK_GEMM_CFG_256x256;
  }
  if (config == RLK_GEMM_CFG_192x192) {
    if (vec && allow_pingpong && K % kTileK == 0)
      return launch_loop<Shape192x192, kLoopPingPong, 3>(W, X, C, ldc, M, N, K, out_f32, stream);
    config = RLK_GEMM_CFG_256x128;
  }
  if (config == RLK_GEMM_CFG_192x256) {
    if (vec && allow_pingpong && K % kTileK == 0)
      return launch_loop<Shape192x256, kLoopPingPong>(W, X, C, ldc, M, N, K, out_f32, stream);
    config = RLK_GEMM_CFG_256x256;
  }
  switch (config) {
    case RLK_GEMM_CFG_256x256:
      return launch_shape<Shape256x256>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_256x128:
      return launch_shape<Shape256x128>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_256x64:
      return launch_shape<Shape256x64, false>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_128x128:
      return launch_shape<Shape128x128>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_128x64:
      return launch_shape<Shape128x64>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_64x64:
      return launch_shape<Shape64x64>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_64x16:
      return launch_shape<Shape64x16>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    case RLK_GEMM_CFG_16x16:
      return launch_shape<Shape16x16>(W, X, C, ldc, M, N, K, vec, allow_pingpong, out_f32, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace rlk
