// SwiGLU for gfx950: the elementwise activation between the two FFN GEMMs, and the
// packed gate/up projection with the activation fused into its epilogue.
//
// Stands in for swiglu_forward / swiglu_backward / swiglu_packed_forward /
// swiglu_packed_backward (reference csrc/cuda/activation/activation.cu:20-31, 62-135;
// csrc/bindings/ops.cpp:400-419) and for the fused decode projection
// rl_engine/backends/rocm/gemm/swiglu_gemm.py:13-86.
//
// Arithmetic (token-local, so batch invariant):
//   g, u  = the bf16-ROUNDED gate and up projections, widened to fp32
//   s     = rcp(1 + e(-g))             v_rcp_f32 (within 1 ulp of the quotient);
//                                      e(x) = v_exp_f32(x * log2(e))
//   y     = bf16((g * s) * u)
//   d_up  = bf16(dy * (g * s));   d_gate = bf16((dy * u) * (s * (1 + g * (1 - s))))
// The elementwise kernels also serve fp16 and fp32 tensors (the reference dispatches on the
// element type, activation.cu:240-284): same fp32 arithmetic, one rounding to the element type.
// The fused kernel rounds its two fp32 accumulators to bf16 before the activation, so it
// returns exactly what the GEMM followed by the elementwise kernel returns.
#include "linear_logp_common.h"
#include "det_gemm_body.h"
#include "det_gemm_solo.h"
#include "rlk_host.h"

namespace rlk {

// ---------------------------------------------------------------------------
// Elementwise kernels: eight features per thread, 16-byte accesses.
// gate[m * ld_g + c], up[m * ld_u + c]: a packed [T, 2 I] buffer is the case
// up = gate + I, ld_g = ld_u = 2 I.
// ---------------------------------------------------------------------------

struct SwigluArgs {
  const char* gate;
  const char* up;
  const char* dy;  // backward only
  char* y;         // forward: y; backward: d_gate
  char* y2;        // backward: d_up
  int64_t ld_g, ld_u, ld_dy, ld_y, ld_y2;  // in elements
  int rows, cols;
};

// ELEM: rlk_dtype of the tensors. Arithmetic is fp32 for every type; results are rounded to
// the element type once (round to nearest even), fp32 results are stored as they are.
template <int ELEM>
struct ActElem;
template <>
struct ActElem<RLK_DTYPE_BF16> {
  typedef bf16_bits type;
  static __device__ __forceinline__ float widen(bf16_bits v) { return bf16_to_f32(v); }
  static __device__ __forceinline__ bf16_bits narrow(float v) { return to_bf16_bits(v); }
};
template <>
struct ActElem<RLK_DTYPE_FP16> {
  typedef _Float16 type;
  static __device__ __forceinline__ float widen(_Float16 v) { return (float)v; }
  static __device__ __forceinline__ _Float16 narrow(float v) { return (_Float16)v; }
};
template <>
struct ActElem<RLK_DTYPE_FP32> {
  typedef float type;
  static __device__ __forceinline__ float widen(float v) { return v; }
  static __device__ __forceinline__ float narrow(float v) { return v; }
};

template <int ELEM>
__device__ __forceinline__ void load8(const char* base, int64_t index, bool vec, int valid, float (&out)[8]) {
  typedef typename ActElem<ELEM>::type T;
  const T* p = reinterpret_cast<const T*>(base) + index;
  if (vec && valid >= 8) {
    T raw[8];
    constexpr int kVecs = (int)sizeof(T) * 8 / 16;  // 16-byte accesses
#pragma unroll
    for (int i = 0; i < kVecs; ++i)
      reinterpret_cast<u32x4_t*>(raw)[i] = reinterpret_cast<const u32x4_t*>(p)[i];
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = ActElem<ELEM>::widen(raw[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = i < valid ? ActElem<ELEM>::widen(p[i]) : 0.f;
  }
}

template <int ELEM>
__device__ __forceinline__ void store8(char* base, int64_t index, bool vec, int valid, const float (&v)[8]) {
  typedef typename ActElem<ELEM>::type T;
  T* p = reinterpret_cast<T*>(base) + index;
  T raw[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) raw[i] = ActElem<ELEM>::narrow(v[i]);
  if (vec && valid >= 8) {
    constexpr int kVecs = (int)sizeof(T) * 8 / 16;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) reinterpret_cast<u32x4_t*>(p)[i] = reinterpret_cast<const u32x4_t*>(raw)[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (i < valid) p[i] = raw[i];
  }
}

template <bool BACKWARD, int ELEM>
__global__ __launch_bounds__(256) void swiglu_kernel(SwigluArgs a, bool vec) {
  const int groups = (a.cols + 7) / 8;
  const int64_t total = (int64_t)a.rows * groups;
  for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * 256) {
    const int row = (int)(idx / groups);
    const int col = (int)(idx - (int64_t)row * groups) * 8;
    const int valid = a.cols - col;
    float g[8], u[8];
    load8<ELEM>(a.gate, (int64_t)row * a.ld_g + col, vec, valid, g);
    load8<ELEM>(a.up, (int64_t)row * a.ld_u + col, vec, valid, u);
    if (!BACKWARD) {
      float y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) y[i] = swiglu_f32(g[i], u[i]);
      store8<ELEM>(a.y, (int64_t)row * a.ld_y + col, vec, valid, y);
    } else {
      float dy[8], dg[8], du[8];
      load8<ELEM>(a.dy, (int64_t)row * a.ld_dy + col, vec, valid, dy);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float s = sigmoid_f32(g[i]);
        du[i] = dy[i] * (g[i] * s);
        dg[i] = (dy[i] * u[i]) * (s * (1.0f + g[i] * (1.0f - s)));
      }
      store8<ELEM>(a.y, (int64_t)row * a.ld_y + col, vec, valid, dg);
      store8<ELEM>(a.y2, (int64_t)row * a.ld_y2 + col, vec, valid, du);
    }
  }
}

// Rows start on 16-byte boundaries and hold whole 16-byte vectors.
static bool rows_aligned16(const void* p, int64_t ld, int elem_bytes) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (ld * elem_bytes) % 16 == 0;
}

template <int ELEM>
static void launch_swiglu_typed(const SwigluArgs& a, bool vec, bool backward, unsigned blocks, hipStream_t stream) {
  if (backward) {
    hipLaunchKernelGGL((swiglu_kernel<true, ELEM>), dim3(blocks), dim3(256), 0, stream, a, vec);
  } else {
    hipLaunchKernelGGL((swiglu_kernel<false, ELEM>), dim3(blocks), dim3(256), 0, stream, a, vec);
  }
}

hipError_t swiglu_launch(const void* gate, int64_t ld_g, const void* up, int64_t ld_u, const void* dy, int64_t ld_dy,
                         void* out, int64_t ld_out, void* out2, int64_t ld_out2, int rows, int cols, bool backward,
                         int dtype, hipStream_t stream) {
  if (rows == 0 || cols == 0) return hipSuccess;
  SwigluArgs a;
  a.gate = reinterpret_cast<const char*>(gate);
  a.up = reinterpret_cast<const char*>(up);
  a.dy = reinterpret_cast<const char*>(dy);
  a.y = reinterpret_cast<char*>(out);
  a.y2 = reinterpret_cast<char*>(out2);
  a.ld_g = ld_g;
  a.ld_u = ld_u;
  a.ld_dy = ld_dy;
  a.ld_y = ld_out;
  a.ld_y2 = ld_out2;
  a.rows = rows;
  a.cols = cols;
  const int eb = dtype == RLK_DTYPE_FP32 ? 4 : 2;
  bool vec = rows_aligned16(gate, ld_g, eb) && rows_aligned16(up, ld_u, eb) && rows_aligned16(out, ld_out, eb);
  if (backward) vec = vec && rows_aligned16(dy, ld_dy, eb) && rows_aligned16(out2, ld_out2, eb);
  const int64_t total = (int64_t)rows * ((cols + 7) / 8);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  switch (dtype) {
    case RLK_DTYPE_BF16:
      launch_swiglu_typed<RLK_DTYPE_BF16>(a, vec, backward, (unsigned)blocks, stream);
      break;
    case RLK_DTYPE_FP16:
      launch_swiglu_typed<RLK_DTYPE_FP16>(a, vec, backward, (unsigned)blocks, stream);
      break;
    case RLK_DTYPE_FP32:
      launch_swiglu_typed<RLK_DTYPE_FP32>(a, vec, backward, (unsigned)blocks, stream);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Packed gate/up projection with the activation in the epilogue.
// W is the packed weight [2 * I, K]; a workgroup owns S::BN / 2 features of both halves.
// ---------------------------------------------------------------------------

template <class S, bool WSTREAM>
__global__ __launch_bounds__(S::kThreads) void det_gemm_swiglu_kernel(MatView W, MatView X, bf16_bits* __restrict__ Y,
                                                                       int64_t ldy, int M, int I, int K, int tiles_m,
                                                                       int tiles_n, int group_m) {
  static_assert(S::TN == 4 && pingpong_supported<S>(), "gated tiles use the 4 x 2 ping-pong layout");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int kTileFeatures = S::BN / 2;

  const int total = tiles_m * tiles_n;
  const int id = xcd_compact_id(blockIdx.x, total);
  const int per_group = group_m * tiles_n;
  const int group = id / per_group;
  const int first_m = group * group_m;
  const int width = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
  const int within = id - group * per_group;
  const int tile_m = first_m + within % width;
  const int tile_n = within / width;
  const int f0 = tile_n * kTileFeatures;
  const int m0 = tile_m * S::BM;

  f32x4_t acc[S::TN][S::TM];
  tile_mainloop_pingpong<S, false, false, GatedRowMap<S>, 1, 2, WSTREAM>(W, X, f0, m0, K, lds, acc);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wave_n = wave % S::WN;
  const int wave_m = wave / S::WN;
  const int f_run = f0 + wave_n * 32 + (lane >> 4) * 8;  // first of this lane's 8 consecutive features
  const int m_lane = m0 + wave_m * 16 * S::TM + (lane & 15);
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int m = m_lane + jm * 16;
    if (m >= M) continue;
    float y[8];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        y[h * 4 + q] = swiglu_f32(round_through_bf16(acc[h][jm][q]), round_through_bf16(acc[h + 2][jm][q]));
    const int64_t at = (int64_t)m * ldy + f_run;
    store8<RLK_DTYPE_BF16>(reinterpret_cast<char*>(Y), at, (reinterpret_cast<uintptr_t>(Y + at) & 15) == 0, I - f_run, y);
  }
}

// The same with one wave per SIMD, a workgroup per CU (det_gemm_solo.h). Training: gate and up weights apart, and both projections
// are stored beside the activation, for the backward.
struct GatedTraining {
  const bf16_bits* up_weight;
  bf16_bits *gate, *up;
};

// KT MFMA tiles of 16 features each, a lane's 4 KT of them consecutive, at `row`, the wave's first feature of a token.
template <int KT>
__device__ __forceinline__ void store_gated_span(bf16_bits* row, int grp, bool live, const f32x4_t (&y)[KT]) {
  bf16_bits* const mine = row + grp * (4 * KT);
  if constexpr (KT == 4) {
    solo_store_span(row, grp, live, y[0], y[1], y[2], y[3]);
  } else if constexpr (KT == 2) {
    if (live)
      *reinterpret_cast<u32x4_t*>(mine) = u32x4_t{pack_bf16x2(y[0][0], y[0][1]), pack_bf16x2(y[0][2], y[0][3]),
                                                  pack_bf16x2(y[1][0], y[1][1]), pack_bf16x2(y[1][2], y[1][3])};
  } else if (live) {  // 24 bytes, or 8
#pragma unroll
    for (int jn = 0; jn < KT; ++jn)
      *reinterpret_cast<u32x2_t*>(mine + jn * 4) = u32x2_t{pack_bf16x2(y[jn][0], y[jn][1]), pack_bf16x2(y[jn][2], y[jn][3])};
  }
}

template <int KT>
__device__ __forceinline__ void store_gated_run(bf16_bits* to, int inside, int alignment, const f32x4_t (&y)[KT]) {
  uint32_t packed[2 * KT];
#pragma unroll
  for (int jn = 0; jn < KT; ++jn) {
    packed[2 * jn] = pack_bf16x2(y[jn][0], y[jn][1]);
    packed[2 * jn + 1] = pack_bf16x2(y[jn][2], y[jn][3]);
  }
  solo_store_run<4 * KT>(to, inside, alignment, packed);
}

template <class Layout, bool TRAINING>
__global__ __launch_bounds__(SoloShape::kThreads) void det_gemm_swiglu_solo_kernel(MatView W, MatView X,
                                                                                   bf16_bits* __restrict__ Y, int64_t ldy,
                                                                                   int M, int I, int K, int tiles_m,
                                                                                   int tiles_n, int group_m, GatedTraining training) {
  using S = typename Layout::Shape;
  constexpr int kTiles = S::TN / 2;  // MFMA tiles of a wave that hold gate features, and that hold up features
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (TRAINING && (wave & 1)) W.ptr = training.up_weight;
  auto tile_at = [&](int block, int& f0, int& m0) __attribute__((always_inline)) {
    const TileOrder at = tile_order(block, tiles_m, tiles_n, group_m);
    f0 = at.tile_n * (S::BN / 2);
    m0 = at.tile_m * S::BM;
  };
  auto done = [&](int block, SoloAccOf<S>& acc, char*) __attribute__((always_inline)) -> bool {
    int f0, m0;
    tile_at(block, f0, m0);
    const int lane = solo_lane(), grp = lane >> 4;
    const int f_wave = f0 + wave % S::WN * (16 * kTiles), m_wave = m0 + wave / S::WN * (16 * S::TM);
    const int m_lane = m_wave + (lane & 15);
    const bool whole = f_wave + 16 * kTiles <= I && (reinterpret_cast<uintptr_t>(Y) & 15) == 0 && (ldy & 7) == 0;
    auto activate = [&](int jm, f32x4_t (&y)[kTiles], f32x4_t (&g)[kTiles], f32x4_t (&u)[kTiles]) __attribute__((always_inline)) {
#pragma unroll
      for (int jn = 0; jn < kTiles; ++jn)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          g[jn][q] = round_through_bf16(acc[jn][jm][q]);
          u[jn][q] = round_through_bf16(acc[jn + kTiles][jm][q]);
          y[jn][q] = swiglu_f32(g[jn][q], u[jn][q]);
        }
    };
    if (whole) {
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        f32x4_t y[kTiles], g[kTiles], u[kTiles];
        activate(jm, y, g, u);
        const int m = m_lane + jm * 16;
        const int64_t at = (int64_t)m * ldy + f_wave;
        store_gated_span<kTiles>(Y + at, grp, m < M, y);
        if constexpr (TRAINING) {
          store_gated_span<kTiles>(training.gate + at, grp, m < M, g);
          store_gated_span<kTiles>(training.up + at, grp, m < M, u);
        }
      }
      return m_wave + 16 * S::TM <= M;
    }
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      f32x4_t y[kTiles], g[kTiles], u[kTiles];
      activate(jm, y, g, u);
      const int m = m_lane + jm * 16, f = f_wave + grp * (4 * kTiles);
      if (m >= M) continue;
      const int64_t at = (int64_t)m * ldy + f;
      store_gated_run<kTiles>(Y + at, I - f, solo_row_alignment(Y, ldy), y);
      if constexpr (TRAINING) {
        store_gated_run<kTiles>(training.gate + at, I - f, solo_row_alignment(training.gate, ldy), g);
        store_gated_run<kTiles>(training.up + at, I - f, solo_row_alignment(training.up, ldy), u);
      }
    }
    return false;
  };
  // (the three pieces of twelve features may leave as two stores)
  constexpr int kStores = (kTiles > 2 ? 2 : 1) * S::TM * (TRAINING ? 3 : 1);
  solo_tiles<SoloGatedRows<S, TRAINING>, kStores, false, Layout>(W, X, K, blockIdx.x, gridDim.x, tiles_m * tiles_n, lds, tile_at, done);
}

// The same for few tokens: four waves over one wave column of BN / 2 gate rows and the up rows of the same features, all of
// the tokens of a launch in one tile.
// Bound by HBM: the weight is read once (201 MB of gate_up in 39 us, 5.2 TB/s), four waves read every weight row from LDS
// (448 + 160 rows a K tile of 96 x 64, 608 of about 1300 cycles that its 12 KiB of weight take at that rate).
template <class S, int KS, int NS, bool WSTREAM>
__global__ __launch_bounds__(S::kThreads) void det_gemm_swiglu_few_kernel(MatView W, MatView X, bf16_bits* __restrict__ Y,
                                                                           int64_t ldy, int M, int I, int K) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int kTiles = S::TN / 2;
  const int f0 = xcd_compact_id(blockIdx.x, gridDim.x) * (S::BN / 2);

  f32x4_t acc[S::TN][S::TM];
  tile_mainloop_quad<S, KS, NS, WSTREAM, GatedSharedRowMap<S>>(W, X, f0, 0, K, lds, acc);

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int f_run = f0 + (lane >> 4) * 4 * kTiles;  // first of this lane's 4 kTiles consecutive features
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int m = (wave * S::TM + jm) * 16 + (lane & 15);
    if (m >= M) continue;
    bf16_bits* out = Y + (int64_t)m * ldy + f_run;
    const bool whole = f_run + 4 * kTiles <= I && (reinterpret_cast<uintptr_t>(out) & 7) == 0;
#pragma unroll
    for (int t = 0; t < kTiles; ++t) {
      float y[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        y[q] = swiglu_f32(round_through_bf16(acc[t][jm][q]), round_through_bf16(acc[t + kTiles][jm][q]));
      const uint32_t packed[2] = {pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
      if (whole) {
        *reinterpret_cast<u32x2_t*>(out + t * 4) = u32x2_t{packed[0], packed[1]};
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (f_run + t * 4 + q < I) out[t * 4 + q] = (bf16_bits)((packed[q >> 1] >> ((q & 1) * 16)) & 0xffffu);
      }
    }
  }
}

// BN rows (BN / 2 features), 64 TM tokens, KS K tiles a stage, NS stages.
template <int BN, int TM, int KS, int NS, bool WSTREAM = false>
static hipError_t launch_gated_few(const MatView& W, const MatView& X, void* Y, int64_t ldy, int M, int I, int K,
                                   hipStream_t stream) {
  using S = TileShape<BN, 64 * TM, 1, 4>;
  if constexpr (!WSTREAM) {
    if (streamed_weight(2 * (int64_t)I, K, M, S::BM)) return launch_gated_few<BN, TM, KS, NS, true>(W, X, Y, ldy, M, I, K, stream);
  }
  auto kernel = det_gemm_swiglu_few_kernel<S, KS, NS, WSTREAM>;
  constexpr int kLds = NS * KS * S::kStageBytes;
  static_assert(kLds <= 160 * 1024, "stages exceed the LDS");
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((I + BN / 2 - 1) / (BN / 2)), dim3(S::kThreads), kLds, stream, W, X,
                     reinterpret_cast<bf16_bits*>(Y), ldy, M, I, K);
  return hipGetLastError();
}

template <int BN, int BM, bool TRAINING>
static hipError_t launch_gated_solo(const MatView& W, const MatView& X, void* Y, int64_t ldy, int M, int I, int K,
                                    const GatedTraining& training, hipStream_t stream) {
  using Layout = SoloLayout<false, false, TileShape<BN, BM, 2, 2>>;
  auto kernel = det_gemm_swiglu_solo_kernel<Layout, TRAINING>;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), Layout::kLds, once);
  if (err != hipSuccess) return err;
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (I + BN / 2 - 1) / (BN / 2);
  const int cus = device_cu_count();
  const int grid = tiles_m * tiles_n < cus ? tiles_m * tiles_n : cus;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(SoloShape::kThreads), Layout::kLds, stream, W, X,
                     reinterpret_cast<bf16_bits*>(Y), ldy, M, I, K, tiles_m, tiles_n, tiles_m < 8 ? tiles_m : 8, training);
  return hipGetLastError();
}

using GatedShape256 = TileShape<256, 256, 4, 2>;

template <class S, bool WSTREAM = false>
static hipError_t launch_gated(const MatView& W, const MatView& X, void* Y, int64_t ldy, int M, int I, int K,
                               hipStream_t stream) {
  if constexpr (!WSTREAM) {
    if (streamed_weight(2 * (int64_t)I, K, M, S::BM)) return launch_gated<S, true>(W, X, Y, ldy, M, I, K, stream);
  }
  auto kernel = det_gemm_swiglu_kernel<S, WSTREAM>;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), S::kLdsBytes, once);
  if (err != hipSuccess) return err;
  const int tiles_m = (M + S::BM - 1) / S::BM;
  const int tiles_n = (I + S::BN / 2 - 1) / (S::BN / 2);
  const int group_m = tiles_m < 8 ? tiles_m : 8;
  hipLaunchKernelGGL(kernel, dim3(tiles_m * tiles_n), dim3(S::kThreads), S::kLdsBytes, stream, W, X,
                     reinterpret_cast<bf16_bits*>(Y), ldy, M, I, K, tiles_m, tiles_n, group_m);
  return hipGetLastError();
}

// The tiles of the fused gate/up above 128 tokens, weight rows (gate and up) x tokens on four waves, and what a round of them takes
// relative to 256 x 256 (us at K = 4096); a round that fills part of the chip takes its share of that, and no less than
// kGatedPartial. Fitted to 140 shapes (I = 3072, 6144, 12288 with K = 4096, 6144 with 2048; 130 to 8200 tokens), 0.6 % above the
// best tile of each. What takes the time of the small ones is the loads of one round, so a tile no larger than gives every CU one.
// Eight waves in 256 rows x 256 / 192 / 128 / 64 tokens -> these, us, weights in turn: I = 3072 at 146 / 228 / 411 / 605 / 947 / 1214 tokens
// 58.7 / 58.0 / 57.5 / 57.9 / 56.9 / 59.5 -> 27.2 / 27.1 / 36.0 / 37.7 / 48.2 / 54.6, 6144 at 150 / 250 / 349 / 725 / 1319 59.7 / 59.7 / 56.7
// / 68.5 / 132 -> 35.1 / 41.4 / 49.2 / 59.7 / 111, 12288 at 231 / 310 / 474 / 987 66.2 / 73.8 / 87.1 / 171 -> 60.9 / 66.3 / 77.6 / 149, K = 2048
// at 163 / 448 / 1929 32.7 / 32.1 / 93.5 -> 20.3 / 27.3 / 77.3. (The projection and the activation as two launches: 27.1 at I = 3072
// and 146 tokens, 39 to 42 at 6144 up to 254, elsewhere slower.)
typedef hipError_t (*GatedLaunch)(const MatView&, const MatView&, void*, int64_t, int, int, int, const GatedTraining&, hipStream_t);
struct GatedTile {
  int bn, bm;
  double us;
  GatedLaunch launch, launch_training;
};
template <int BN, int BM>
constexpr GatedTile gated_tile(double us) {
  return {BN, BM, us, launch_gated_solo<BN, BM, false>, launch_gated_solo<BN, BM, true>};
}
static const GatedTile kGatedTiles[] = {
    gated_tile<256, 256>(97.0),
    gated_tile<192, 256>(78.4),
    gated_tile<256, 192>(79.0),
    gated_tile<192, 192>(60.0),
    gated_tile<256, 128>(59.0),
    gated_tile<192, 128>(46.6),
    gated_tile<128, 192>(47.7),
    gated_tile<128, 128>(36.1),
    gated_tile<64, 192>(24.5),
    gated_tile<64, 128>(20.0),
};
constexpr double kGatedPartial = 0.82;
static const GatedTile& pick_gated_tile(int M, int I, int cus) {
  const GatedTile* best = kGatedTiles;
  double best_us = 1e300;
  for (const GatedTile& t : kGatedTiles) {
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((I + t.bn / 2 - 1) / (t.bn / 2));
    const double us = rounds_of_workgroups(tiles, cus, kGatedPartial) * t.us;
    if (us < best_us * 0.999) {
      best_us = us;
      best = &t;
    }
  }
  return *best;
}

// Up to 16 tokens the streaming kernel serves the packed projection (the same panels of 16 weight
// rows, eight gate and eight up), from 129 tokens on the gated tile kernels.
static bool streams_gated(int M, int K) { return M <= 16 && K >= 1024; }
// From 17 to 128 tokens a gated tile on four waves, no wider than gives every CU one: gate_up of 12288 at 64 tokens ran on 192
// of 256 CUs as 128-row tiles, and the projection was written, read again and activated by a second launch. Weights from
// HBM, two launches -> one, us (K = 4096, I = 12288 / 6144 / 3072): 17 tokens 42.1 / 23.6 / 15.0 -> 37.1 / 20.8 / 13.7, 64: 45.4
// / 27.6 / 20.8 -> 39.1 / 25.8 / 17.6, 128: 50.5 / 37.4 / 23.4 -> 45.0 / 32.6 / 25.0 (not used: the many token rows beside 32
// weight rows per tile; K = 2048: 12.6 -> 10.5).
static bool few_gated(int M, int I, int K) {
  return M > 16 && M <= 128 && K % 128 == 0 && K >= 512 && (M <= 96 || K <= 2048 || I > 16 * device_cu_count());
}

bool det_gemm_swiglu_fused_supported(const MatView& W, const MatView& X, int M, int K) {
  auto native = [](const MatView& v) {
    return v.k_stride == 1 && (v.row_stride % kChunkElems) == 0 && pitch_fits_lane_offsets(v.row_stride) &&
           (reinterpret_cast<uintptr_t>(v.ptr) & 15) == 0;
  };
  return native(W) && native(X) && (K % kTileK) == 0 && (M > 128 || streams_gated(M, K) || few_gated(M, W.rows / 2, K));
}

// Y[M, I] = swiglu(X @ W[0:I]^T, X @ W[I:2I]^T). `workspace` ([M, 2 I] bf16) is used only when
// the fused kernels do not apply (other layouts, ragged K, 97 to 128 tokens of a small weight), where the
// projection and the activation run as two kernels with the same result.
hipError_t det_gemm_swiglu_launch(const MatView& W, const MatView& X, void* Y, int64_t ldy, void* workspace, int M,
                                  int I, int K, hipStream_t stream) {
  if (det_gemm_swiglu_fused_supported(W, X, M, K)) {
    if (streams_gated(M, K)) return det_gemm_stream_gated_launch(W, X, Y, ldy, M, I, K, stream);
    if (few_gated(M, I, K)) {
      const int cus = device_cu_count();
      if (M <= 64) {
        if (I <= 16 * cus) return launch_gated_few<32, 1, 2, 6>(W, X, Y, ldy, M, I, K, stream);
        if (I <= 32 * cus) return launch_gated_few<64, 1, 2, 4>(W, X, Y, ldy, M, I, K, stream);
        if (I <= 48 * cus) return launch_gated_few<96, 1, 1, 7>(W, X, Y, ldy, M, I, K, stream);
        return launch_gated_few<128, 1, 1, 6>(W, X, Y, ldy, M, I, K, stream);
      }
      if (I <= 16 * cus) return launch_gated_few<32, 2, 1, 7>(W, X, Y, ldy, M, I, K, stream);
      if (I <= 32 * cus) return launch_gated_few<64, 2, 1, 6>(W, X, Y, ldy, M, I, K, stream);
      if (I <= 48 * cus) return launch_gated_few<96, 2, 1, 5>(W, X, Y, ldy, M, I, K, stream);
      return launch_gated_few<128, 2, 1, 4>(W, X, Y, ldy, M, I, K, stream);
    }
    const int cus = device_cu_count();
    const bool fits = solo_offsets_fit(W, (int64_t)I + 128) && solo_offsets_fit(X);
    const int64_t t256 = (int64_t)((M + 255) / 256) * ((I + 127) / 128);
    const GatedTile& tile = fits ? pick_gated_tile(M, I, cus) : kGatedTiles[0];
    // (256 x 256 on eight waves: few tiles, a weight that is read past the caches, operands of 4 GiB)
    if (tile.launch == kGatedTiles[0].launch && !(fits && solo_tiles_pay(t256, cus) && !streamed_weight(2 * (int64_t)I, K, M, 256)))
      return launch_gated<GatedShape256>(W, X, Y, ldy, M, I, K, stream);
    return tile.launch(W, X, Y, ldy, M, I, K, GatedTraining{}, stream);
  }
  if (workspace == nullptr) return hipErrorInvalidValue;
  hipError_t err = det_gemm_launch(W, X, workspace, 2 * (int64_t)I, M, 2 * I, K, false, RLK_GEMM_CFG_AUTO, stream);
  if (err != hipSuccess) return err;
  const bf16_bits* gu = reinterpret_cast<const bf16_bits*>(workspace);
  return swiglu_launch(gu, 2 * (int64_t)I, gu + I, 2 * (int64_t)I, nullptr, 0, Y, ldy, nullptr, 0, M, I, false,
                       RLK_DTYPE_BF16, stream);
}

// gate[M, I], up[M, I] and Y[M, I] = swiglu(gate, up) of two weights, in one launch above 128 tokens: the activation's launch read both
// projections again, and tiles of both together fill the chip better than those of each. Three launches -> one, us (tokens, I, K):
// 4096, 12288, 4096 629 -> 601; 2026, 12288, 4096 337 -> 296; 359, 12288, 4096 109 -> 75; 803, 6144, 4096 98 -> 80; 923, 3072, 4096 73 -> 51; 215, 3072,
// 4096 37 -> 26; 736, 6144, 2048 62 -> 41; of 46 shapes none slower (2110, 12288, 4096: 371 both).
hipError_t det_gemm_swiglu_training_launch(const MatView& W_gate, const MatView& W_up, const MatView& X, void* gate, void* up, void* Y,
                                           int64_t ldy, int M, int I, int K, hipStream_t stream) {
  // (what holds of the gate weight's rows holds of the up weight's: the same pitch, and the alignment is looked at)
  const bool fused = M > 128 && det_gemm_swiglu_fused_supported(W_gate, X, M, K) && (reinterpret_cast<uintptr_t>(W_up.ptr) & 15) == 0 &&
                     ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up)) & 15) == 0 && solo_offsets_fit(W_gate) &&
                     solo_offsets_fit(X);
  if (fused) {
    const GatedTraining training{W_up.ptr, reinterpret_cast<bf16_bits*>(gate), reinterpret_cast<bf16_bits*>(up)};
    return pick_gated_tile(M, I, device_cu_count()).launch_training(W_gate, X, Y, ldy, M, I, K, training, stream);
  }
  hipError_t err = det_gemm_launch(W_gate, X, gate, ldy, M, I, K, false, RLK_GEMM_CFG_AUTO, stream);
  if (err != hipSuccess) return err;
  err = det_gemm_launch(W_up, X, up, ldy, M, I, K, false, RLK_GEMM_CFG_AUTO, stream);
  if (err != hipSuccess) return err;
  return swiglu_launch(gate, ldy, up, ldy, nullptr, 0, Y, ldy, nullptr, 0, M, I, false, RLK_DTYPE_BF16, stream);
}

}  // namespace rlk
