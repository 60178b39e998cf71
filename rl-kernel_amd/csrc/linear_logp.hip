// Fused linear-LogP for gfx950: lm_head GEMM -> online log-sum-exp over the
// vocabulary in a fixed order -> target-token gather. The [tokens, vocab] logits
// never leave registers.
//
// Stands in for rl_engine._C.fused_linear_logp_sm90 (reference
// csrc/cuda/logprob/fused_linear_logp_sm90.cu:104-325, 488-513, 2040-2176), for
// triton_deterministic_linear_logp (rl_engine/backends/shared/triton/logprob/
// linear_logp.py:277-418, 631-700) and for the unfused ROCm route
// DetGemmOp().linear + hip_deterministic_logp_tile_stats
// (rl_engine/integrations/common/linear_logp.py:1083-1102).
//
// Reduction contract (everything that decides the bits of logp / lse; all of it
// is a function of the vocabulary axis only, never of the token count, the
// position of a token in the batch or the launch geometry):
//   z_v   = fp32 MFMA chain of det_gemm over the hidden dimension, + bias_v
//   y_v   = z_v                      (v < real vocabulary bound)
//         = -inf                     (padded lane)
//         then y_v * (1 / temperature) when a temperature is given
//   tile  = 256 consecutive vocabulary columns; stream j (0..15) of a tile is
//           its columns [16 j, 16 j + 16)
//   split = 4 consecutive tiles (1024 columns); n_split = ceil(V / 1024)
//   stream chain (per split, per j), tiles ascending, state (m, s) = (-inf, 0):
//           t = max of the 16 y;  n = max(m, t);
//           if n > -inf:  s = s * e(m - n) + (((e(y0 - n) + e(y1 - n)) + ...) + e(y15 - n));  m = n
//   split merge:  M = max_j m_j;  S = sum over j ascending of s_j * e(m_j - M)  (terms with m_j = -inf skipped)
//   final merge over splits ascending with the same formula;
//   lse = M + log(S);  zt = y_target;  logp = min(zt - lse, 0)
//   e(x) = v_exp_f32(x * log2(e)) with an unfused fp32 multiply.
#include "det_gemm_solo.h"
#include "linear_logp_common.h"
#include "rlk_host.h"

namespace rlk {

struct LogpArgs {
  MatView W;  // [V, D] lm_head weight, rows = vocabulary
  MatView H;  // [T, D] hidden states, rows = tokens
  const int64_t* target;     // [T] global vocabulary ids
  const float* bias;         // [V] or null
  const float* temperature;  // [T] or null
  float* part;               // [3][n_split][T]: max, sum, target logit
  float* logits;             // [T, logits_ld] fp32 biased logits (no temperature), or null: not wanted
  int64_t logits_ld;
  int T, V, D;
  int vocab_limit;  // local column bound of the real vocabulary (<= V)
  int64_t vocab_start;
  int tiles_m, n_split, group_m;
};

// One (token tile, split). LOOP: 0 generic element loader, 1 register-staged 16-byte loads, 2 direct-to-LDS ping-pong.
template <class S, int LOOP>
__device__ __forceinline__ void logp_partial_tile(const LogpArgs& a, int m0, int split, char* lds) {
  static_assert(S::BN == kLogpTileCols && S::kRun == 16 && S::WN == 4, "stream layout is pinned");
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wave_n = wave % S::WN;
  const int wave_m = wave / S::WN;
  const int l16 = lane & 15;
  const int grp = lane >> 4;
  const int stream = wave_n * 4 + grp;
  const int tok_local = wave_m * 16 * S::TM + l16;

  float run_m[S::TM], run_s[S::TM], run_zt[S::TM], inv_t[S::TM];
  int tgt[S::TM];
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int m = m0 + tok_local + jm * 16;
    run_m[jm] = kNegInf;
    run_s[jm] = 0.f;
    run_zt[jm] = 0.f;
    inv_t[jm] = 1.0f;
    tgt[jm] = -1;
    if (m < a.T) {
      const int64_t local = a.target[m] - a.vocab_start;
      tgt[jm] = (local >= 0 && local < a.vocab_limit) ? (int)local : -1;
      if (a.temperature) inv_t[jm] = 1.0f / a.temperature[m];
    }
  }

  for (int t = 0; t < kLogpSplitTiles; ++t) {
    const int v0 = split * kLogpSplitCols + t * kLogpTileCols;
    if (v0 >= a.V) break;
    f32x4_t acc[S::TN][S::TM];
    if constexpr (LOOP == 2) {
      tile_mainloop_pingpong<S>(a.W, a.H, v0, m0, a.D, lds, acc);
    } else {
      tile_mainloop_staged<S, LOOP == 1>(a.W, a.H, v0, m0, a.D, lds, acc);
    }

    const int col0 = v0 + stream * 16;  // first column of this lane's run
    const int span0 = v0 + wave_n * 64;  // first column of the wave's four runs
    // whole spans into 16-byte aligned rows are stored by the four lanes of a token together (wave uniform)
    const bool span_stores = a.logits != nullptr && span0 + 64 <= a.V && (a.logits_ld & 3) == 0 &&
                             (reinterpret_cast<uintptr_t>(a.logits) & 15) == 0;
    float bias_run[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) bias_run[c] = 0.f;
    if (a.bias) {
#pragma unroll
      for (int c = 0; c < 16; ++c) bias_run[c] = (col0 + c < a.V) ? a.bias[col0 + c] : 0.f;
    }
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      float y[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) y[c] = biased_logit(acc[c >> 2][jm][c & 3], a.bias != nullptr, bias_run[c], col0 + c, a.vocab_limit);
      if (a.logits) {  // the same accumulators the reduction sees, stored before the temperature
        const int m = m0 + tok_local + jm * 16;
        float* row = a.logits + (int64_t)(m < a.T ? m : 0) * a.logits_ld;
        if (span_stores) store_logit_span(row, span0, grp, m < a.T, y);
        else if (m < a.T) store_logit_run(row, col0, a.V, y);
      }
      if (a.temperature) {
#pragma unroll
        for (int c = 0; c < 16; ++c) y[c] = y[c] * inv_t[jm];
      }
      logp_fold_run(y, tgt[jm] - col0, run_m[jm], run_s[jm], run_zt[jm]);
    }
  }

  // Fold the 16 streams of every token in ascending stream order. The main loop
  // ended on a barrier, so the staging LDS is free.
  float* xm = reinterpret_cast<float*>(lds);
  float* xs = xm + kLogpStreams * S::BM;
  float* xz = xs + kLogpStreams * S::BM;
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int slot = stream * S::BM + tok_local + jm * 16;
    xm[slot] = run_m[jm];
    xs[slot] = run_s[jm];
    xz[slot] = run_zt[jm];
  }
  __syncthreads();
  for (int tok = threadIdx.x; tok < S::BM; tok += S::kThreads) {
    const int m = m0 + tok;
    if (m >= a.T) continue;
    float big, sum, zt;
    logp_merge_streams(xm + tok, xs + tok, xz + tok, S::BM, big, sum, zt);
    const int64_t plane = (int64_t)a.n_split * a.T;
    const int64_t at = (int64_t)split * a.T + m;
    a.part[at] = big;
    a.part[plane + at] = sum;
    a.part[2 * plane + at] = zt;
  }
}

// ST: the tile of a last row of token tiles that has at most ST::BM tokens left (S where it is not smaller).
template <class S, class ST, int LOOP>
__global__ __launch_bounds__(S::kThreads) void linear_logp_partial_kernel(LogpArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int total = a.tiles_m * a.n_split;
  const int id = xcd_compact_id(blockIdx.x, total);
  const int per_group = a.group_m * a.n_split;
  const int group = id / per_group;
  const int first_m = group * a.group_m;
  const int width = (a.tiles_m - first_m) < a.group_m ? (a.tiles_m - first_m) : a.group_m;
  const int within = id - group * per_group;
  const int tile_m = first_m + within % width;
  const int split = within / width;
  const int m0 = tile_m * S::BM;

  if constexpr (ST::BM < S::BM) {
    if (m0 + ST::BM >= a.T) {
      logp_partial_tile<ST, LOOP>(a, m0, split, lds);
      return;
    }
  }
  logp_partial_tile<S, LOOP>(a, m0, split, lds);
}

// One wave per SIMD (det_gemm_solo.h): the loads of a unit's vocabulary tile run ahead under the tile before and its fold, and
// stored logits leave under the next tile's products. A lane holds two runs of 16 columns, i.e. two streams, of eight tokens.
// Bound by the package's power cap, with stored logits also by HBM. Ping-pong -> this, us, V = 151936, D = 4096, the same weights in one
// process: 2048 tokens 1873 -> 1854, 4200 3816 -> 3712, 8192 7064 -> 7038 (one part in 300, 1449 TFLOP/s; 7027 -> 6870 on another
// machine), 8200 7654 -> 7077; with stored logits at 2048 tokens 2152 -> 2085, 4120 4330 -> 4175. (A workgroup per CU
// that goes through many units, as in the GEMM, measures the same up to 10 rounds of them; behind 18 the workgroups that share
// panels have drifted apart: 1 % slower. The two runs of a token folded side by side: 4 % slower.)
// ST: the tile of a last row of token tiles that has at most ST::BM tokens left, a four-wave loop over 256 columns x ST::BM tokens.
template <bool LOGITS, class S>
__device__ __forceinline__ void logp_fold_tile(const LogpArgs& a, const f32x4_t (&acc)[S::TN][S::TM], int jm, int h, int span0, int col0,
                                               bool span_stores, int grp, int split, int m, int tgt, float inv_t, float& run_m,
                                               float& run_s) {
  __builtin_amdgcn_sched_barrier(0);  // one run of 16 at a time: the accumulators and the next fragments leave few registers
  float y[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) y[c] = solo_result(acc[4 * h + (c >> 2)][jm][c & 3]);
  if (span0 + 64 > a.vocab_limit) {  // uniform: the last columns
#pragma unroll
    for (int c = 0; c < 16; ++c) y[c] = col0 + c < a.vocab_limit ? y[c] : kNegInf;
  }
  if constexpr (LOGITS) {  // the same accumulators the reduction sees, stored before the temperature
    float* row = a.logits + (int64_t)(m < a.T ? m : 0) * a.logits_ld;
    if (span_stores) store_logit_span(row, span0, grp, m < a.T, y);
    else if (m < a.T) store_logit_run(row, col0, a.V, y);
  }
  // by one without a temperature: a branch around it costs the compiler its grip on the accumulators (1000 spilled registers)
#pragma unroll
  for (int c = 0; c < 16; ++c) y[c] = y[c] * inv_t;
  const int at = tgt - col0;
  float zt = 0.f;
  logp_fold_run(y, at, run_m, run_s, zt);
  if (at >= 0 && at < 16) a.part[(2 * (int64_t)a.n_split + split) * a.T + m] = zt;  // (logp_store_units() writes the others' zeros)
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ int logp_target(const LogpArgs& a, int m) {
  if (m >= a.T) return -1;
  const int64_t local = a.target[m] - a.vocab_start;
  return local >= 0 && local < a.vocab_limit ? (int)local : -1;
}
__device__ __forceinline__ float logp_inverse_temperature(const LogpArgs& a, int m) {
  return m < a.T && a.temperature ? 1.0f / a.temperature[m] : 1.0f;
}

// The stream merge of `tokens` tokens whose states lie in LDS, streams `tokens` floats apart; token i of them is row m_of(i). A target
// among the columns [v_first, v_end) of the unit has had its logit stored by the fold.
template <class RowOf>
__device__ __forceinline__ void logp_store_units(const LogpArgs& a, int split, int v_first, int v_end, const float* xm, const float* xs,
                                                 int tokens, RowOf m_of) {
  const int64_t plane = (int64_t)a.n_split * a.T;
  for (int i = threadIdx.x; i < tokens; i += SoloShape::kThreads) {
    const int m = m_of(i);
    if (m >= a.T) continue;
    float big, sum, unused;
    logp_merge_streams(xm + i, xs + i, xs + i, tokens, big, sum, unused);
    const int64_t at = (int64_t)split * a.T + m;
    a.part[at] = big;
    a.part[plane + at] = sum;
    const int tgt = logp_target(a, m);
    if (tgt < v_first || tgt >= v_end) a.part[2 * plane + at] = 0.f;
  }
}

template <bool LOGITS, class S, int NS>
__device__ __forceinline__ void logp_small_unit(const LogpArgs& a, int m0, int split, char* lds) {
  static_assert(S::WN == 2 && S::WM == 2 && S::TN == 8, "a lane holds two streams");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = lane >> 4;
  const int wave_n = wave % S::WN;
  const int tok_local = wave / S::WN * 16 * S::TM + (lane & 15);
  float run_m[2][S::TM], run_s[2][S::TM];
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    run_m[0][jm] = run_m[1][jm] = kNegInf;
    run_s[0][jm] = run_s[1][jm] = 0.f;
  }
  for (int t = 0; t < kLogpSplitTiles; ++t) {
    const int v0 = split * kLogpSplitCols + t * kLogpTileCols;
    if (v0 >= a.V) break;
    f32x4_t acc[S::TN][S::TM];
    tile_mainloop_quad<S, 1, NS, false>(a.W, a.H, v0, m0, a.D, lds, acc);
    const int col = v0 + wave_n * 128 + grp * 32;  // a lane's 32 consecutive columns
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      const int m = m0 + tok_local + jm * 16;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        logp_fold_tile<LOGITS, S>(a, acc, jm, h, v0 + wave_n * 128 + 64, col + 16 * h, false, grp, split, m, logp_target(a, m),
                                  logp_inverse_temperature(a, m), run_m[h][jm], run_s[h][jm]);
    }
  }
  float* const xm = reinterpret_cast<float*>(lds);  // the loop ended on a barrier
  float* const xs = xm + kLogpStreams * S::BM;
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int tok = tok_local + jm * 16;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xm[(wave_n * 8 + grp * 2 + h) * S::BM + tok] = run_m[h][jm];
      xs[(wave_n * 8 + grp * 2 + h) * S::BM + tok] = run_s[h][jm];
    }
  }
  __syncthreads();
  const int v_first = split * kLogpSplitCols;
  logp_store_units(a, split, v_first, v_first + kLogpSplitCols, xm, xs, S::BM, [&](int i) { return m0 + i; });
  __syncthreads();
}

struct LogpNoRest {
  static constexpr int BM = 0;
};

template <bool LOGITS, class ST>
__global__ __launch_bounds__(SoloShape::kThreads) void linear_logp_solo_kernel(LogpArgs a) {
  using S = SoloShape;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_n = wave % S::WN, wave_m = wave / S::WN;
  const int units = a.tiles_m * a.n_split;
  if constexpr (ST::BM > 0) {
    if ((int)blockIdx.x >= units) {
      logp_small_unit<LOGITS, ST, kSoloLdsBytes / ST::kStageBytes>(a, a.tiles_m * S::BM, blockIdx.x - units, lds);
      return;
    }
  }
  const int id = xcd_compact_id(blockIdx.x, units);
  const int per_group = a.group_m * a.n_split;
  const int group = id / per_group;
  const int first_m = group * a.group_m;
  const int width = (a.tiles_m - first_m) < a.group_m ? (a.tiles_m - first_m) : a.group_m;
  const int within = id - group * per_group;
  const int m0 = (first_m + within % width) * S::BM;
  const int split = within / width;
  if constexpr (ST::BM > 0) {
    if (m0 + ST::BM >= a.T) {
      logp_small_unit<LOGITS, ST, kSoloLdsBytes / ST::kStageBytes>(a, m0, split, lds);
      return;
    }
  }
  const int v_first = split * kLogpSplitCols;
  const int tiles = min(kLogpSplitTiles, (a.V - v_first + kLogpTileCols - 1) / kLogpTileCols);

  float run_m[2][S::TM], run_s[2][S::TM];
#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    run_m[0][jm] = run_m[1][jm] = kNegInf;
    run_s[0][jm] = run_s[1][jm] = 0.f;
  }
  auto tile_at = [&](int t, int& v0, int& m) __attribute__((always_inline)) {
    v0 = v_first + t * kLogpTileCols;
    m = m0;
  };
  auto done = [&](int t, SoloAcc& acc, char* scratch) __attribute__((always_inline)) -> bool {
    const int lane = solo_lane(), grp = lane >> 4;
    const int tok_local = wave_m * 128 + (lane & 15);
    const int span = v_first + t * kLogpTileCols + wave_n * 128;
    // (read before the first logits are stored, or each would wait for the stores before it)
    int tgt[S::TM];
    float inv_t[S::TM];
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      tgt[jm] = logp_target(a, m0 + tok_local + jm * 16);
      inv_t[jm] = logp_inverse_temperature(a, m0 + tok_local + jm * 16);
    }
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        logp_fold_tile<LOGITS, S>(a, acc, jm, h, span + h * 64, span + h * 64 + grp * 16, span + h * 64 + 64 <= a.V, grp,
                                  split, m0 + tok_local + jm * 16, tgt[jm], inv_t[jm], run_m[h][jm], run_s[h][jm]);
    if (t + 1 < tiles) return LOGITS && span + 128 <= a.V && m0 + S::BM <= a.T;

    // the 16 streams of the unit, 128 tokens at a time
    constexpr int kTokens = 128, kRows = S::TM / 2;
    float* const xm = reinterpret_cast<float*>(scratch);
    float* const xs = xm + kLogpStreams * kTokens;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        const int jm = pass * kRows + r, tok = wave_m * 64 + r * 16 + (lane & 15);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          xm[(wave_n * 8 + h * 4 + grp) * kTokens + tok] = run_m[h][jm];
          xs[(wave_n * 8 + h * 4 + grp) * kTokens + tok] = run_s[h][jm];
        }
      }
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      wg_barrier();
      logp_store_units(a, split, v_first, v_first + kLogpSplitCols, xm, xs, kTokens, [&](int i) { return m0 + (i >> 6) * 128 + pass * 64 + (i & 63); });
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      wg_barrier();
    }
    return false;
  };
  auto keep = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm)
      asm volatile("" : "+v"(run_m[0][jm]), "+v"(run_m[1][jm]), "+v"(run_s[0][jm]), "+v"(run_s[1][jm]));
  };
  solo_tiles<SoloPlainRows<SoloShape>, LOGITS ? 55 : 0, true>(a.W, a.H, a.D, 0, 1, tiles, lds, tile_at, done, keep);
}

// Few token tiles: a split of 1024 columns gives the chip only tiles_m * ceil(V / 1024)
// workgroups of four K loops each. Streams are independent until the stream merge, so here a
// workgroup takes four of the sixteen streams of a split, i.e. the 64-column slice
// [64 g, 64 g + 64) of each of the split's four tiles, as ONE 256-row GEMM tile (wave column t
// holds tile t's slice): four times the workgroups, one K loop each. The online chain of a
// (token, stream) still visits the tiles in ascending order: wave column t folds its sixteen
// columns into the state that column t - 1 left in LDS. Per-(split, stream) states go to
// linear_logp_stream_merge_kernel, which repeats the in-kernel stream merge above. Same bits
// as every other configuration.
template <class S, int NS, bool WSTREAM>
__global__ __launch_bounds__(S::kThreads) void linear_logp_streamgroup_kernel(LogpArgs a, float* __restrict__ spart,
                                                                              int split_first, int split_count) {
  static_assert(S::BN == kLogpTileCols && S::kRun == 16 && S::WN == 4, "wave column = tile of the split");
  constexpr int kGroups = kLogpStreams / 4;  // stream groups per split
  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int total = a.tiles_m * split_count * kGroups;  // this launch covers splits [split_first, + split_count)
  const int id = xcd_compact_id(blockIdx.x, total);
  const int tile_m = id % a.tiles_m;
  const int unit = id / a.tiles_m;
  const int split = split_first + unit / kGroups;
  const int sg = unit % kGroups;
  const int m0 = tile_m * S::BM;
  const int n0 = split * kLogpSplitCols + sg * 64;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int tile = wave % S::WN;
  const int wave_m = wave / S::WN;
  const int l16 = lane & 15;
  const int grp = lane >> 4;  // stream inside the group
  const int tok_local = wave_m * 16 * S::TM + l16;

  f32x4_t acc[S::TN][S::TM];
  tile_mainloop_pingpong<S, false, false, StridedColumnRowMap<S, kLogpTileCols>, 1, NS, WSTREAM>(a.W, a.H, n0, m0, a.D, lds, acc);

  const int v0 = split * kLogpSplitCols + tile * kLogpTileCols;
  const int col0 = v0 + (sg * 4 + grp) * 16;  // first column of this lane's run
  float bias_run[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) bias_run[c] = (a.bias && col0 + c < a.V) ? a.bias[col0 + c] : 0.f;

  // The main loop ended on a barrier, so the staging LDS is free: states [3][4 streams][BM].
  float* sm = reinterpret_cast<float*>(lds);
  float* ss = sm + 4 * S::BM;
  float* sz = ss + 4 * S::BM;
#pragma unroll 1
  for (int t = 0; t < kLogpSplitTiles; ++t) {
    if (tile == t && v0 < a.V) {  // a tile past the vocabulary leaves the states alone
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        const int slot = grp * S::BM + tok_local + jm * 16;
        const int m = m0 + tok_local + jm * 16;
        int tgt = -1;
        float inv_t = 1.0f;
        if (m < a.T) {
          const int64_t local = a.target[m] - a.vocab_start;
          tgt = (local >= 0 && local < a.vocab_limit) ? (int)local : -1;
          if (a.temperature) inv_t = 1.0f / a.temperature[m];
        }
        float run_m = kNegInf, run_s = 0.f, run_zt = 0.f;
        if (t > 0) {
          run_m = sm[slot];
          run_s = ss[slot];
          run_zt = sz[slot];
        }
        float y[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) y[c] = biased_logit(acc[c >> 2][jm][c & 3], a.bias != nullptr, bias_run[c], col0 + c, a.vocab_limit);
        if (a.logits && m < a.T) store_logit_run(a.logits + (int64_t)m * a.logits_ld, col0, a.V, y);
        if (a.temperature) {
#pragma unroll
          for (int c = 0; c < 16; ++c) y[c] = y[c] * inv_t;
        }
        logp_fold_run(y, tgt - col0, run_m, run_s, run_zt);
        sm[slot] = run_m;
        ss[slot] = run_s;
        sz[slot] = run_zt;
      }
    }
    __syncthreads();
  }

  const int64_t plane = (int64_t)a.n_split * kLogpStreams * a.T;
  for (int idx = threadIdx.x; idx < 4 * S::BM; idx += S::kThreads) {
    const int sl = idx / S::BM;
    const int m = m0 + idx % S::BM;
    if (m >= a.T) continue;
    const int64_t at = ((int64_t)split * kLogpStreams + sg * 4 + sl) * a.T + m;
    spart[at] = sm[idx];
    spart[plane + at] = ss[idx];
    spart[2 * plane + at] = sz[idx];
  }
}

// The same with one wave per SIMD (det_gemm_solo.h), a workgroup per CU: a wave has two of the four tiles' slices, and the state goes
// through LDS once, from the waves of tiles 0 and 1 to those of 2 and 3. The next GEMM tile's loads run under the folds.
struct SoloStreamRows {
  static __device__ __forceinline__ int64_t row(int r, int last, int) {
    return min((r >> 6) * kLogpTileCols + SoloPlainRows<SoloShape>::feature(r & 63), last);
  }
  static __device__ __forceinline__ int features(const MatView& W) { return W.rows; }
};
template <int BM>
struct LogpStreamsSolo {
  using Layout = SoloLayout<false, false, TileShape<256, BM, 2, 2>>;
  static constexpr int kStateBytes = 3 * (kLogpStreams / 4) * BM * 4;
  static constexpr int kLds = Layout::kLds + (Layout::kRing ? kStateBytes : 0);  // (else in the spare part)
  static_assert(kLds <= 160 * 1024, "a ring and the states");
};
template <bool LOGITS, int BM>
__global__ __launch_bounds__(SoloShape::kThreads) void linear_logp_streamgroup_solo_kernel(LogpArgs a, float* __restrict__ spart) {
  using L = LogpStreamsSolo<BM>;
  using S = typename L::Layout::Shape;
  constexpr int kGroups = kLogpStreams / 4;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave_n = wave % S::WN, wave_m = wave / S::WN;
  const int total = a.tiles_m * a.n_split * kGroups;
  auto unit_at = [&](int i, int& split, int& sg, int& m0) __attribute__((always_inline)) {
    const int id = xcd_compact_id(i, total), unit = id / a.tiles_m;
    m0 = id % a.tiles_m * BM;
    split = unit / kGroups;
    sg = unit % kGroups;
  };
  auto tile_at = [&](int i, int& n0, int& m0) __attribute__((always_inline)) {
    int split, sg;
    unit_at(i, split, sg, m0);
    n0 = min(split * kLogpSplitCols + sg * 64, a.V - 1);  // (columns past the vocabulary are masked)
  };
  auto done = [&](int i, SoloAccOf<S>& acc, char* spare) __attribute__((always_inline)) -> bool {
    int split, sg, m0;
    unit_at(i, split, sg, m0);
    const int lane = solo_lane(), grp = lane >> 4;
    const int tok_local = wave_m * (BM / 2) + (lane & 15);
    float* const sm = reinterpret_cast<float*>(L::Layout::kRing ? lds + L::Layout::kLds : spare);
    float *const ss = sm + kGroups * BM, *const sz = ss + kGroups * BM;
    const int span = split * kLogpSplitCols + wave_n * 2 * kLogpTileCols + sg * 64;  // of the wave's first tile
    const int64_t plane = (int64_t)a.n_split * kLogpStreams * a.T;
    const int64_t at = ((int64_t)split * kLogpStreams + sg * 4 + grp) * a.T + m0 + tok_local;
#pragma unroll 1
    for (int turn = 0; turn < 2; ++turn) {
      if (wave_n == turn) {
#pragma unroll
        for (int jm = 0; jm < S::TM; ++jm) {
          const int slot = grp * BM + tok_local + jm * 16, m = m0 + tok_local + jm * 16;
          const int tgt = logp_target(a, m);
          const float inv_t = logp_inverse_temperature(a, m);
          float run_m = kNegInf, run_s = 0.f, run_zt = 0.f;
          if (turn == 1) {
            run_m = sm[slot];
            run_s = ss[slot];
            run_zt = sz[slot];
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int span0 = span + h * kLogpTileCols, col0 = span0 + grp * 16;
            __builtin_amdgcn_sched_barrier(0);
            float y[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) y[c] = solo_result(acc[4 * h + (c >> 2)][jm][c & 3]);
            if (span0 + 64 > a.vocab_limit) {  // uniform: the last columns
#pragma unroll
              for (int c = 0; c < 16; ++c) y[c] = col0 + c < a.vocab_limit ? y[c] : kNegInf;
            }
            if constexpr (LOGITS) {
              float* row = a.logits + (int64_t)(m < a.T ? m : 0) * a.logits_ld;
              if (span0 + 64 <= a.V) store_logit_span(row, span0, grp, m < a.T, y);
              else if (m < a.T) store_logit_run(row, col0, a.V, y);
            }
#pragma unroll
            for (int c = 0; c < 16; ++c) y[c] = y[c] * inv_t;  // (by one without a temperature, see logp_fold_tile)
            logp_fold_run(y, tgt - col0, run_m, run_s, run_zt);
            __builtin_amdgcn_sched_barrier(0);
          }
          if (turn == 0) {
            sm[slot] = run_m;
            ss[slot] = run_s;
            sz[slot] = run_zt;
          } else if (m < a.T) {
            spart[at + jm * 16] = run_m;
            spart[plane + at + jm * 16] = run_s;
            spart[2 * plane + at + jm * 16] = run_zt;
          }
        }
      }
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      wg_barrier();
    }
    return LOGITS && span + kLogpTileCols + 64 <= a.V && m0 + BM <= a.T;
  };
  constexpr int kStores = LOGITS ? (8 * S::TM < 55 ? 8 * S::TM : 55) : 0;
  solo_tiles<SoloStreamRows, kStores, true, typename L::Layout>(a.W, a.H, a.D, blockIdx.x, gridDim.x, total, lds, tile_at, done);
}

// Per-(split, stream) states [3][n_split * 16][T] -> per-split partials [3][n_split][T], streams
// ascending: the arithmetic of the stream merge at the end of linear_logp_partial_kernel.
__global__ __launch_bounds__(256) void linear_logp_stream_merge_kernel(const float* __restrict__ spart,
                                                                      float* __restrict__ part, int T, int n_split) {
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= T * n_split) return;
  const int m = idx % T;
  const int split = idx / T;
  const int64_t splane = (int64_t)n_split * kLogpStreams * T;
  const float* xm = spart + (int64_t)split * kLogpStreams * T + m;
  float big, sum, zt;
  logp_merge_streams(xm, xm + splane, xm + 2 * splane, T, big, sum, zt);
  const int64_t plane = (int64_t)n_split * T;
  const int64_t at = (int64_t)split * T + m;
  part[at] = big;
  part[plane + at] = sum;
  part[2 * plane + at] = zt;
}

// Final merge over splits. 16 tokens per workgroup, 64 threads per token: the maximum and
// the rescaled terms s_p * e(m_p - M) are computed by all threads (neither depends on an
// order), then one thread per token adds the terms of a chunk in ascending split order,
// chunk after chunk. The target logit has a single non-zero contribution, so its sum is
// exact in any order. The kernel waits for one round of loads after the other, so the threads per token set its time
// (16 -> 64, V = 151936: 8.8 -> 5.9 us at 16 tokens, 10.8 -> 7.1 at 256, 13.8 -> 8.7 at 4000).
constexpr int kMergeTokens = 16;
constexpr int kMergeLanes = 64;                           // threads per token
constexpr int kMergeChunk = 2 * kMergeLanes;              // splits staged per round
constexpr int kMergeThreads = kMergeTokens * kMergeLanes;  // 1024

__global__ __launch_bounds__(kMergeThreads) void linear_logp_merge_kernel(const float* __restrict__ part,
                                                                          float* __restrict__ logp,
                                                                          float* __restrict__ lse,
                                                                          float* __restrict__ target_logit, int T,
                                                                          int n_split, bool clamp,
                                                                          const int64_t* __restrict__ target,
                                                                          int64_t target_lo, int64_t target_hi,
                                                                          const float* __restrict__ temperature) {
  __shared__ float red[kMergeLanes][kMergeTokens];
  __shared__ float terms[kMergeChunk][kMergeTokens];
  const int tk = threadIdx.x % kMergeTokens;
  const int sp = threadIdx.x / kMergeTokens;
  const int m = blockIdx.x * kMergeTokens + tk;
  const bool live = m < T;
  const int64_t plane = (int64_t)n_split * T;

  float big = kNegInf, zt = 0.f;
  if (live) {
    for (int p = sp; p < n_split; p += kMergeLanes) {
      big = fmaxf(big, part[(int64_t)p * T + m]);
      zt = zt + part[2 * plane + (int64_t)p * T + m];
    }
  }
  red[sp][tk] = big;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kMergeLanes; ++j) big = fmaxf(big, red[j][tk]);
  __syncthreads();
  red[sp][tk] = zt;
  __syncthreads();
  if (sp == 0) {
    zt = 0.f;
#pragma unroll
    for (int j = 0; j < kMergeLanes; ++j) zt = zt + red[j][tk];
  }

  float sum = 0.f;
  for (int c0 = 0; c0 < n_split; c0 += kMergeChunk) {
#pragma unroll
    for (int i = 0; i < kMergeChunk / kMergeLanes; ++i) {
      const int local = i * kMergeLanes + sp;
      const int p = c0 + local;
      float term = 0.f;
      if (live && p < n_split) {
        const float pm = part[(int64_t)p * T + m];
        const float scaled = part[plane + (int64_t)p * T + m] * pinned_exp(pm - big);
        term = (pm > kNegInf) ? scaled : 0.f;
      }
      terms[local][tk] = term;
    }
    __syncthreads();
    if (sp == 0) {
      const int count = (n_split - c0) < kMergeChunk ? (n_split - c0) : kMergeChunk;
      for (int j = 0; j < count; ++j) sum = sum + terms[j][tk];
    }
    __syncthreads();
  }
  if (sp == 0 && live) {
    float l = big + logf(sum);
    // A temperature that is not a positive number scales nothing meaningful: both results of the row are NaN.
    const bool bad_temperature = temperature != nullptr && !(temperature[m] > 0.f);
    // A target id outside [target_lo, target_hi) names no column this call reduces over: the row's log-prob is
    // NaN instead of a number made of a zero target logit (lse is that of the row all the same).
    const bool bad_target = target != nullptr && (target[m] < target_lo || target[m] >= target_hi);
    if (bad_temperature) l = __builtin_nanf("");
    if (lse) lse[m] = l;
    if (logp) {
      float value = clamp ? fminf(zt - l, 0.f) : zt - l;
      if (bad_temperature || bad_target) value = __builtin_nanf("");  // fminf would drop a NaN operand
      logp[m] = value;
    }
    if (target_logit) target_logit[m] = zt;
  }
}

hipError_t linear_logp_merge_launch(const float* part, float* logp, float* lse, float* target_logit, int T,
                                    int n_split, bool clamp, hipStream_t stream, const int64_t* target,
                                    int64_t target_lo, int64_t target_hi, const float* temperature) {
  hipLaunchKernelGGL(linear_logp_merge_kernel, dim3((T + kMergeTokens - 1) / kMergeTokens), dim3(kMergeThreads), 0,
                     stream, part, logp, lse, target_logit, T, n_split, clamp, target, target_lo, target_hi,
                     temperature);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

using LogpShape256 = TileShape<256, 256, 4, 2>;
using LogpShape192 = TileShape<256, 192, 4, 2>;
using LogpShape128 = TileShape<256, 128, 4, 2>;
using LogpShape64 = TileShape<256, 64, 4, 2>;
using LogpShape16 = TileShape<256, 16, 4, 1>;

int linear_logp_split_count(int V) { return (V + kLogpSplitCols - 1) / kLogpSplitCols; }

constexpr int kStreamGroupMaxTokens = 1024;  // token counts the stream-group kernels serve

size_t linear_logp_workspace_bytes(int T, int V) {
  if (T <= 0) return 0;
  // per-split partials, plus per-(split, stream) states where the stream-group kernel may run
  const size_t per_split = (size_t)3 * linear_logp_split_count(V) * (size_t)T * sizeof(float);
  return T <= kStreamGroupMaxTokens ? per_split * (1 + kLogpStreams) : per_split;
}

// Groups of eight token tiles share the weight's panels in an XCD's L2. One to three tiles behind one or two whole groups would
// read the whole weight again and are spread over the groups instead (256-token tiles, the only ones that come in such
// numbers by the automatic choice). Groups of eight / spread, us, a last tile of 40 / of 250 tokens: V = 131072, D = 2048 with 9
// tiles 1062 / 1006, 1055 / 1032, 11: 1237 / 1195, 1227 / 1244, 17: 1866 / 1823, 1889 / 1867, 19: 2092 / 2074, 2103 / 2077; V =
// 151936, D = 4096 with 9: 2261 / 2087, 2241 / 2226, 11: 2671 / 2547, 2638 / 2640, 18: 4229 / 4149, 4244 / 4184, 19: 4603 / 4617,
// 4549 / 4560. Behind three groups it is no gain: 25 tiles 2730 / 2716, 5925 / 5963, 26: 2763 / 2748, 6309 / 6325, 27: 2938 / 2980,
// 6306 / 6384; nor with four to seven tiles (21 as three groups of seven: 2197 / 2258).
template <class S>
static int token_tiles_per_group(int tiles) {
  if (tiles < 8) return tiles;
  const int groups = tiles / 8, rest = tiles % 8;
  const bool spread = S::BM == 256 && groups <= 2 && rest >= 1 && rest <= 3;
  return spread ? (tiles + groups - 1) / groups : 8;
}

template <class S, int LOOP, class ST = S>
static hipError_t launch_logp(LogpArgs a, hipStream_t stream) {
  auto kernel = linear_logp_partial_kernel<S, ST, LOOP>;
  constexpr int kMergeBytes = 3 * kLogpStreams * S::BM * (int)sizeof(float);
  constexpr int kLds = S::kLdsBytes > kMergeBytes ? S::kLdsBytes : kMergeBytes;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  a.tiles_m = (a.T + S::BM - 1) / S::BM;
  a.group_m = token_tiles_per_group<S>(a.tiles_m);
  hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.n_split), dim3(S::kThreads), kLds, stream, a);
  return hipGetLastError();
}

// A last token tile with few tokens is read beside the others (its workgroups share their weight panels) or behind them, in units of
// their own: behind eight or more whole tiles, whose groups of eight it would widen (beside / behind, us, D = 4096, V = 151936: 2100
// tokens 2044 / 1971, 3100 with logits 3390 / 3240, 5130 4832 / 4632, 8200 7497 / 7052; V = 32768, D = 2048, 4110 with logits 690 /
// 626), behind fewer where the last round of workgroups has little room for units of the whole size (1290 tokens, 745 units: 1380 /
// 1343, but 1030, 596 units, with logits 1224 / 1266; 1850, 1043 units, with logits 1983 / 2080).
static bool logp_rest_behind(int whole_tiles, int n_split, int cus) {
  return whole_tiles >= 8 || whole_tiles * n_split % cus * 4 >= 3 * cus;
}

template <class ST>
static hipError_t launch_logp_solo(LogpArgs a, hipStream_t stream) {
  auto kernel = a.logits != nullptr ? linear_logp_solo_kernel<true, ST> : linear_logp_solo_kernel<false, ST>;
  static PerDeviceOnce once[2];
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kSoloLdsBytes, once[a.logits != nullptr]);
  if (err != hipSuccess) return err;
  const int whole = a.T / SoloShape::BM;
  const bool behind = ST::BM > 0 && logp_rest_behind(whole, a.n_split, device_cu_count());
  a.tiles_m = behind ? whole : (a.T + SoloShape::BM - 1) / SoloShape::BM;
  a.group_m = token_tiles_per_group<LogpShape256>(a.tiles_m);
  hipLaunchKernelGGL(kernel, dim3((a.tiles_m + (behind ? 1 : 0)) * a.n_split), dim3(SoloShape::kThreads), kSoloLdsBytes, stream, a);
  return hipGetLastError();
}

// Where one wave per SIMD is the faster loop: as for the GEMM (ping-pong / one wave, us: V = 18992 at 2000 tokens, 152 units of four
// tiles, 282 / 293, at 8192, 608 units, 991 / 992; V = 37984 at 1700 tokens, 266 units, 629 / 639, at 2560, 380 units, 674 / 653), and
// with stored logits from a round on (V = 18992 at 4000 tokens, 304 units, 733 / 700).
static bool logp_solo_pays(const LogpArgs& a) {
  const bool spans = a.logits == nullptr || ((a.logits_ld & 3) == 0 && (reinterpret_cast<uintptr_t>(a.logits) & 15) == 0);
  if (!spans || a.bias != nullptr || !solo_offsets_fit(a.W) || !solo_offsets_fit(a.H)) return false;
  const int cus = device_cu_count();
  const int whole = a.T / SoloShape::BM, rest = a.T % SoloShape::BM;
  // Units of a last tile of up to 128 tokens that come behind the others. Eight waves are ahead, four / eight in us,
  //   where they open a round behind one or two of few token tiles: V = 32768, D = 2880 at 2158 tokens (256 + 32 units) 500 / 423; V = 24576,
  //   D = 1024 at 2635 (240 + 24) 209 / 182; V = 49152, D = 2048 at 2646 (480 + 48) 549 / 492; V = 37984, D = 1024 at 1658 (228 + 38) 208 / 190, but
  //   with stored logits, where the rounds before are not nearly full, 261 / 274 at 1624; from 12 token tiles on V = 37984, D = 2048 at 3436
  //   652 / 680, V = 24576, D = 4096 at 5478 1112 / 1167;
  //   with stored logits just above one round: V = 32768, D = 2048 at 2311 (288 + 32) 445 / 415; V = 37984, D = 4096 at 1820 (266 + 38) 730 / 733;
  //   but V = 50257, D = 4096 at 1564 (300 + 50) 752 / 771, V = 37984, D = 2880 at 2108 (304 + 38) 563 / 574.
  if (rest >= 1 && rest <= 128 && logp_rest_behind(whole, a.n_split, cus)) {
    const int64_t ahead = (int64_t)whole * a.n_split, all = ahead + a.n_split;
    const bool opens = ahead <= 2 * cus && (all - 1) / cus > (ahead - 1) / cus;
    if (rest > 64 && whole < 12 && opens && (a.logits == nullptr || ((ahead - 1) % cus + 1) * 16 >= 15 * cus)) return false;
    if (a.logits != nullptr && ahead > cus && 8 * ahead <= 9 * cus) return false;
  }
  const int64_t units = (int64_t)((a.T + 127) / SoloShape::BM) * a.n_split;
  if (units < cus) return 10 * units >= 7 * cus;  // (160 units, V = 32768, D = 2048 at 1356 tokens with logits, 206 / 213; 190, V = 37984 at 1193, 346 / 333)
  return solo_tiles_pay(units, cus) || a.logits != nullptr;
}

// 256-token tiles; a last one with few tokens runs as a tile of its size. With the groups above, us: V = 151936, D = 4096 at
// 2100 tokens 2179 -> 2051 (with stored logits 2491 -> 2343), 4120: 3812 -> 3775 (4381 -> 4319); V = 131072, D = 2048 at 1030
// tokens 597 -> 529, 2100: 1046 -> 988; V = 18992, D = 4096 at 1100 tokens 302 -> 271.
static hipError_t launch_logp_256(const LogpArgs& a, hipStream_t stream) {
  const int rest = a.T % LogpShape256::BM;
  if (logp_solo_pays(a)) {
    if (rest >= 1 && rest <= 64) return launch_logp_solo<TileShape<256, 64, 2, 2>>(a, stream);
    if (rest >= 1 && rest <= 128) return launch_logp_solo<TileShape<256, 128, 2, 2>>(a, stream);
    return launch_logp_solo<LogpNoRest>(a, stream);
  }
  if (rest >= 1 && rest <= LogpShape64::BM) return launch_logp<LogpShape256, 2, LogpShape64>(a, stream);
  if (rest >= 1 && rest <= LogpShape128::BM) return launch_logp<LogpShape256, 2, LogpShape128>(a, stream);
  return launch_logp<LogpShape256, 2>(a, stream);
}

// Up to 128 tokens every weight tile is used by one workgroup only: three stages for the
// 64- and 128-token tiles (120 / 144 KiB); the 256-token tile has room for two.
template <class S, bool WSTREAM = false>
static hipError_t launch_streamgroup_range(LogpArgs a, float* spart, int split_first, int split_count,
                                           hipStream_t stream) {
  if constexpr (S::BM <= 128 && !WSTREAM) {
    if (a.T <= S::BM && streamed_weight(a.V, a.D, a.T, S::BM))
      return launch_streamgroup_range<S, true>(a, spart, split_first, split_count, stream);
  }
  constexpr int kStages = S::BM <= 128 ? 3 : 2;
  auto kernel = linear_logp_streamgroup_kernel<S, kStages, WSTREAM>;
  constexpr int kLdsBytes = kStages * S::kStageBytes;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLdsBytes, once);
  if (err != hipSuccess) return err;
  a.tiles_m = (a.T + S::BM - 1) / S::BM;
  hipLaunchKernelGGL(kernel, dim3(a.tiles_m * split_count * (kLogpStreams / 4)), dim3(S::kThreads), kLdsBytes, stream,
                     a, spart, split_first, split_count);
  return hipGetLastError();
}

// A 256-token launch whose last round would fill at most half of the chip ends in 128-token tiles: the splits those cover.
static int balanced_tail_splits(int T, int n_split, int cus) {
  const int per_split = (T + 255) / 256 * (kLogpStreams / 4);
  if (per_split > cus || cus % per_split != 0) return 0;
  const int tail = n_split % (cus / per_split);
  return tail * per_split * 2 <= cus && n_split > tail ? tail : 0;
}

template <int BM>
static hipError_t launch_streams_solo_tile(LogpArgs a, float* spart, hipStream_t stream) {
  auto kernel = a.logits != nullptr ? linear_logp_streamgroup_solo_kernel<true, BM> : linear_logp_streamgroup_solo_kernel<false, BM>;
  static PerDeviceOnce once[2];
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), LogpStreamsSolo<BM>::kLds, once[a.logits != nullptr]);
  if (err != hipSuccess) return err;
  a.tiles_m = (a.T + BM - 1) / BM;
  const int64_t tiles = (int64_t)a.tiles_m * a.n_split * (kLogpStreams / 4);
  const int cus = device_cu_count();
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles < cus ? tiles : cus)), dim3(SoloShape::kThreads), LogpStreamsSolo<BM>::kLds, stream, a,
                     spart);
  return hipGetLastError();
}

static hipError_t launch_stream_merge(const LogpArgs& a, const float* spart, hipStream_t stream) {
  const int threads = a.T * a.n_split;
  hipLaunchKernelGGL(linear_logp_stream_merge_kernel, dim3((threads + 255) / 256), dim3(256), 0, stream, spart, a.part, a.T, a.n_split);
  return hipGetLastError();
}

// `balance`: with the 256-token tile, a last round that would fill at most half of the chip
// runs as 128-token tiles instead (twice the workgroups, each about 0.57 of the time): for
// 256 tokens and V = 151936, 596 workgroups are 2.33 rounds of 256; 512 of them plus 168
// half-height ones are two rounds and a short one (350 -> 290 us). Same bits: the tile height
// is not part of the contract.
template <class S>
static hipError_t launch_streamgroup(LogpArgs a, bool balance, hipStream_t stream) {
  float* spart = a.part + (size_t)3 * a.n_split * a.T;  // behind the per-split partials
  int main_splits = a.n_split;
  if (balance && S::BM == 256) main_splits -= balanced_tail_splits(a.T, a.n_split, device_cu_count());
  hipError_t err = launch_streamgroup_range<S>(a, spart, 0, main_splits, stream);
  if (err != hipSuccess) return err;
  if (main_splits < a.n_split) {
    err = launch_streamgroup_range<LogpShape128>(a, spart, main_splits, a.n_split - main_splits, stream);
    if (err != hipSuccess) return err;
  }
  return launch_stream_merge(a, spart, stream);
}

// Whether the one-wave-per-SIMD form takes the operands.
static bool streams_solo_fits(const LogpArgs& a) {
  const bool spans = a.logits == nullptr || ((a.logits_ld & 3) == 0 && (reinterpret_cast<uintptr_t>(a.logits) & 15) == 0);
  return spans && a.bias == nullptr && solo_offsets_fit(a.W, 3 * kLogpTileCols + 64) && solo_offsets_fit(a.H);
}
static hipError_t launch_streams_solo(const LogpArgs& a, int bm, hipStream_t stream) {
  float* spart = a.part + (size_t)3 * a.n_split * a.T;
  const hipError_t err = bm == 256   ? launch_streams_solo_tile<256>(a, spart, stream)
                         : bm == 192 ? launch_streams_solo_tile<192>(a, spart, stream)
                                     : launch_streams_solo_tile<128>(a, spart, stream);
  return err == hipSuccess ? launch_stream_merge(a, spart, stream) : err;
}

// What the eight-wave stream groups take: rounds of workgroups x tokens per tile / relative throughput, of the tile for T tokens.
static double streams_cost(int T, int n_split, int bm, double quality, double partial_floor = 0.9) {
  return rounds_of_workgroups((int64_t)((T + bm - 1) / bm) * n_split * (kLogpStreams / 4), device_cu_count(), partial_floor) * bm / quality;
}
struct StreamsChoice {
  int config;
  double cost;
};
static StreamsChoice best_streams(int T, int n_split) {
  // 128 / 256 / 192 tokens, us: V = 151936, D = 4096 at 300 tokens 482 / 523 / 432, 540: 779 / 737 / 608, 700: 914 / 746 / 811; V = 37984
  // at 300: 137 / 199 / 161, 450: 193 / 203 / 166, 800: 307 / 303 / 256; V = 32768, D = 2048 at 300: 84 / 74 / 62, 700: 122 / 128 / 109.
  const int tail = balanced_tail_splits(T, n_split, device_cu_count());
  const double c256 = tail ? streams_cost(T, n_split - tail, 256, 1.0) + streams_cost(T, tail, 128, 0.76) : streams_cost(T, n_split, 256, 1.0);
  const double c192 = streams_cost(T, n_split, 192, 0.945), c128 = streams_cost(T, n_split, 128, 0.76);
  if (T <= 128) return {RLK_LOGP_CFG_128_STREAMS, c128};
  if (T <= 256) return {RLK_LOGP_CFG_256_STREAMS, c256};
  if (c192 < c256 && c192 < c128) return {RLK_LOGP_CFG_192_STREAMS, c192};
  return c128 < c256 ? StreamsChoice{RLK_LOGP_CFG_128_STREAMS, c128} : StreamsChoice{RLK_LOGP_CFG_256_STREAMS, c256};
}

// The tokens of a tile of the one-wave-per-SIMD form, 0 for the eight-wave one. 256 tokens with stored logits do not fit its registers. Costs
// fitted to 64 shapes of six heads and 100 to 1024 tokens, on the eight-wave form's scale. It runs where it has the same tile in no more
// rounds (0.63 and 0.82 of the cost, 2 to 8 % of the time) or a better one; what lies above is faster on one machine and slower on
// another (no logits, 203 tokens, V = 151936, D = 4096: 344 / 336 and 325 / 341; 226, 37984, 4096: 109 / 101 and 109 / 116; logits, 484, 151936, 4096
// 589 / 621). Eight waves -> this, us (tokens, V, D): 168, 18992, 4096 85 -> 52; 237, 32768, 2048 59 -> 42; 121, 50257, 2048 55 -> 46; 266, 37984, 4096
// 138 -> 122; 595, 131072, 2048 394 -> 348; 891, 151936, 4096 1013 -> 964; with stored logits 127, 32768, 2048 54 -> 42; 548, 151936, 4096 678 -> 640;
// 753, 131072, 2048 502 -> 451; it stays with eight at 698, 37984, 4096 (230 / 248) and 995, 32768, 2048 (154 / 160).
static int pick_streams_solo(const LogpArgs& a) {
  // One token tile of 128. A weight that HBM alone sets the pace of is read past the caches (V = 151936, D = 4096 at 76 / 99 tokens 253 / 257,
  // 258 / 260; V = 131072, D = 2048 at 83 tokens 147 / 145). Where most CUs have one tile, its fold and the stores of its logits run
  // behind the loads of nothing else, and four waves lose what they are ahead with weights that come from HBM (eight / four, us):
  //   with stored logits from 100 tiles on until every CU has two: 96, 24576, 4096 (96 tiles) 83.5 / 83.2; 96, 37984, 4096 (152) 96.2 / 102.6; 96,
  //   50257, 4096 (200) 112.4 / 122.1; 120, 80000, 4096 (316) 203.8 / 212.2; 96, 131072, 2048 (512) 172 / 168; 1.08 and 1.04 times at 62000 rows of
  //   181 MiB, 1.00 and 0.98 at 37984 of 185, 0.95 at 31014 of 113;
  //   without them from 144 tiles to a round: 96, 32768, 4096 (128) 90.2 / 89.5; 120, 40960, 4096 (160) 96.6 / 98.5; 120, 60000, 4096 (236) 119.9 /
  //   123.6; 120, 66000, 2048 (260) 117.6 / 114.6; 96, 32000, 8192 146.7 / 148.1; 1.05 times at 50257 rows of 294 MiB, 1.01 of 245, 0.97 of 184.
  // A vocabulary that ends in the first half of a split has two of its four tiles empty, which eight waves leave out: 79, 500, 256 18.2 /
  // 20.3, with logits 18.7 / 23.6; 100, 512, 1024 25.5 / 26.2, 26.3 / 28.6; 289, 500, 576 with logits 22.8 / 26.4, but D = 2048 34.9 / 33.9, 35.4 /
  // 36.3, and at 129 to 256 tokens, for which the eight waves' tile is one of 256 tokens, 165, 500, 576 30.7 / 24.8.
  if (a.V <= 2 * kLogpTileCols && a.D < 2048 && (a.T <= 128 || a.T > 256)) return 0;
  if (a.T <= 128) {
    const int64_t mib = ((int64_t)a.V * a.D) >> 19, tiles = (int64_t)a.n_split * (kLogpStreams / 4);
    const int cus = device_cu_count();
    if (mib >= 1024) return 0;
    if (a.logits != nullptr ? 64 * tiles > 25 * cus && tiles < 2 * cus && mib >= 192
                            : tiles <= cus && mib >= (16 * tiles > 9 * cus ? 224 : 480))
      return 0;
  }
  constexpr double kPartial = 0.965;
  const double eight = best_streams(a.T, a.n_split).cost;
  if (a.logits != nullptr) {
    const double c128 = streams_cost(a.T, a.n_split, 128, 1.012, kPartial), c192 = streams_cost(a.T, a.n_split, 192, 1.157, kPartial);
    const double best = c192 < c128 ? c192 : c128;
    return best > 0.83 * eight ? 0 : c192 < c128 ? 192 : 128;
  }
  const double c128 = streams_cost(a.T, a.n_split, 128, 1.437, kPartial), c192 = streams_cost(a.T, a.n_split, 192, 1.574, kPartial);
  const double c256 = streams_cost(a.T, a.n_split, 256, 1.585, kPartial);
  const int tokens = c256 <= c192 && c256 <= c128 ? 256 : c192 < c128 ? 192 : 128;
  const double best = tokens == 256 ? c256 : tokens == 192 ? c192 : c128;
  return best > 0.64 * eight ? 0 : tokens;
}

int pick_linear_logp_config(int T, int V) {
  // Measured at V = 151936, D = 4096: the 64-token tile (two workgroups per CU, direct-to-LDS
  // loop) is the fastest from decode sizes up to 64 tokens, the 256-token tile from 1024 tokens on
  // even where it leaves the last round of workgroups part empty.
  if (T <= 64) return RLK_LOGP_CFG_64_STREAMS;
  if (T > kStreamGroupMaxTokens) return RLK_LOGP_CFG_256;
  return best_streams(T, linear_logp_split_count(V)).config;
}

hipError_t linear_logp_launch(const MatView& H, const MatView& W, const int64_t* target, const float* bias,
                              const float* temperature, float* logp, float* lse, float* target_logit,
                              float* logits, int64_t logits_ld, float* workspace, int T, int D, int V,
                              int64_t vocab_start, int vocab_limit, int config, hipStream_t stream) {
  LogpArgs a;
  a.logits = logits;
  a.logits_ld = logits_ld;
  a.W = W;
  a.H = H;
  a.target = target;
  a.bias = bias;
  a.temperature = temperature;
  a.part = workspace;
  a.T = T;
  a.V = V;
  a.D = D;
  a.vocab_limit = vocab_limit;
  a.vocab_start = vocab_start;
  a.n_split = linear_logp_split_count(V);
  a.tiles_m = 0;
  a.group_m = 1;
  const bool vec = W.k_stride == 1 && H.k_stride == 1 && (W.row_stride % kChunkElems) == 0 &&
                   (H.row_stride % kChunkElems) == 0 && (reinterpret_cast<uintptr_t>(W.ptr) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(H.ptr) & 15) == 0 && (D % kChunkElems) == 0 &&
                   pitch_fits_lane_offsets(W.row_stride) && pitch_fits_lane_offsets(H.row_stride);
  const bool force_staged = (config & RLK_LOGP_CFG_FORCE_STAGED) != 0;
  config &= ~RLK_LOGP_CFG_FORCE_STAGED;
  const int requested = config;
  if (config == RLK_LOGP_CFG_AUTO) config = pick_linear_logp_config(T, V);
  const int loop = !vec ? 0 : (D % kTileK == 0 && !force_staged) ? 2 : 1;
  // The stream-group kernels have the direct-to-LDS loop only and a bounded workspace.
  if (loop != 2 || T > kStreamGroupMaxTokens) {
    if (config == RLK_LOGP_CFG_64_STREAMS) config = RLK_LOGP_CFG_64;
    if (config == RLK_LOGP_CFG_128_STREAMS) config = RLK_LOGP_CFG_128;
    if (config == RLK_LOGP_CFG_192_STREAMS || config == RLK_LOGP_CFG_256_STREAMS) config = RLK_LOGP_CFG_256;
  }
  if (!vec && config == RLK_LOGP_CFG_256) config = RLK_LOGP_CFG_128;  // which has the element-wise loader
  hipError_t err;
  const bool streams = config == RLK_LOGP_CFG_128_STREAMS || config == RLK_LOGP_CFG_192_STREAMS || config == RLK_LOGP_CFG_256_STREAMS;
  const int solo_tokens = requested == RLK_LOGP_CFG_AUTO && streams && streams_solo_fits(a) ? pick_streams_solo(a) : 0;
  if (solo_tokens != 0) {
    err = launch_streams_solo(a, solo_tokens, stream);
  } else switch (config) {
    case RLK_LOGP_CFG_64_STREAMS:
      err = launch_streamgroup<LogpShape64>(a, false, stream);
      break;
    case RLK_LOGP_CFG_128_STREAMS:
      err = launch_streamgroup<LogpShape128>(a, false, stream);
      break;
    case RLK_LOGP_CFG_192_STREAMS:
      err = launch_streamgroup<LogpShape192>(a, false, stream);
      break;
    case RLK_LOGP_CFG_256_STREAMS:
      err = launch_streamgroup<LogpShape256>(a, requested == RLK_LOGP_CFG_AUTO, stream);
      break;
    case RLK_LOGP_CFG_256:
      err = loop == 2 ? launch_logp_256(a, stream) : launch_logp<LogpShape256, 1>(a, stream);
      break;
    case RLK_LOGP_CFG_128:
      err = loop == 2   ? launch_logp<LogpShape128, 2>(a, stream)
            : loop == 1 ? launch_logp<LogpShape128, 1>(a, stream)
                        : launch_logp<LogpShape128, 0>(a, stream);
      break;
    case RLK_LOGP_CFG_64:
      err = loop == 2   ? launch_logp<LogpShape64, 2>(a, stream)
            : loop == 1 ? launch_logp<LogpShape64, 1>(a, stream)
                        : launch_logp<LogpShape64, 0>(a, stream);
      break;
    case RLK_LOGP_CFG_16:
      err = loop >= 1 ? launch_logp<LogpShape16, 1>(a, stream) : launch_logp<LogpShape16, 0>(a, stream);
      break;
    default:
      return hipErrorInvalidValue;
  }
  if (err != hipSuccess) return err;
  // The whole-vocabulary entries (those that write logp) mark rows whose target lies outside the real vocabulary;
  // a shard's target logit is legitimately 0 for a target another shard owns.
  return linear_logp_merge_launch(workspace, logp, lse, target_logit, T, a.n_split, true, stream,
                                  logp != nullptr ? target : nullptr, vocab_start, vocab_start + vocab_limit,
                                  temperature);
}

}  // namespace rlk
