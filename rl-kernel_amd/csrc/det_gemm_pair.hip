// The two products of a linear layer's backward in one launch:
//   dX[M, K_in]     = dY[M, N_out] W[N_out, K_in]      (weight read K-major)
//   dW[N_out, K_in] = dY^T X                           (both operands read K-major)
// Neither waits for the other, and each has its own number of tiles, so launched one after the other each pays for a last
// round of workgroups that leaves compute units idle. In one launch the workgroups of the second product take the compute
// units that the first has no tile for. The tiles, loops and so the bits are those of det_gemm.hip: workgroups of a tile each, or, where
// there is enough for 256 x 256 tiles, one workgroup per CU that goes through a share of both products.
#include "det_gemm_solo_body.h"
#include "rlk_host.h"

namespace rlk {

struct PairProblem {
  MatView W, X;
  void* C;
  int64_t ldc;
  int M, N, K;
  int tiles_m, tiles_n, group_m;
};

// Workgroups [0, first_blocks) own the tiles of the product that starts first, the others those of the second.
// first_blocks is a whole multiple of the XCD count, so that both products keep their XCD-compact tile order; the
// workgroups behind the first product's last tile have nothing to do.
// (dX in small tiles keeps the stages of launch_small_kmajor, without its prefetching wave: a ninth wave has no registers
// beside eight of the dW tile's.)
template <class SX, int KSX, int NSX, class SW>
__global__ __launch_bounds__(SX::kThreads) void det_gemm_pair_kernel(PairProblem dx, PairProblem dw, int first_blocks,
                                                                     bool dx_first) {
  static_assert(SX::kThreads == SW::kThreads, "one workgroup size");
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const bool second = (int)blockIdx.x >= first_blocks;
  const int block = second ? (int)blockIdx.x - first_blocks : (int)blockIdx.x;
  if (second != dx_first) {
    if (block < dx.tiles_m * dx.tiles_n)
      det_gemm_tile<SX, kLoopPingPongKMajor, false, KSX, NSX, false>(dx.W, dx.X, dx.C, dx.ldc, dx.M, dx.N, dx.K,
                                                                     dx.tiles_m, dx.tiles_n, dx.group_m, block, lds);
  } else {
    if (block < dw.tiles_m * dw.tiles_n)
      det_gemm_tile<SW, kLoopPingPongBothKMajor, false, 1, 2, false>(dw.W, dw.X, dw.C, dw.ldc, dw.M, dw.N, dw.K,
                                                                     dw.tiles_m, dw.tiles_n, dw.group_m, block, lds);
  }
}

// The same with one wave per SIMD (det_gemm_solo.h), 256 x BM tiles of dX and 256 x 256 of dW, one workgroup per CU with a share of both
// products fixed by the host: the tiles of `first` in turn, then those of the other product, of which workgroups [0, late), which have one tile of the
// first more, take late_tiles each and the others the rest.
struct SoloShares {
  bool dx_first;
  int late, late_tiles;
};
struct SoloPair {
  SoloProblem dx, dw;
  SoloShares shares;
};
// Read from the arguments when its turn comes: as values of the kernel, the two products are in scalar registers at once, and spill a
// hundred.
__device__ __forceinline__ SoloProblem solo_argument(bool is_dx) {
  const __attribute__((address_space(4))) SoloPair* args =
      (const __attribute__((address_space(4))) SoloPair*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  SoloProblem p;
  __builtin_memcpy(&p, is_dx ? &args->dx : &args->dw, sizeof(p));
  return p;
}
template <int BM>
using SoloDx = SoloLayout<true, false, TileShape<256, BM, 2, 2>>;
using SoloDw = SoloLayout<true, true>;
template <int BM>
__global__ __launch_bounds__(SoloShape::kThreads) void det_gemm_pair_solo_kernel(SoloPair pair) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const SoloShares shares = pair.shares;
  const int group = blockIdx.x, groups = gridDim.x;
  for (int product = 0; product < 2; ++product) {
    const bool is_dx = (product == 0) == shares.dx_first;
    const SoloProblem p = solo_argument(is_dx);
    const int tiles = p.tiles_m * p.tiles_n;
    int at = group, step = groups, total = tiles;
    if (product == 1) {
      const int of_late = min(shares.late * shares.late_tiles, tiles);
      const bool late = group < shares.late;
      at = late ? group : of_late + group - shares.late;
      step = late ? shares.late : groups - shares.late;
      total = late ? of_late : tiles;
    }
    if (at >= total) continue;
    if (is_dx) solo_product<SoloDx<BM>>(p, at, step, total, lds);
    else solo_product<SoloDw>(p, at, step, total, lds);
    wg_barrier();  // the next product's loads overwrite what the last reads are of
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

using Pair256x256 = TileShape<256, 256, 4, 2>;
using Pair256x192 = TileShape<256, 192, 4, 2>;
using Pair256x128 = TileShape<256, 128, 4, 2>;
using Pair128x128 = TileShape<128, 128, 4, 2>;
using Pair64x64 = TileShape<64, 64, 4, 2>;

// The tiles of a configuration, features x tokens for dX, inputs x outputs for dW, and their relative throughput on a full
// chip (the K-major column of kTileCandidates; 128 x 128 falls behind it beside the dW tiles, 0.62 -> 0.53).
struct PairTiles {
  int dx_bn, dx_bm;
  double dx_quality;
  int dw_bn, dw_bm;
  double dw_quality;
};
static const PairTiles kPairTiles[RLK_LINEAR_BWD_CFG_COUNT] = {
    {}, {},  // automatic, two launches
    {256, 256, 1.00, 256, 256, 1.00}, {256, 128, 0.70, 256, 256, 1.00}, {256, 256, 1.00, 256, 128, 0.70},
    {256, 128, 0.70, 256, 128, 0.70}, {128, 128, 0.53, 256, 256, 1.00}, {64, 64, 0.25, 256, 256, 1.00},
    {256, 192, 0.90, 256, 256, 1.00},
};

template <class S>
static PairProblem pair_problem(const GemmProblem& p) {
  PairProblem r{p.W, p.X, p.C, p.ldc, p.M, p.N, p.K, (p.M + S::BM - 1) / S::BM, (p.N + S::BN - 1) / S::BN, 1};
  r.group_m = r.tiles_m < 8 ? r.tiles_m : 8;
  return r;
}

template <class SX, int KSX, int NSX, class SW>
static hipError_t launch_pair(const GemmProblem& dx, const GemmProblem& dw, bool dx_first, hipStream_t stream) {
  auto kernel = det_gemm_pair_kernel<SX, KSX, NSX, SW>;
  constexpr int kLdsX = KSX * NSX * SX::kStageBytes, kLdsW = 2 * SW::kStageBytes;
  constexpr int kLds = kLdsX > kLdsW ? kLdsX : kLdsW;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  const PairProblem a = pair_problem<SX>(dx), b = pair_problem<SW>(dw);
  const int tiles_dx = a.tiles_m * a.tiles_n, tiles_dw = b.tiles_m * b.tiles_n;
  const int first = ((dx_first ? tiles_dx : tiles_dw) + kXcds - 1) / kXcds * kXcds;
  const int second = dx_first ? tiles_dw : tiles_dx;
  hipLaunchKernelGGL(kernel, dim3(first + second), dim3(SX::kThreads), kLds, stream, a, b, first, dx_first);
  return hipGetLastError();
}

static int64_t tile_count(const GemmProblem& p, int bn, int bm) { return (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn); }

// The length of a tile in K tiles of 256 x 256: beside its K tiles each has a cost, and a K tile of fewer tokens takes its part of the
// time. (What it takes of the power, solo_pair_us(), is another part.)
constexpr double kSoloTileCost = 7.0;
static double solo_tile_length(const GemmProblem& p, int bm = 256) {
  return (((int64_t)p.K + kTileK - 1) / kTileK + kSoloTileCost) * (bm == 256 ? 1.0 : bm == 192 ? 0.83 : 0.55);
}

// The shares of the one-wave-per-SIMD launch, and what the workgroup with the most to do has. The product with the longer tiles comes
// first; `late` workgroups have one of its tiles more than the others, and late_tiles is what evens that out.
static SoloShares solo_shares(const GemmProblem& dx, const GemmProblem& dw, int bm, int groups, double* longest) {
  const double length_dx = solo_tile_length(dx, bm), length_dw = solo_tile_length(dw);
  const int64_t tiles_dx = tile_count(dx, 256, bm), tiles_dw = tile_count(dw, 256, 256);
  SoloShares s{length_dx >= length_dw, 0, 0};
  const int64_t na = s.dx_first ? tiles_dx : tiles_dw, nb = s.dx_first ? tiles_dw : tiles_dx;
  const double la = s.dx_first ? length_dx : length_dw, lb = s.dx_first ? length_dw : length_dx;
  const int64_t rounds = na / groups, late = na % groups;
  s.late = (int)late;
  *longest = 1e300;
  const double even = ((na * la + nb * lb) / groups - (rounds + 1) * la) / lb;  // late_tiles, if all had the same
  const int64_t least = even > 0.0 ? (int64_t)even : 0;
  for (int64_t t = least; t <= (even > 0.0 ? least + 1 : least); ++t) {
    const int64_t of_late = late * t < nb ? late * t : nb;
    const int64_t others = (nb - of_late + groups - late - 1) / (groups - late);
    double span = rounds * la + others * lb;
    if (late > 0 && (rounds + 1) * la + t * lb > span) span = (rounds + 1) * la + t * lb;
    if (span < *longest) {
      *longest = span;
      s.late_tiles = (int)t;
    }
  }
  return s;
}
static int solo_groups(const GemmProblem& dx, const GemmProblem& dw, int bm) {
  const int64_t tiles = tile_count(dx, 256, bm) + tile_count(dw, 256, 256);
  const int cus = device_cu_count();
  return (int)(tiles < cus ? tiles : cus);
}
// What that launch takes: the longest share at a rate, and all the work at a rate that the package's power gives, fitted to the three
// tiles of dX on 94 shapes of 500 to 8000 tokens (4.4 %; the cheapest of the three is 0.2 % above the best). On the scale of pair_us(),
// whose figures are 7 % below what a chip at its power cap takes. Where the rule takes it, best other configuration -> this, us
// (tokens, inputs, outputs, tokens per tile of dX):
//   2047, 4096, 4096, 256: 112.2 -> 102.7    601, 14336, 4096, 256: 166 -> 139     2910, 4096, 12288, 256: 465 -> 416   4120, 4096, 151936: 7524 -> 7230
//   1508, 4096, 4096, 192: 87.9 -> 81.1      842, 6144, 2048, 192: 53.5 -> 48.1    2095, 4096, 6144, 192: 175 -> 165    1506, 4096, 24576: 500 -> 475
//   1024, 4096, 4096, 128: 64.0 -> 60.3      1519, 2048, 6144, 128: 80.2 -> 73.0   908, 4096, 24576, 128: 370 -> 349    1030, 4096, 151936: 2590 -> 2373
//   8094, 4096, 14336, 256: 1339 -> 1335     528, 6144, 4096, 128: 69.9 -> 72.7
// where it does not: 8192, 1024, 1024: 98 / 146    603, 3072, 4096: 42.5 / 45.7    663, 2048, 6144: 46.8 / 61.9. Small tiles of dX (few
// tokens: 64 or 128 outputs by as many tokens) are not compared: with a weight from HBM a tile of 128 tokens takes 0.9 us a K tile
// instead of 0.6 (608, 4096, 6144: 80 / 92; 631, 4096, 3072: 42 / 38).
constexpr double kPairScale = 0.935, kPairScaleFew = 1.0;  // few tokens: up to 640 (593, 6144, 4096: 71 / 75; 591, 4096, 4096: 53 / 49)
static double solo_pair_us(const GemmProblem& dx, const GemmProblem& dw, int bm, int cus) {
  double longest;
  solo_shares(dx, dw, bm, solo_groups(dx, dw, bm), &longest);
  const double work_dx = tile_count(dx, 256, bm) * solo_tile_length(dx) * (bm == 256 ? 1.0 : bm == 192 ? 0.70 : 0.73);
  const double work_dw = tile_count(dw, 256, 256) * solo_tile_length(dw);
  // One tile's K tiles, one after the other: what its loads take where few tiles share them. A long reduction against few tiles stays with
  // the smaller ones for it (lm_head backwards, us, this / theirs: 353, 4096, 151936 2550 / 1980; 729, 2048, 50257 813 / 607; 978, 2048,
  // 32768 486 / 431; 298, 4096, 18992 269 / 248).
  const bool cached = (int64_t)dx.N * dx.K * 2 < ((int64_t)40 << 20);
  const double k_tile_us = bm == 256 ? 1.15 : bm == 192 ? 0.97 : cached ? 0.70 : 0.85;
  const double chain_dx = k_tile_us * dx.K / kTileK, chain_dw = 1.15 * dw.K / kTileK;
  const double chain = chain_dx > chain_dw ? chain_dx : chain_dw, us = 0.89 * longest + 0.455 * (work_dx + work_dw) / cus;
  return (dw.K <= 640 ? kPairScaleFew : kPairScale) * (chain > us ? chain : us);
}
static bool solo_pair_serves(const GemmProblem& dx, const GemmProblem& dw) {
  return solo_kmajor_fits(dx.W) && solo_kmajor_fits(dx.X) && solo_kmajor_fits(dw.W) && solo_kmajor_fits(dw.X);
}
template <int BM>
static hipError_t launch_pair_solo(const GemmProblem& dx, const GemmProblem& dw, hipStream_t stream) {
  auto kernel = det_gemm_pair_solo_kernel<BM>;
  constexpr int kLds = SoloDx<BM>::kLds > SoloDw::kLds ? SoloDx<BM>::kLds : SoloDw::kLds;
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  const int groups = solo_groups(dx, dw, BM);
  double longest;
  const SoloPair pair{solo_problem<typename SoloDx<BM>::Shape>(dx.W, dx.X, dx.C, dx.ldc, dx.M, dx.N, dx.K),
                      solo_problem(dw.W, dw.X, dw.C, dw.ldc, dw.M, dw.N, dw.K), solo_shares(dx, dw, BM, groups, &longest)};
  hipLaunchKernelGGL(kernel, dim3(groups), dim3(SoloShape::kThreads), kLds, stream, pair);
  return hipGetLastError();
}

// When the last of the workgroups of two products ends, first product first, each compute unit taking the next tile when it
// is free: n1 tiles of t1, then n2 of t2, on `cus` compute units.
static double pair_span(int64_t n1, double t1, int64_t n2, double t2, int cus) {
  const int64_t full = n1 / cus, late = n1 % cus;  // `late` compute units have one tile of the first product more
  const double base = full * t1;
  int64_t early_rounds = 0, late_rounds = 0, done = 0;
  double span = late ? base + t1 : base;
  while (done < n2) {  // the next round to start is the earlier of the two groups'
    const double early_at = base + early_rounds * t2, late_at = base + t1 + late_rounds * t2;
    const bool early = late == 0 || early_at <= late_at;
    const int64_t group = early ? cus - late : late;
    (early ? early_rounds : late_rounds) += 1;
    done += group;
    const double end = (early ? early_at : late_at) + t2;
    if (end > span) span = end;
  }
  return span;
}

// The estimate of a launch, fitted to 282 shapes (64 to 8192 tokens, 21 layers and vocabularies, every configuration and
// the two launches measured, weights right behind their forward). Over them the choice takes 0.6 % longer than the best
// configuration of each shape, 0.870 of the two launches' time, and is never more than 2 % slower than them; over 72 shapes of
// 12 layers that it was not fitted to 1.4 % longer (at worst 38 %), 0.810, and never more than 2 % slower.
//
// A tile on a full chip, us: 11 + 21 K / 1024 for 256 x 256 outputs (see remainder_launch_pays), other shapes by area and
// quality; a tile of dW, whose reduction is short, starts faster.
constexpr double kStartUs = 11.0, kStartDwUs = 9.0, kLaunchUs = 5.0;  // the last: a second launch
static double tile_us(int bn, int bm, double quality, double start, int K) {
  return (start + 21.0 * K / 1024.0) * bn * bm / 65536.0 / quality;
}
// dX reads its weight from HBM where the memory-side cache cannot still hold it from the forward. Its small tiles miss
// their prefetching wave then (304 tokens, 24576 outputs: 255 us as two launches, 279 as one; 201 tokens, 14336 outputs, 112
// MiB: 126 and 160). Up to 272 tokens from 96 MiB on, which the forward of so few reads past the caches (streamed_weight), and
// where other weights were read in between: 128 x 128 tiles of dX then take longer than 64 x 64 ones, and the two launches'
// dW by the short-reduction kernel is the faster one. Forward and backward, us, two launches / priced as cached / as from HBM:
// 4096 inputs, 12288 outputs at 128 / 193 / 256 tokens 106 / 117 / 106, 139 / 176 / 139, 139 / 174 / 139; a gated FFN of 4096 x
// 12288 at 193 / 256 tokens 438 / 505 / 424, 459 / 519 / 449, of 4096 x 6144 253 / 268 / 247, 262 / 280 / 253. Above, the same
// price chooses the slower form (4096 inputs, 12288 outputs, two launches / one: 257 tokens 179 / 183, 272: 182 / 182, 288: 185 /
// 184, 512: 205 / 193).
static bool weight_from_hbm(const GemmProblem& dx, int tokens, BackwardOf of) {
  const int64_t bytes = (int64_t)dx.N * dx.K * 2;
  if (of != BackwardOf::kLogp && tokens <= 272 && (of == BackwardOf::kManyWeights || bytes >= ((int64_t)96 << 20))) return true;
  return bytes >= ((int64_t)112 << 20);
}
static double dx_tile_us(const PairTiles& t, const GemmProblem& dx, int tokens, BackwardOf of) {
  const bool waits = t.dx_bn < 256 && weight_from_hbm(dx, tokens, of);
  return tile_us(t.dx_bn, t.dx_bm, t.dx_quality, kStartUs, dx.K) * (waits ? 1.2 : 1.0);
}
static double dw_tile_us(const PairTiles& t, const GemmProblem& dw) {
  return tile_us(t.dw_bn, t.dw_bm, t.dw_quality, kStartDwUs, dw.K);
}

// The time of the one launch: the work of all tiles at the full chip's rate, or the span of tiles of which some run with
// much of the chip idle. A tile takes 0.6 of its time alone (256 x 256, K = 4096: 95 -> 65 us, 256 x 128: 68 -> 48.5), the
// whole of it on a full chip and wherever its weight comes at the HBM latency (256 x 256 at K = 37984 / 151936: 790 / 3127
// -> 740 / 2900).
// Up to kFewTokens a weight from HBM keeps the small tiles of dX waiting, and the dW tiles beside them run at 0.7 of their
// time: 37984 outputs, 4096 inputs, 128 x 128 tiles of dX, us at 520 / 688 / 784 / 1024 tokens: 429 / 484 / 548 / 641, by this
// estimate 447 / 486 / 554 / 643, with the whole time 472 / 563 / 645 / 741. (Not beside the rest of a dX whose whole tiles
// ran before: too few tiles of it.) Right behind the LogP forward part of a weight of up to 180 MiB still lies in the
// memory-side cache: 18992 outputs at 400 / 512 tokens 170 / 174 us, by this estimate 208, 227 from HBM.
constexpr int kFewTokens = 1024;
static double pair_us(const GemmProblem& dx, const GemmProblem& dw, const PairTiles& t, int cus, BackwardOf of) {
  const bool from_hbm = weight_from_hbm(dx, dw.K, of);
  const bool waiting = t.dx_bn < 256 && from_hbm && dw.K <= kFewTokens && dx.M == dw.K;
  const bool partly_cached = waiting && of == BackwardOf::kLogp && (int64_t)dx.N * dx.K * 2 < ((int64_t)180 << 20);
  const double tx = dx_tile_us(t, dx, dw.K, of) * (partly_cached ? 0.92 : 1.0), tw = dw_tile_us(t, dw) * (waiting ? 0.7 : 1.0);
  const int64_t nx = tile_count(dx, t.dx_bn, t.dx_bm), nw = tile_count(dw, t.dw_bn, t.dw_bm);
  const double work = (nx * tx + nw * tw) / cus;
  const double span = tx >= tw ? pair_span(nx, tx, nw, tw, cus) : pair_span(nw, tw, nx, tx, cus);
  const double alone = from_hbm ? 1.0 : 0.6;
  const double us = span * (alone + (1.0 - alone) * (work / span));
  return work > us ? work : us;
}

static bool one_launch_serves(const GemmProblem& dx, const GemmProblem& dw) {
  return dx.X.k_stride == 1 && dx.W.k_stride != 1 && dw.X.k_stride != 1 && dw.W.k_stride != 1 &&
         det_gemm_takes_kmajor(dx.W, dx.X, dx.K) && det_gemm_takes_kmajor(dw.W, dw.X, dw.K);
}

static double best_pair_us(const GemmProblem& dx, const GemmProblem& dw, int cus, BackwardOf of, int* config) {
  double best = 1e300;
  for (int c = RLK_LINEAR_BWD_CFG_SEPARATE + 1; c < RLK_LINEAR_BWD_CFG_COUNT; ++c) {
    const double us = pair_us(dx, dw, kPairTiles[c], cus, of);
    if (us < best) {
      best = us;
      *config = c;
    }
  }
  return best;
}

// The rows [0, rows) of dX, and the ones behind them.
static GemmProblem head_of(GemmProblem dx, int rows) {
  dx.M = dx.X.rows = rows;
  return dx;
}
static GemmProblem tail_of(GemmProblem dx, int rows) {
  dx.X.ptr += (int64_t)rows * dx.X.row_stride;
  dx.C = reinterpret_cast<bf16_bits*>(dx.C) + (int64_t)rows * dx.ldc;
  dx.M = dx.X.rows = dx.M - rows;
  return dx;
}

// One launch where the estimate says 2 % less than the two launches' own. Both sides measured, us, 256 CUs, weights and
// activations of three layers in turn (tokens, inputs, outputs: two launches -> one):
//   128, 4096, 4096: 31 -> 22        300, 4096, 4096: 45 -> 35      700, 4096, 4096: 62 -> 56     1400, 4096, 4096: 97 -> 85
//   2047, 4096, 4096: 117 -> 110     300, 4096, 6144: 66 -> 50      1400, 4096, 6144: 157 -> 132  2047, 4096, 6144: 190 -> 163
//   6000, 4096, 6144: 500 -> 445     128, 4096, 1536: 17 -> 12      2047, 4096, 1536: 58 -> 50    200, 12288, 4096: 96 -> 79
//   500, 12288, 4096: 130 -> 113     300, 1024, 4096: 26 -> 18      4120, 1024, 4096: 103 -> 73
// where the rounds are whole it stays with two (4096, 4096, 4096: 205 = 205), and with up to 256 tokens against a large
// weight, whose dW is a stream of stores of its own (det_gemm_shortk_kernel; 128, 4096, 24576: 153 as two, 184 as one; 136:
// 199 as two, 160 as one).
// A token count just above a multiple of 256 (see remainder_launch_pays): the whole tiles of dX first, then the few tokens
// behind them beside dW.
//
// The LogP's own two launches take less than the estimate up to kFewTokens where the weight comes from HBM: dX in 128 x 64
// tiles 0.84 of it (priced at 0.93), dW of whole K tiles, with a native feature operand from 512 tokens on, 0.82 to 0.93.
// Gradients right behind the forward, us, two launches / as chosen before these two, the 0.7 and the 0.92 above / now (tokens,
// inputs, outputs):
//   512, 4096, 37984: 416 / 439 / 416      304, 5120, 32000: 347 / 387 / 347      400, 4096, 18992: 210 / 210 / 170
//   768, 4096, 37984: 530 / 557 / 499      600, 5120, 32000: 497 / 530 / 476      768, 4096, 18992: 266 / 266 / 235
//   768, 5120, 32000: 520 / 546 / 546      800, 4096, 64000: 982 / 932 / 959      520, 4096, 16384: 215 / 172 / 172
// 396 measured forms of 12 layers take 0.920 of the two launches' time (0.935), and are up to 5 % slower than them (13).
constexpr double kFewTokensDx = 0.93, kFewTokensDw = 0.92;
LinearBackwardPlan linear_backward_plan(const GemmProblem& dx, const GemmProblem& dw, BackwardOf of) {
  LinearBackwardPlan plan{RLK_LINEAR_BWD_CFG_SEPARATE, 0};
  if (!one_launch_serves(dx, dw)) return plan;
  const bool from_hbm = weight_from_hbm(dx, dw.K, of);
  if (of != BackwardOf::kManyWeights && from_hbm && det_gemm_shortk_supported(dw.W, dw.X, dw.M, dw.N, dw.K) &&
      det_gemm_shortk_pays(dw.M, dw.N))
    return plan;
  const int cus = device_cu_count();
  const double partial = from_hbm ? 1.0 : 0.9;
  int dx_outputs;
  double us_dx = det_gemm_kmajor_us(dx.M, dx.N, dx.K, true, false, partial, &dx_outputs);
  double us_dw = det_gemm_kmajor_us(dw.M, dw.N, dw.K, true, true, partial);
  if (of == BackwardOf::kLogp && from_hbm && dx.M <= kFewTokens) {
    if (dx_outputs == 128 * 64) us_dx *= kFewTokensDx;
    if (dx.M % kTileK == 0) us_dw *= kFewTokensDw;
  }
  double best = 0.98 * (us_dx + us_dw + kLaunchUs);
  int config;
  const double together = best_pair_us(dx, dw, cus, of, &config);
  if (together < best) {
    best = together;
    plan.config = config;
  }
  const int rest = dx.M % 256;
  if (dx.M > 256 && rest >= 1 && rest <= 64) {
    const int whole = dx.M - rest;
    const double head = det_gemm_kmajor_us(whole, dx.N, dx.K, true, false, partial);
    const double with_rest = head + kLaunchUs + best_pair_us(tail_of(dx, whole), dw, cus, of, &config);
    if (with_rest < best) {
      best = with_rest;
      plan = {config, whole};
    }
  }
  const bool small_dx = plan.config != RLK_LINEAR_BWD_CFG_SEPARATE && kPairTiles[plan.config].dx_bn < 256 && plan.head_rows == 0;
  // Nor are those of 256 x 128 of dW, which are chosen where its few tiles of 256 x 256 would leave compute units idle (theirs / 192
  // tokens on four waves, us: 1614, 2048, 2048 33.1 / 39.7; 3358, 1024, 4096 55.0 / 64.5; 803, 4096, 1024 21.1 / 25.0; 2960, 4096, 1024 51.3 /
  // 59.8; 6069, 2880, 1440 107.1 / 118.1).
  const bool half_dw = plan.config != RLK_LINEAR_BWD_CFG_SEPARATE && kPairTiles[plan.config].dw_bm < 256;
  // Below its fit solo_pair_us() took what eight waves do faster. Their launch / the one that it chose, us: behind the forward up to 256
  // tokens, 157, 12288, 4096 122.5 / 126.6, 163, 14336, 4096 141.4 / 144.3; with weights of which the forward left nothing in the caches up to
  // 448, the backward alone at 129, 12288, 4096 72.8 / 76.7, 264: 84.2 / 88.6, 440, 6144, 4096 67.6 / 70.9, 380, 14336, 4096 108.4 / 111.6.
  const int least_tokens = of == BackwardOf::kManyWeights ? 449 : 257;
  if (!small_dx && !half_dw && dw.K >= least_tokens && solo_pair_serves(dx, dw)) {
    for (const int bm : {256, 192, 128}) {
      const double us = solo_pair_us(dx, dw, bm, cus);
      if (us < best) {
        best = us;
        plan.solo_tokens = bm;
      }
    }
  }
  return plan;
}

hipError_t linear_backward_launch(GemmProblem dx, const GemmProblem& dw, LinearBackwardPlan plan, hipStream_t stream) {
  if (!one_launch_serves(dx, dw)) plan = {RLK_LINEAR_BWD_CFG_SEPARATE, 0};
  if (plan.solo_tokens != 0 && solo_pair_serves(dx, dw))
    return plan.solo_tokens == 256   ? launch_pair_solo<256>(dx, dw, stream)
           : plan.solo_tokens == 192 ? launch_pair_solo<192>(dx, dw, stream)
                                     : launch_pair_solo<128>(dx, dw, stream);
  if (plan.head_rows > 0) {
    const GemmProblem head = head_of(dx, plan.head_rows);
    const hipError_t err = det_gemm_launch(head.W, head.X, head.C, head.ldc, head.M, head.N, head.K, false, RLK_GEMM_CFG_AUTO, stream);
    if (err != hipSuccess) return err;
    dx = tail_of(dx, plan.head_rows);
  }
  const PairTiles& t = kPairTiles[plan.config];
  const bool dx_first =
      plan.config != RLK_LINEAR_BWD_CFG_SEPARATE && dx_tile_us(t, dx, dw.K, BackwardOf::kLinear) >= dw_tile_us(t, dw);
  switch (plan.config) {
    case RLK_LINEAR_BWD_CFG_SEPARATE: {
      const hipError_t err = det_gemm_launch(dx.W, dx.X, dx.C, dx.ldc, dx.M, dx.N, dx.K, false, RLK_GEMM_CFG_AUTO, stream);
      if (err != hipSuccess) return err;
      return det_gemm_launch(dw.W, dw.X, dw.C, dw.ldc, dw.M, dw.N, dw.K, false, RLK_GEMM_CFG_AUTO, stream);
    }
    case RLK_LINEAR_BWD_CFG_256x256_256x256:
      return launch_pair<Pair256x256, 1, 2, Pair256x256>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_256x128_256x256:
      return launch_pair<Pair256x128, 1, 2, Pair256x256>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_256x256_256x128:
      return launch_pair<Pair256x256, 1, 2, Pair256x128>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_256x128_256x128:
      return launch_pair<Pair256x128, 1, 2, Pair256x128>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_128x128_256x256:
      return launch_pair<Pair128x128, 2, 2, Pair256x256>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_64x64_256x256:
      return launch_pair<Pair64x64, 2, 4, Pair256x256>(dx, dw, dx_first, stream);
    case RLK_LINEAR_BWD_CFG_256x192_256x256:
      return launch_pair<Pair256x192, 1, 2, Pair256x256>(dx, dw, dx_first, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace rlk
