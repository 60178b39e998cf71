// A workgroup's share of a product's 256 x 256 tiles on the loop of det_gemm_solo.h, with the rounding and the stores.
#pragma once

#include "det_gemm_body.h"
#include "det_gemm_solo.h"

namespace rlk {

// C[M, N] = X[M, K] W[N, K]^T in tiles_m x tiles_n tiles.
struct SoloProblem {
  MatView W, X;
  bf16_bits* C;
  int64_t ldc;
  int M, N, K;
  int tiles_m, tiles_n, group_m;
};
template <class S = SoloShape>
inline SoloProblem solo_problem(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K) {
  SoloProblem p{W, X, reinterpret_cast<bf16_bits*>(C), ldc, M, N, K, (M + S::BM - 1) / S::BM, (N + S::BN - 1) / S::BN, 1};
  p.group_m = p.tiles_m < 8 ? p.tiles_m : 8;
  return p;
}

// The tiles first, first + step, ... < total in the order of tile_order(); at least one.
template <class Layout>
__device__ __forceinline__ void solo_product(const SoloProblem& p, int first, int step, int total, char* lds) {
  using S = typename Layout::Shape;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto tile_at = [&](int block, int& n0, int& m0) __attribute__((always_inline)) {
    const TileOrder at = tile_order(block, p.tiles_m, p.tiles_n, p.group_m);
    n0 = at.tile_n * S::BN;
    m0 = at.tile_m * S::BM;
  };
  auto done = [&](int block, SoloAccOf<S>& acc, char*) __attribute__((always_inline)) -> bool {
    int n0, m0;
    tile_at(block, n0, m0);
    const int lane = solo_lane(), grp = lane >> 4;
    constexpr int kWaveN = 16 * S::TN, kWaveM = 16 * S::TM;
    const int n_wave = n0 + wave % S::WN * kWaveN, m_wave = m0 + wave / S::WN * kWaveM;
    const int m_lane = m_wave + (lane & 15);
    if (n_wave + kWaveN <= p.N && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && (p.ldc & 7) == 0) {
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        bf16_bits* const row = p.C + (int64_t)(m_lane + jm * 16) * p.ldc + n_wave;
#pragma unroll
        for (int h = 0; h < S::TN / 4; ++h) {
          const auto &a = acc[4 * h][jm], &b = acc[4 * h + 1][jm], &c = acc[4 * h + 2][jm], &d = acc[4 * h + 3][jm];
          if constexpr (Layout::kW) solo_store_span_kmajor(row + h * 64, grp, m_lane + jm * 16 < p.M, a, b, c, d);
          else solo_store_span(row + h * 64, grp, m_lane + jm * 16 < p.M, a, b, c, d);
        }
        if constexpr (S::TN % 4 != 0) {  // 32 features, of which a lane has eight
          const auto &a = acc[S::TN - 2][jm], &b = acc[S::TN - 1][jm];
          if (m_lane + jm * 16 < p.M)
            *reinterpret_cast<u32x4_t*>(row + S::TN / 4 * 64 + grp * 8) =
                u32x4_t{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
        }
      }
      return m_wave + kWaveM <= p.M;
    }
    const int alignment = solo_row_alignment(p.C, p.ldc);
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      const int m = m_lane + jm * 16;
      if (m >= p.M) continue;
      bf16_bits* const row = p.C + (int64_t)m * p.ldc;
      auto run = [&](auto tiles, int jn, int n) __attribute__((always_inline)) {  // a lane's consecutive features: four of each MFMA tile
        constexpr int kTiles = decltype(tiles)::value;
        uint32_t packed[2 * kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
          packed[2 * t] = pack_bf16x2(acc[jn + t][jm][0], acc[jn + t][jm][1]);
          packed[2 * t + 1] = pack_bf16x2(acc[jn + t][jm][2], acc[jn + t][jm][3]);
        }
        solo_store_run<4 * kTiles>(row + n, p.N - n, alignment, packed);
      };
      if constexpr (Layout::kW) {
#pragma unroll
        for (int jn = 0; jn < S::TN; ++jn) run(IntTag<1>{}, jn, n_wave + jn * 16 + grp * 4);
      } else {
#pragma unroll
        for (int h = 0; h < S::TN / 4; ++h) run(IntTag<4>{}, 4 * h, n_wave + h * 64 + grp * 16);
        if constexpr (S::TN % 4 != 0) run(IntTag<2>{}, S::TN - 2, n_wave + S::TN / 4 * 64 + grp * 8);
      }
    }
    return false;
  };
  solo_tiles<SoloPlainRows<S>, S::TN / 2 * S::TM, false, Layout>(p.W, p.X, p.K, first, step, total, lds, tile_at, done);
}

}  // namespace rlk
