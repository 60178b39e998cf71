// What one workgroup of a det_gemm launch does: which tile it owns, the main loop, the rounding and the store. Shared by the
// launches of one product (det_gemm.hip) and of two at once (det_gemm_pair.hip).
#pragma once

#include "det_gemm_tile.h"

namespace rlk {

// LOOP selects the main loop: kLoopGeneric (any strides, element loads),
// kLoopStaged (16-byte loads through registers) or kLoopPingPong (direct-to-LDS
// loads, two wave groups half an iteration apart). All three run the same MFMA chain.
// The K-major variants are the ping-pong loop with the weight operand (B[K,N], N contiguous),
// the activation operand (x[k * ld + m], tokens contiguous) or both read through transposing
// LDS loads.
enum : int {
  kLoopGeneric = 0,
  kLoopStaged = 1,
  kLoopPingPong = 2,
  kLoopPingPongKMajor = 3,   // weight K-major
  kLoopPingPongXKMajor = 4,  // activation K-major
  kLoopPingPongBothKMajor = 5,
  kLoopStagedKMajor = 7,     // register-staged, weight K-major (the small tiles), K % 64 == 0
  kLoopStagedKMajorTail = 8, // the same with a zero-filled last K tile
  kLoopPingPongWStream = 9,  // kLoopPingPong with the weight read past the caches
  kLoopQuad = 10,            // four waves 2 x 2
  kLoopQuadWStream = 11,     // the same with the weight read past the caches
  kLoopQuadPrefetch = 12     // the same with a wave that prefetches the weight panel
};
constexpr bool loop_weight_kmajor(int loop) {
  return loop == kLoopPingPongKMajor || loop == kLoopPingPongBothKMajor || loop == kLoopStagedKMajor ||
         loop == kLoopStagedKMajorTail;
}
constexpr bool loop_act_kmajor(int loop) { return loop == kLoopPingPongXKMajor || loop == kLoopPingPongBothKMajor; }

// The small K-major tiles have a wave that prefetches their weight panel when two or more workgroups read it.
template <int LOOP, int KS>
constexpr bool has_prefetch_wave() {
  return (LOOP == kLoopPingPongKMajor && KS > 1) || LOOP == kLoopQuadPrefetch;
}
constexpr int kPrefetchDumpBytes = kWave * 4;

// Tile raster: XCD-compact ids, then column groups of group_m token tiles so
// the tiles resident on one XCD share weight and activation panels in its L2.
struct TileOrder {
  int id, within, width, tile_m, tile_n;
};
__device__ __forceinline__ TileOrder tile_order(int block, int tiles_m, int tiles_n, int group_m) {
  TileOrder o;
  o.id = xcd_compact_id(block, tiles_m * tiles_n);
  const int per_group = group_m * tiles_n;
  const int group = o.id / per_group;
  const int first_m = group * group_m;
  o.width = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
  o.within = o.id - group * per_group;
  o.tile_m = first_m + o.within % o.width;
  o.tile_n = o.within / o.width;
  return o;
}

// One tile of a launch: workgroup `block` of the tiles_m x tiles_n that the problem consists of.
template <class S, int LOOP, bool OUT_F32, int KS, int NS, bool PREFETCH = has_prefetch_wave<LOOP, KS>()>
__device__ __forceinline__ void det_gemm_tile(const MatView& W, const MatView& X, void* __restrict__ C, int64_t ldc, int M,
                                              int N, int K, int tiles_m, int tiles_n, int group_m, int block, char* lds) {
  const int total = tiles_m * tiles_n;
  const TileOrder at = tile_order(block, tiles_m, tiles_n, group_m);
  const int id = at.id, within = at.within, width = at.width, tile_m = at.tile_m, tile_n = at.tile_n;
  const int n0 = tile_n * S::BN;
  const int m0 = tile_m * S::BM;

  if constexpr (PREFETCH) {
    if (threadIdx.x >= S::kThreads) {
      // the workgroups of this panel that run on this XCD: their ids are neighbours
      const int panel = id - within % width;
      const int lo = max(panel, xcd_compact_id(block % kXcds, total));
      const int hi = min(panel + width, xcd_compact_id(block % kXcds, total) + xcd_id_count(block, total));
      if constexpr (LOOP == kLoopQuadPrefetch)
        prefetch_quad_panel<S, KS, NS>(W, n0, K, id - lo, hi - lo, lds + NS * KS * S::kStageBytes);
      else
        prefetch_kmajor_panel<S, KS, NS>(W, n0, K - K % (KS * kTileK), id - lo, hi - lo, lds + NS * KS * S::kStageBytes);
      return;
    }
  }
  f32x4_t acc[S::TN][S::TM];
  if constexpr (LOOP == kLoopQuad || LOOP == kLoopQuadWStream || LOOP == kLoopQuadPrefetch) {
    tile_mainloop_quad<S, KS, NS, LOOP == kLoopQuadWStream>(W, X, n0, m0, K, lds, acc);
  } else if constexpr (LOOP == kLoopStagedKMajor || LOOP == kLoopStagedKMajorTail) {
    tile_mainloop_staged_kmajor<S, KS, LOOP == kLoopStagedKMajorTail>(W, X, n0, m0, K, lds, acc);
  } else if constexpr (LOOP == kLoopPingPongWStream) {
    tile_mainloop_pingpong<S, false, false, PlainRowMap<S>, KS, NS, true>(W, X, n0, m0, K, lds, acc);
  } else if constexpr (LOOP >= kLoopPingPongKMajor) {
    // whole stages through the ping-pong loop, the rest of a reduction length that they do not divide behind it
    // (Single K tiles: the mask and the one call below. With a signed remainder, or as the loop that deeper stages need,
    // the compiler brings the tail's addresses into the main loop: weight gradients of 65 to 1000 tokens 2 to 6 % slower.)
    const int k_whole = KS == 1 ? K & ~(kTileK - 1) : K - K % (KS * kTileK);
    if (k_whole > 0) {
      tile_mainloop_pingpong<S, loop_weight_kmajor(LOOP), loop_act_kmajor(LOOP), PlainRowMap<S>, KS, NS>(
          W, X, n0, m0, k_whole, lds, acc);
    } else {  // fewer than 64 K values: the tail step is the whole reduction
#pragma unroll
      for (int jn = 0; jn < S::TN; ++jn)
#pragma unroll
        for (int jm = 0; jm < S::TM; ++jm) acc[jn][jm] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (KS == 1) {
      if (k_whole != K) tile_tail_step<S, loop_weight_kmajor(LOOP), loop_act_kmajor(LOOP)>(W, X, n0, m0, k_whole, K, lds, acc);
    } else {
      for (int k0 = k_whole; k0 < K; k0 += kTileK)
        tile_tail_step<S, loop_weight_kmajor(LOOP), loop_act_kmajor(LOOP)>(W, X, n0, m0, k0, min(k0 + kTileK, K), lds, acc);
    }
  } else if constexpr (LOOP == kLoopPingPong) {
    tile_mainloop_pingpong<S, false, false, PlainRowMap<S>, KS, NS>(W, X, n0, m0, K, lds, acc);
  } else {
    tile_mainloop_staged<S, LOOP == kLoopStaged>(W, X, n0, m0, K, lds, acc);
  }

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wave_n = wave % S::WN;
  const int wave_m = wave / S::WN;
  const int n_run = n0 + wave_n * 16 * S::TN + (lane >> 4) * S::kRun;  // first feature of this lane's run
  const int m_lane = m0 + wave_m * 16 * S::TM + (lane & 15);

  if constexpr (loop_weight_kmajor(LOOP)) {
    // No run permutation on this path: MFMA tile jn holds features jn*16 + (lane>>4)*4 + q.
    const int n_tile = n0 + wave_n * 16 * S::TN + (lane >> 4) * 4;
    if constexpr (!OUT_F32 && S::TN == 4) {
      // bf16 results of a wave whose 64 features all lie inside N, rows 16-byte aligned (both uniform over the
      // wave): a lane holds four 8-byte pieces of a token's row, 32 bytes apart. A 4 x 4 transpose of the pieces
      // between the four lanes of a token (two butterfly stages of lane swaps over distances 32 and 16: the
      // piece that lane g held at position c ends at lane c, position g) gives every lane the 16 consecutive
      // features 16 g .. 16 g + 15, stored as two 16-byte halves: 128 contiguous bytes per token and instruction
      // pair instead of 32 per instruction.
      // Ordinary stores. Non-temporal ones make a GEMM that is relaunched on the same operands 4-5 % faster (gate_up
      // at 4096 tokens 574 -> 550 us): the result then bypasses the 256 MB memory-side cache and the weights stay in
      // it from one launch to the next. With weights that come from HBM, as in a model with more than one layer,
      // they measured the same or 1 % slower, and gate_up and down launched alternately 0.6 % slower; not used.
      const int n_wave = n0 + wave_n * 64;
      const bool whole_span = n_wave + 64 <= N && (reinterpret_cast<uintptr_t>(C) & 15) == 0 && (ldc & 7) == 0;
      if (whole_span) {
        const int grp = lane >> 4;
#pragma unroll
        for (int jm = 0; jm < S::TM; ++jm) {
          uint32_t w[4][2];
#pragma unroll
          for (int jn = 0; jn < 4; ++jn) {
            w[jn][0] = pack_bf16x2(acc[jn][jm][0], acc[jn][jm][1]);
            w[jn][1] = pack_bf16x2(acc[jn][jm][2], acc[jn][jm][3]);
          }
#pragma unroll
          for (int c = 0; c < 2; ++c)  // lane bit 5 <-> piece bit 1
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const auto r = __builtin_amdgcn_permlane32_swap(w[c][e], w[c + 2][e], false, false);
              w[c][e] = r[0];
              w[c + 2][e] = r[1];
            }
#pragma unroll
          for (int c = 0; c < 4; c += 2)  // lane bit 4 <-> piece bit 0
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const auto r = __builtin_amdgcn_permlane16_swap(w[c][e], w[c + 1][e], false, false);
              w[c][e] = r[0];
              w[c + 1][e] = r[1];
            }
          const int m = m_lane + jm * 16;
          if (m < M) {
            bf16_bits* dst = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc + n_wave + grp * 16;
            *reinterpret_cast<u32x4_t*>(dst) = u32x4_t{w[0][0], w[0][1], w[1][0], w[1][1]};
            *reinterpret_cast<u32x4_t*>(dst + 8) = u32x4_t{w[2][0], w[2][1], w[3][0], w[3][1]};
          }
        }
        return;
      }
    }
#pragma unroll
    for (int jm = 0; jm < S::TM; ++jm) {
      const int m = m_lane + jm * 16;
      if (m >= M) continue;
#pragma unroll
      for (int jn = 0; jn < S::TN; ++jn) {
        const int n = n_tile + jn * 16;
        if (OUT_F32) {
          float* dst = reinterpret_cast<float*>(C) + (int64_t)m * ldc + n;
          if (n + 4 <= N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
            *reinterpret_cast<f32x4_t*>(dst) = acc[jn][jm];
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (n + q < N) dst[q] = acc[jn][jm][q];
          }
        } else {
          bf16_bits* dst = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc + n;
          const uint32_t lo = pack_bf16x2(acc[jn][jm][0], acc[jn][jm][1]);
          const uint32_t hi = pack_bf16x2(acc[jn][jm][2], acc[jn][jm][3]);
          if (n + 4 <= N && (reinterpret_cast<uintptr_t>(dst) & 7) == 0) {
            *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{lo, hi};
          } else {
            const uint32_t packed[2] = {lo, hi};
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (n + q < N) dst[q] = (bf16_bits)((packed[q >> 1] >> ((q & 1) * 16)) & 0xffffu);
          }
        }
      }
    }
    return;
  }

  if constexpr (!OUT_F32 && S::TN == 4) {
    // bf16 results of a wave whose 64 features all lie inside N, rows 16-byte aligned (both uniform over the wave):
    // a lane holds the 16 consecutive features 16 g .. 16 g + 15 of a token as two 16-byte halves, so a store
    // instruction would write 16-byte pieces 32 bytes apart. Two lane swaps (over distance 16 between the halves,
    // then over distance 32) rotate (half, lane bit 5, lane bit 4) into (lane bit 4, half, lane bit 5): store s of
    // lane g then holds features 32 s + 8 g .. + 7, 64 contiguous bytes per token and instruction.
    const int n_wave = n0 + wave_n * 64;
    const bool whole_span = n_wave + 64 <= N && (reinterpret_cast<uintptr_t>(C) & 15) == 0 && (ldc & 7) == 0;
    if (whole_span) {
      const int grp = lane >> 4;
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        uint32_t half[2][4];
#pragma unroll
        for (int jn = 0; jn < 4; ++jn) {
          half[jn >> 1][2 * (jn & 1)] = pack_bf16x2(acc[jn][jm][0], acc[jn][jm][1]);
          half[jn >> 1][2 * (jn & 1) + 1] = pack_bf16x2(acc[jn][jm][2], acc[jn][jm][3]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto r = __builtin_amdgcn_permlane16_swap(half[0][e], half[1][e], false, false);
          const auto t = __builtin_amdgcn_permlane32_swap(r[0], r[1], false, false);
          half[0][e] = t[0];
          half[1][e] = t[1];
        }
        const int m = m_lane + jm * 16;
        if (m < M) {
          bf16_bits* dst = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc + n_wave + grp * 8;
          *reinterpret_cast<u32x4_t*>(dst) = u32x4_t{half[0][0], half[0][1], half[0][2], half[0][3]};
          *reinterpret_cast<u32x4_t*>(dst + 32) = u32x4_t{half[1][0], half[1][1], half[1][2], half[1][3]};
        }
      }
      return;
    }
  }

#pragma unroll
  for (int jm = 0; jm < S::TM; ++jm) {
    const int m = m_lane + jm * 16;
    if (m >= M) continue;
    if (OUT_F32) {
      float* row = reinterpret_cast<float*>(C) + (int64_t)m * ldc;
      const bool vec_ok = (n_run + S::kRun <= N) && ((reinterpret_cast<uintptr_t>(row + n_run) & 15) == 0);
      if (vec_ok) {
#pragma unroll
        for (int jn = 0; jn < S::TN; ++jn) *reinterpret_cast<f32x4_t*>(row + n_run + jn * 4) = acc[jn][jm];
      } else {
#pragma unroll
        for (int jn = 0; jn < S::TN; ++jn)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (n_run + jn * 4 + q < N) row[n_run + jn * 4 + q] = acc[jn][jm][q];
      }
    } else {
      bf16_bits* row = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc;
      uint32_t packed[2 * S::TN];
#pragma unroll
      for (int jn = 0; jn < S::TN; ++jn) {
        packed[2 * jn] = pack_bf16x2(acc[jn][jm][0], acc[jn][jm][1]);
        packed[2 * jn + 1] = pack_bf16x2(acc[jn][jm][2], acc[jn][jm][3]);
      }
      // an odd number of MFMA tiles per wave makes a run an odd multiple of 8 bytes: 8-byte stores
      constexpr int kAlign = (S::TN % 2 == 0) ? 16 : 8;
      const bool vec_ok =
          (n_run + S::kRun <= N) && ((reinterpret_cast<uintptr_t>(row + n_run) & (kAlign - 1)) == 0);
      if (vec_ok) {
        if (S::TN % 2 == 1) {
#pragma unroll
          for (int v = 0; v < S::TN; ++v)
            *reinterpret_cast<u32x2_t*>(row + n_run + v * 4) = u32x2_t{packed[2 * v], packed[2 * v + 1]};
        } else if (S::TN >= 2) {
#pragma unroll
          for (int v = 0; v < S::TN / 2; ++v)
            *reinterpret_cast<u32x4_t*>(row + n_run + v * 8) =
                u32x4_t{packed[4 * v], packed[4 * v + 1], packed[4 * v + 2], packed[4 * v + 3]};
          if (S::TN % 2)
            *reinterpret_cast<u32x2_t*>(row + n_run + (S::TN - 1) * 4) =
                u32x2_t{packed[2 * S::TN - 2], packed[2 * S::TN - 1]};
        } else {
          *reinterpret_cast<u32x2_t*>(row + n_run) = u32x2_t{packed[0], packed[1]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < S::kRun; ++e)
          if (n_run + e < N) row[n_run + e] = (bf16_bits)((packed[e >> 1] >> ((e & 1) * 16)) & 0xffffu);
      }
    }
  }
}

}  // namespace rlk
