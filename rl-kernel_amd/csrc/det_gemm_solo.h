// One wave per SIMD: four waves, each a 128 x 128 quarter of a 256 x 256 tile, and one stream of loads over all the tiles of a
// workgroup.
//
// A square wave tile reads 16 fragments from LDS per 64 MFMAs (the 64 x 128 wave tiles of the ping-pong loop: 12 per 32). Its
// 256 accumulator registers and two sets of 16 fragments need the whole unified register file of a SIMD, so a wave has no
// partner to hide its stalls; what keeps the matrix pipe busy is that everything else is spread between the MFMAs, one
// instruction at a time: a fragment read of the next K step every four, a load every eight.
//
//   * The LDS holds five parts of 32 KiB, a part being the weight rows or the token rows of one K tile: both parts of K tiles t
//     and t + 1, and a spare. Under the first K step of tile t the weight rows of tile t + 2 arrive in the spare, under the
//     second its token rows in the place of the weight rows of tile t, which every wave has then read, and the place of the
//     token rows of tile t becomes the spare. So a wave starts eight loads in either step and there is one barrier per K tile.
//     (All sixteen loads in one step: 12 % slower. Stages of 32 K values, which need no spare, move half lines, and the
//     second half comes from the L2 again: 11 to 30 % slower.)
//   * Behind the last K tile of an output tile the loads go on with the first of the next one, whose operands are in LDS when the
//     results have been stored: a tile pays neither for its first loads nor for its stores.
//   * The MFMAs are written in assembly with the accumulator as one operand: left to the compiler, which has not a register to
//     spare, accumulators are copied at the loop's end.
//
// Bound by the package's power cap on all but zeros and short reductions. Weights of three layers in turn, us, ping-pong kernel ->
// this: qkv (6144 x 4096) at 16384 tokens 558 -> 539 (1531 TFLOP/s), 4096 outputs with K = 512 88.5 -> 74.4, gate_up with its
// activation and down at 4096 tokens 849 -> 828; one tile per workgroup 98.3 -> 97.1 (4096 x 4096 at 4096). On zeros 470 -> 442,
// with one tile of K = 12288 179 -> 188: 1110 cycles a K step of 1024, 20 of them the barrier, 20 the loads. The vendor library's
// kernel, which has the same geometry, takes 1100 and 3 % less time at the cap. solo_tiles_pay() says where it runs.
//
// K-major operands (SoloLayout) come from transposing reads of half a fragment each, 24 or 32 of them a K step, and need no vector
// instruction beside a load: with a compare and a select each to zero what lies past a ragged reduction they were 3 to 4 % slower.
// Ping-pong -> this, us: both operands K-major, 4096 outputs, K = 4096, 12288 rows 316 -> 292, K = 4120 with 151936 rows 4057 ->
// 3689; a K-major weight, 4096 x 12288 with K = 4096 297 -> 291, 4096 x 4096 98.5 -> 96.7. Where a launch leaves the last round
// half empty, or holds two products (det_gemm_pair.hip), more.
//
// Smaller shapes (192 x 256, 256 x 192 in five parts; 192 x 192, 256 x 128, 192 x 128 in a ring of three or four stages of a K tile,
// token rows a step behind weight rows) have the same wave layout, half a tile by half. What bounds them is LDS and, in one
// round with a weight from HBM, the loads; kTileCandidates has what they measured beside eight waves.
//
// Same MFMA chain per output element as every other loop. Needs 16-byte aligned rows and rows whose byte offsets inside a tile stay
// below 4 GiB (solo_offsets_fit(); 2 GiB beside a K-major operand, solo_kmajor_fits()); K % 64 == 0 with two native operands.
#pragma once

#include "det_gemm_tile.h"

namespace rlk {

using SoloShape = TileShape<256, 256, 2, 2>;
constexpr int kSoloPartBytes = 256 * kRowBytes;
constexpr int kSoloParts = 5;
constexpr int kSoloLdsBytes = kSoloParts * kSoloPartBytes;

// `rows`: from the first row of a tile to its last.
inline bool solo_offsets_fit(const MatView& v, int64_t rows = SoloShape::BN) {
  return v.row_stride >= 0 && v.row_stride < ((int64_t)1 << 31) && rows * v.row_stride * 2 + 8192 < ((int64_t)1 << 32);
}

// Which weight row, counted from the first one of the tile's features, LDS row r of the weight part holds.
// Plain: a wave's 128 features are two spans of 64, and in each of them a lane owns 16 consecutive ones, as with the four MFMA
// tiles of a 64-feature wave column (weight_row_of_lds_row):
//   acc[4 h + jn][jm][q] is feature 128 wave_n + 64 h + 16 (lane >> 4) + 4 jn + q of token 128 wave_m + 16 jm + (lane & 15).
// Gated: half as many features of both halves of a packed gate/up weight [2 I, K], with T = TN / 2,
//   acc[jn][jm][q] the gate and acc[T + jn][jm][q] the up projection of feature 16 T wave_n + 4 T (lane >> 4) + 4 jn + q.
// (Of a wave's 96 features the last 32 are a span of two MFMA tiles, a lane's eight features.)
template <class S>
struct SoloPlainRows {
  static __device__ __forceinline__ int feature(int r) {
    constexpr int kWaveRows = 16 * S::TN;
    const int in_wave = r % kWaveRows, span = in_wave & ~63;
    const bool half = kWaveRows % 64 != 0 && span + 64 > kWaveRows;
    return r - in_wave + span + ((r & 15) >> 2) * (half ? 8 : 16) + (((in_wave - span) >> 4) & 3) * 4 + (r & 3);
  }
  static __device__ __forceinline__ int64_t row(int r, int last, int) { return min(feature(r), last); }
  static __device__ __forceinline__ int features(const MatView& W) { return W.rows; }
};
// SPLIT: of two weights [I, K]. Odd waves load the up rows, even ones the gate rows: W.ptr is the one or the other.
template <class S, bool SPLIT = false>
struct SoloGatedRows {
  static __device__ __forceinline__ int64_t row(int r, int last, int half_rows) {
    constexpr int kWaveRows = 16 * S::TN, kTiles = S::TN / 2;
    const int wave = r / kWaveRows, tile = r % kWaveRows / 16;
    const int f = wave * (kWaveRows / 2) + ((r & 15) >> 2) * (4 * kTiles) + tile % kTiles * 4 + (r & 3);
    return min(f, last) + (SPLIT ? 0 : tile / kTiles * half_rows);
  }
  static __device__ __forceinline__ int features(const MatView& W) { return SPLIT ? W.rows : W.rows / 2; }
};

// How the operands lie in memory. A K-major part holds four columns of 64 rows (features, tokens), each 64 K rows of 128 bytes, in the
// layout of the ping-pong loop (kmajor_swizzle); a wave loads one column, eight K rows a block, and reads two columns, two
// transposing reads a fragment. In a K-major weight's tile acc[jn][jm][q] is feature 128 wave_n + 16 jn + 4 (lane >> 4) + q.
// With a K-major operand the reduction may end inside a K tile. What lies past its end is outside the buffer's range, which reads
// zeros, in either operand: a K-major buffer ends behind the last K row (a block's scalar offset never exceeds its size, or the
// check, offset >= size - scalar offset, would wrap), and chunks of a native one get an offset beyond it (whole chunks are read:
// K % 8 == 0 or MatView::k_padded).
template <bool W_KMAJOR, bool X_KMAJOR, class SHAPE = SoloShape>
struct SoloLayout {
  using Shape = SHAPE;
  static constexpr bool kW = W_KMAJOR, kX = X_KMAJOR, kTail = W_KMAJOR || X_KMAJOR;
  static_assert((!W_KMAJOR || SHAPE::BN == 256) && (!X_KMAJOR || SHAPE::BM == 256), "a column for each wave");
  // Stages of a whole K tile where three or more of them fit, else five parts.
  static constexpr int kStages = kSoloLdsBytes / SHAPE::kStageBytes;
  static constexpr bool kRing = kStages >= 3;
  static constexpr int kLds = kRing ? kStages * SHAPE::kStageBytes : kSoloLdsBytes;
};
constexpr uint32_t kSoloRange = 0x7fff0000, kSoloOutside = 0x80000000;  // of a native buffer, bytes; what takes an offset out of it

// Whether a tile's offsets fit beside a K-major operand.
inline bool solo_kmajor_fits(const MatView& v) {
  if (v.k_stride != 1) return v.k_stride >= 0 && v.k_stride < ((int64_t)1 << 23);  // 64 K rows
  return v.row_stride >= 0 && v.row_stride < ((int64_t)1 << 21);                   // 256 rows
}

// Half a K-major fragment: four K values of this lane's row. (The qualifier: see read_kmajor_fragment.)
typedef const __attribute__((address_space(3))) char* lds_bytes_t;  // 32 bits whatever the compiler knows of the pointer
__device__ __forceinline__ u32x2_t solo_read_transposed(lds_bytes_t __restrict__ at) {
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
  typedef __attribute__((address_space(3))) bf16x4_t* lds_bf16x4_ptr_t;
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_ptr_t)at));
}

// The lane, hidden from the compiler: what is derived from it outside the K loop is then not kept in registers across the loop,
// which has none to spare (the spilled ones were read back behind the stores of a tile, and waited for them).
__device__ __forceinline__ int solo_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}

// bf16 results of the four lanes of a token (lanes l, l + 16, l + 32, l + 48, 16 consecutive features each) into the 64 features
// at `span`, in two stores of 64 contiguous bytes per token (the lane swaps of det_gemm_tile's epilogue). Every lane of the wave
// calls it; 16-byte aligned.
__device__ __forceinline__ void solo_store_span(bf16_bits* span, int grp, bool live, const f32x4_t& v0, const f32x4_t& v1,
                                                const f32x4_t& v2, const f32x4_t& v3) {
  uint32_t half[2][4] = {{pack_bf16x2(v0[0], v0[1]), pack_bf16x2(v0[2], v0[3]), pack_bf16x2(v1[0], v1[1]), pack_bf16x2(v1[2], v1[3])},
                         {pack_bf16x2(v2[0], v2[1]), pack_bf16x2(v2[2], v2[3]), pack_bf16x2(v3[0], v3[1]), pack_bf16x2(v3[2], v3[3])}};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const auto r = __builtin_amdgcn_permlane16_swap(half[0][e], half[1][e], false, false);
    const auto t = __builtin_amdgcn_permlane32_swap(r[0], r[1], false, false);
    half[0][e] = t[0];
    half[1][e] = t[1];
  }
  if (live) {
    *reinterpret_cast<u32x4_t*>(span + grp * 8) = u32x4_t{half[0][0], half[0][1], half[0][2], half[0][3]};
    *reinterpret_cast<u32x4_t*>(span + grp * 8 + 32) = u32x4_t{half[1][0], half[1][1], half[1][2], half[1][3]};
  }
}

// The same for a K-major weight, whose MFMA tiles hold 16 consecutive features each, a lane four of each tile: v0 to v3 are the tiles
// of the 64 features. A lane's piece of tile t trades places so that store s holds features 32 s + 8 g .. + 7 of lane group g: two
// lane swaps as above, over distance 32 first.
__device__ __forceinline__ void solo_store_span_kmajor(bf16_bits* span, int grp, bool live, const f32x4_t& v0, const f32x4_t& v1,
                                                       const f32x4_t& v2, const f32x4_t& v3) {
  uint32_t piece[4][2] = {{pack_bf16x2(v0[0], v0[1]), pack_bf16x2(v0[2], v0[3])}, {pack_bf16x2(v1[0], v1[1]), pack_bf16x2(v1[2], v1[3])},
                          {pack_bf16x2(v2[0], v2[1]), pack_bf16x2(v2[2], v2[3])}, {pack_bf16x2(v3[0], v3[1]), pack_bf16x2(v3[2], v3[3])}};
#pragma unroll
  for (int s = 0; s < 4; s += 2)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const auto r = __builtin_amdgcn_permlane32_swap(piece[s][e], piece[s + 1][e], false, false);
      const auto t = __builtin_amdgcn_permlane16_swap(r[0], r[1], false, false);
      piece[s][e] = t[0];
      piece[s + 1][e] = t[1];
    }
  if (live) {
    *reinterpret_cast<u32x4_t*>(span + grp * 8) = u32x4_t{piece[0][0], piece[0][1], piece[1][0], piece[1][1]};
    *reinterpret_cast<u32x4_t*>(span + grp * 8 + 32) = u32x4_t{piece[2][0], piece[2][1], piece[3][0], piece[3][1]};
  }
}

// What every row of a bf16 result starts on a multiple of: 16, 8, 4 or 2 bytes.
__device__ __forceinline__ int solo_row_alignment(const void* C, int64_t ld) {
  const int low = (int)((reinterpret_cast<uintptr_t>(C) | (uintptr_t)(2 * ld)) & 15);
  return low == 0 ? 16 : low & -low;
}

// E results of a lane in a row (`packed` in pairs) at `to`, E elements into which the row's alignment goes on; `inside` of them are
// columns of the result. For the waves whose features are not whole 16-byte spans inside the result: the last columns, and rows of
// any pitch. Bound by the addresses that the stores of scattered rows take and by code that is fetched for the first time, so whole
// runs leave in the widest stores there are, from odd addresses on in pairs behind one element, and the last columns in fours. Eight
// waves a tile / four, element by element / this, us: 4000 tokens, K = 512, 4100 outputs 29.7 / 61.0 / 24.7, 4098: 46.3 / 63.3 / 28.9,
// 4097: 56.0 / 62.5 / 30.5, K = 1024, 8274 tokens, 1000 outputs 23.4 / 27.4 / 21.5; a K-major weight, 5152 tokens, 2808 outputs, K =
// 296 20.7 / 25.6 / 18.1; gated, 3000 tokens, K = 512, I = 5004 49.9 / 71.1 / 37.8, 5001: 58.9 / 71.1 / 39.6. (A branch of its own
// for rows on 4 bytes: up to 10 % less there, and accumulators spilled.)
template <int E>
__device__ __forceinline__ void solo_store_run(bf16_bits* to, int inside, int alignment, const uint32_t (&packed)[E / 2]) {
  constexpr int kPairs = E / 2;
  if (inside >= E) {
    if (E % 8 == 0 && alignment == 16) {
#pragma unroll
      for (int i = 0; i + 4 <= kPairs; i += 4)
        *reinterpret_cast<u32x4_t*>(to + 2 * i) = u32x4_t{packed[i], packed[i + 1], packed[i + 2], packed[i + 3]};
    } else if (alignment >= 8) {
#pragma unroll
      for (int i = 0; i < kPairs; i += 2) *reinterpret_cast<u32x2_t*>(to + 2 * i) = u32x2_t{packed[i], packed[i + 1]};
    } else {
      const bool odd = (reinterpret_cast<uintptr_t>(to) & 2) != 0;
      uint32_t* const words = reinterpret_cast<uint32_t*>(to + (odd ? 1 : 0));
#pragma unroll
      for (int i = 0; i + 1 < kPairs; ++i)
        words[i] = odd ? __builtin_amdgcn_alignbit(packed[i + 1], packed[i], 16) : packed[i];
      if (odd) {
        to[0] = (bf16_bits)(packed[0] & 0xffffu);
        to[E - 1] = (bf16_bits)(packed[kPairs - 1] >> 16);
      } else {
        words[kPairs - 1] = packed[kPairs - 1];
      }
    }
  } else if (inside > 0) {  // the last columns: fours, and element by element behind them
    const int fours = alignment >= 8 ? inside & ~3 : 0;
#pragma unroll
    for (int i = 0; i < kPairs; i += 2)
      if (2 * i < fours) *reinterpret_cast<u32x2_t*>(to + 2 * i) = u32x2_t{packed[i], packed[i + 1]};
    if (fours == inside) return;
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e >= fours && e < inside) to[e] = (bf16_bits)((packed[e >> 1] >> ((e & 1) * 16)) & 0xffffu);
  }
}

// One result out of its accumulator register, where it is wanted: the compiler brings all of them into others first, which in a long
// epilogue it does not have.
__device__ __forceinline__ float solo_result(float accumulator) {
  float value;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(value) : "a"(accumulator));
  return value;
}

template <class S>
using SoloAccOf = f32x4_t[S::TN][S::TM];
typedef SoloAccOf<SoloShape> SoloAcc;

// Runs the tiles first, first + step, ... < total (at least one). tile_at(i, n0, m0) says where tile i lies; done(i, acc, scratch)
// takes its results, may use the spare part of the LDS if it ends on a barrier then, and returns whether this wave has issued STORES
// vector memory instructions, no fewer: so many more may then be in flight at the first wait of the next tile. LONG: done() wants
// the registers of the next tile's first fragments, which are read again behind it. keep() runs once per K tile: an empty asm with the
// values that done() carries from tile to tile as its operands keeps them in registers.
struct SoloKeepsNothing {
  __device__ __forceinline__ void operator()() const {}
};
template <class Rows, int STORES, bool LONG = false, class Layout = SoloLayout<false, false>, class TileAt, class Done, class Keep = SoloKeepsNothing>
__device__ __forceinline__ void solo_tiles(const MatView& W, const MatView& X, int K, int first, int step, int total, char* lds,
                                           TileAt tile_at, Done done, Keep keep = Keep()) {
  using S = typename Layout::Shape;
  constexpr int kLoadsW = S::BN / 32, kLoadsX = S::BM / 32;  // load instructions of a wave per part
  // Loads of K tiles behind the next one that may be in flight when that one is waited for.
  constexpr int kAhead = Layout::kRing ? (Layout::kStages - 2) * (kLoadsW + kLoadsX) : kLoadsW;
  constexpr int kBehind = STORES + kAhead < 63 ? STORES + kAhead : 63;
  const int lane = solo_lane();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int grp = lane >> 4;
  const int nk = Layout::kTail ? (K + kTileK - 1) / kTileK : K / kTileK;

  // The load stream: the next K tile of its output tile, at w_at and x_at. A wave loads a quarter of the rows of either part in
  // blocks of eight rows; block j adds (j & 3) KiB as the instruction's offset, which counts for the LDS address and the global one.
  constexpr int kBlockBytes = 1024, kBlocksPerBase = 4;
  // A K-major operand's column is the wave's, block j K rows [8 j, + 8): a lane has one offset for either chunk position that the
  // swizzle gives it, and the block's K rows are the instruction's scalar offset.
  uint32_t off_w[Layout::kW ? 2 : kLoadsW], off_x[Layout::kX ? 2 : kLoadsX];
  const uint32_t block_w = (uint32_t)W.k_stride * 16, block_x = (uint32_t)X.k_stride * 16;  // bytes of eight K rows
  const char *w_at, *x_at;
  uint32_t range_w = Layout::kTail ? kSoloRange : 0xffffffff, range_x = range_w;  // of the K tile's buffers, which begin below it
  int load_tile = first, load_left = nk;
  auto aim_kmajor = [&](const MatView& v, int row0, uint32_t (&off)[2], const char*& at) __attribute__((always_inline)) {
    at = reinterpret_cast<const char*>(v.ptr + row0) - kBlocksPerBase * kBlockBytes;
    const int lane = solo_lane(), rib = lane >> 3;
    const int last = v.rows - kChunkElems - row0;  // rows past the edge: computed, never stored
    const int chunk = wave * 64 + ((lane & 7) ^ kmajor_swizzle_of_row_in_block(rib)) * kChunkElems;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      off[p] = (uint32_t)rib * (uint32_t)v.k_stride * 2 + (uint32_t)min(chunk ^ (p * 2 * kChunkElems), last) * 2;
      asm volatile("" : "+v"(off[p]));
    }
  };
  auto aim = [&]() __attribute__((always_inline)) {
    int n0, m0;
    tile_at(load_tile, n0, m0);
    if constexpr (Layout::kW) aim_kmajor(W, n0, off_w, w_at);
    else w_at = reinterpret_cast<const char*>(W.ptr + (int64_t)n0 * W.row_stride) - kBlocksPerBase * kBlockBytes;
    if constexpr (Layout::kX) aim_kmajor(X, m0, off_x, x_at);
    else x_at = reinterpret_cast<const char*>(X.ptr + (int64_t)m0 * X.row_stride) - kBlocksPerBase * kBlockBytes;
    const int lane = solo_lane();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = j * 8 + (lane >> 3);
      // rows past the edge: computed, never stored
      const uint32_t in_row = ((lane & 7) ^ (lane >> 3)) * 16 + (kBlocksPerBase - j % kBlocksPerBase) * kBlockBytes;
      // (32 bits each: as halves of 64-bit products they took two registers)
      if constexpr (!Layout::kW) {
        if (j < kLoadsW) {
          const uint32_t row_w = (uint32_t)Rows::row(wave * (8 * kLoadsW) + r, Rows::features(W) - n0 - 1, W.rows / 2);
          off_w[j] = row_w * (uint32_t)W.row_stride * 2 + in_row;
          asm volatile("" : "+v"(off_w[j]));
        }
      }
      if constexpr (!Layout::kX) {
        if (j < kLoadsX) {
          const uint32_t row_x = min(wave * (8 * kLoadsX) + r, X.rows - m0 - 1);
          off_x[j] = row_x * (uint32_t)X.row_stride * 2 + in_row;
          asm volatile("" : "+v"(off_x[j]));
        }
      }
    }
  };
  // The K values of the K tile at hand that are there: the last K tile of an output tile (load_left == 1) may hold fewer than 64.
  const int k_rest = K - (nk - 1) * kTileK;
  auto limit = [&]() __attribute__((always_inline)) {
    if constexpr (!Layout::kTail) return;
    const int k_left = load_left > 1 ? kTileK : k_rest;
    if constexpr (Layout::kW) range_w = (uint32_t)W.k_stride * 2 * k_left + kBlocksPerBase * kBlockBytes;
    if constexpr (Layout::kX) range_x = (uint32_t)X.k_stride * 2 * k_left + kBlocksPerBase * kBlockBytes;
    if constexpr (!(Layout::kW && Layout::kX)) {
      if (load_left == 1 && k_rest != kTileK) {
        const int lane = solo_lane();
        const uint32_t out = ((lane & 7) ^ (lane >> 3)) * kChunkElems < k_rest ? 0 : kSoloOutside;
#pragma unroll
        for (int j = 0; j < (Layout::kW ? kLoadsX : kLoadsW); ++j) {
          if constexpr (!Layout::kW) off_w[j] |= out;
          if constexpr (!Layout::kX) off_x[j] |= out;
        }
      }
    }
  };
  aim();
  limit();
  auto advance = [&]() __attribute__((always_inline)) {
    w_at += Layout::kW ? (int64_t)block_w * 8 : kRowBytes;
    x_at += Layout::kX ? (int64_t)block_x * 8 : kRowBytes;
    if (--load_left == 0) {
      load_left = nk;
      load_tile = load_tile + step < total ? load_tile + step : load_tile;  // past the last tile: its first K tiles again, never read
      aim();
    }
    limit();
  };
  auto load = [&](auto weight, auto block, char* part) __attribute__((always_inline)) {
    constexpr int j = decltype(block)::value;
    constexpr bool kWeight = decltype(weight)::value != 0, kKMajor = kWeight ? Layout::kW : Layout::kX;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(kWeight ? w_at : x_at), 0, kWeight ? range_w : range_x, 0x00027000);
    lds_ptr_t to = (lds_ptr_t)(part + (wave * (kWeight ? kLoadsW : kLoadsX) + j / kBlocksPerBase * kBlocksPerBase) * kBlockBytes);
    constexpr int kOffset = j % kBlocksPerBase * kBlockBytes;
    if constexpr (kKMajor) {
      const uint32_t rows_at = (kWeight ? block_w : block_x) * j + (kBlocksPerBase * kBlockBytes - kOffset);
      const uint32_t off = kWeight ? off_w[(j ^ (j >> 1)) & 1] : off_x[(j ^ (j >> 1)) & 1];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 16, off, min(rows_at, kWeight ? range_w : range_x), kOffset, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 16, kWeight ? off_w[j] : off_x[j], 0, kOffset, 0);
    }
  };
  auto for_blocks = [](auto f) __attribute__((always_inline)) {
    f(IntTag<0>{}), f(IntTag<1>{}), f(IntTag<2>{}), f(IntTag<3>{}), f(IntTag<4>{}), f(IntTag<5>{}), f(IntTag<6>{}), f(IntTag<7>{});
  };

  auto load_part = [&](auto weight, char* part) __attribute__((always_inline)) {
    for_blocks([&](auto j) __attribute__((always_inline)) {
      if constexpr (decltype(j)::value < (decltype(weight)::value ? kLoadsW : kLoadsX)) load(weight, j, part);
    });
  };

  SoloAccOf<S> acc;
  struct Frags {
    u32x4_t w[S::TN], x[S::TM];
  };
  const int frag = (grp ^ (l16 & 7)) << 4;  // of the first K step of a K tile; the second one flips bit 6
  typedef const __attribute__((address_space(3))) u32x4_t* lds_chunk_t;
  constexpr int kColumnBytes = kTileK * kRowBytes;  // 64 rows of a K-major part
  const int tr_row = grp * 8 + (l16 >> 2);          // K row of a transposing read, and its place in a column
  const int tr_at = tr_row * kRowBytes + ((((l16 & 3) >> 1) ^ kmajor_swizzle(tr_row)) << 4) + (l16 & 1) * 8;
  const lds_bytes_t w_rows = (lds_bytes_t)lds + (Layout::kW ? wave % S::WN * 2 * kColumnBytes + tr_at : (wave % S::WN * 16 * S::TN + l16) * kRowBytes);
  const lds_bytes_t x_rows = (lds_bytes_t)lds + (Layout::kX ? wave / S::WN * 2 * kColumnBytes + tr_at : (wave / S::WN * 16 * S::TM + l16) * kRowBytes);
  // Reads of a K step, in the order of the fragments' use: w[0], x[0] to x[7], w[1] to w[7], a K-major one in two halves.
  constexpr int kWReads = Layout::kW ? 2 : 1, kXReads = Layout::kX ? 2 : 1;
  constexpr int kReads = S::TN * kWReads + S::TM * kXReads;
  // Where the fragments of K step `second` of the K tile in a part begin. (The four places of a K-major fragment's tiles kept for both K
  // steps, eight vector instructions fewer, which then stand together behind the barrier: 0.5 % slower.)
  auto step_at = [&](lds_bytes_t rows, int part, bool kmajor, bool second) __attribute__((always_inline)) {
    return rows + part + (kmajor ? (second ? kMfmaK * kRowBytes : 0) : (second ? frag ^ 64 : frag));
  };
  auto read = [&](lds_bytes_t w, lds_bytes_t x, int i, Frags& f) __attribute__((always_inline)) {
    const int of_x = i - kWReads, of_w = of_x < 0 ? i : i - S::TM * kXReads;
    const bool is_x = of_x >= 0 && of_x < S::TM * kXReads;
    auto one = [&](auto kmajor, lds_bytes_t at, int n, u32x4_t* frags) __attribute__((always_inline)) {
      if constexpr (decltype(kmajor)::value) {
        const int tile = n / 2, half = n % 2;  // the 16-row tile is bits 5 and 6 of the place, under the swizzle
        const u32x2_t v =
            solo_read_transposed(at + ((tr_at ^ (tile & 3) << 5) - tr_at) + (tile >> 2) * kColumnBytes + half * 4 * kRowBytes);
        frags[tile][2 * half] = v.x;
        frags[tile][2 * half + 1] = v.y;
      } else {
        frags[n] = *(lds_chunk_t)(at + n * 16 * kRowBytes);
      }
    };
    if (is_x) one(BoolTag<Layout::kX>{}, x, of_x, f.x);
    else one(BoolTag<Layout::kW>{}, w, of_w, f.w);
  };

  auto next_part = [](int at) { return at + kSoloPartBytes < kSoloLdsBytes ? at + kSoloPartBytes : 0; };
  // of the K tile at hand; the spare part, in a ring the stage of the K tile before
  constexpr int kWBytes = S::BN * kRowBytes;
  int w_part = 0, x_part = Layout::kRing ? kWBytes : kSoloPartBytes;
  int spare = Layout::kRing ? (Layout::kStages - 1) * S::kStageBytes : 4 * kSoloPartBytes;
#pragma unroll
  for (int t = 0; t < (Layout::kRing ? Layout::kStages - 1 : 2); ++t) {
    load_part(IntTag<1>{}, lds + t * (Layout::kRing ? S::kStageBytes : 2 * kSoloPartBytes));
    load_part(IntTag<0>{}, lds + t * (Layout::kRing ? S::kStageBytes : 2 * kSoloPartBytes) + x_part);
    advance();
  }
  if constexpr (Layout::kRing) load_part(IntTag<1>{}, lds + spare);
  // my part of the first K tile has landed
  __builtin_amdgcn_s_waitcnt(wait_vmcnt(Layout::kRing ? kAhead + kLoadsW : kLoadsW + kLoadsX));
  wg_barrier();
  Frags a, b;
#pragma unroll
  for (int i = 0; i < kReads; ++i) read(step_at(w_rows, w_part, Layout::kW, false), step_at(x_rows, x_part, Layout::kX, false), i, a);

  // One K step: SECOND of its K tile, FIRST K tile of its output tile (whose accumulators start at zero; `behind` says that the
  // STORES stores of the tile before are between the loads waited for and the youngest ones).
  auto k_step = [&](const Frags& now, Frags& next, auto second, auto first_kt, bool behind) __attribute__((always_inline)) {
    constexpr bool kSecond = decltype(second)::value != 0, kFirst = decltype(first_kt)::value != 0;
    char* to;
    if constexpr (kSecond) {
      // my part of K tile t + 1 has landed and my fragments of tile t are in registers
      if (kFirst && STORES > 0 && behind)
        __builtin_amdgcn_s_waitcnt(wait_vmcnt(kBehind) & kWaitLgkm0);
      else
        __builtin_amdgcn_s_waitcnt(wait_vmcnt(kAhead) & kWaitLgkm0);
      wg_barrier();
      to = lds + w_part;
      if constexpr (Layout::kRing) {
        spare = w_part;
        w_part = w_part + S::kStageBytes < Layout::kLds ? w_part + S::kStageBytes : 0;
        x_part = w_part + kWBytes;
      } else {
        spare = x_part;
        w_part = next_part(x_part);
        x_part = next_part(w_part);
      }
    } else {
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      to = lds + spare + (Layout::kRing ? kWBytes : 0);
    }
    const lds_bytes_t w = step_at(w_rows, w_part, Layout::kW, !kSecond), x = step_at(x_rows, x_part, Layout::kX, !kSecond);
    __builtin_amdgcn_sched_barrier(0);
    // the part that is loaded: weight rows under the first K step, token rows under the second, in a ring the other way round
    constexpr bool kLoadsWeight = kSecond == Layout::kRing;
    constexpr int kLoads = kLoadsWeight ? kLoadsW : kLoadsX;
    if constexpr (S::TN * S::TM == 64) for_blocks([&](auto row) __attribute__((always_inline)) {
      constexpr int jn = decltype(row)::value;
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        if constexpr (kFirst && !kSecond)
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        constexpr int kPerRow = kReads / 8, kApart = kPerRow == 2 ? 4 : kPerRow == 3 ? 3 : 2;
        if (jn < 7 ? jm % kApart == 0 : jm < kPerRow) read(w, x, kPerRow * jn + (jn < 7 ? jm / kApart : jm), next);
        if (jm == (kPerRow == 4 ? 3 : 2)) load(IntTag<kLoadsWeight>{}, row, to);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    else for_blocks([&](auto share) __attribute__((always_inline)) {
      // eight shares of the MFMAs, the reads evenly between all but the last few, the loads in the shares from the first on
      constexpr int kMfmas = S::TN * S::TM, q = decltype(share)::value;
#pragma unroll
      for (int i = q * kMfmas / 8; i < (q + 1) * kMfmas / 8; ++i) {
        const int jn = i / S::TM, jm = i % S::TM;
        if constexpr (kFirst && !kSecond)
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        constexpr int kSpan = kMfmas - 4;
#pragma unroll
        for (int r = 0; r < kReads; ++r)
          if (r * kSpan / kReads == i) read(w, x, r, next);
        if (i == q * kMfmas / 8 + (kMfmas >= 16 ? 1 : 0)) {
          if constexpr (q < kLoads) load(IntTag<kLoadsWeight>{}, share, to);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if constexpr (kSecond != Layout::kRing) advance();
  };
  bool behind = false;
  for (int tile = first; tile < total; tile += step) {
    k_step(a, b, IntTag<0>{}, IntTag<1>{}, behind);
    k_step(b, a, IntTag<1>{}, IntTag<1>{}, behind);
    for (int t = 1; t < nk; ++t) {
      keep();
      k_step(a, b, IntTag<0>{}, IntTag<0>{}, false);
      k_step(b, a, IntTag<1>{}, IntTag<0>{}, false);
    }
    // the compiler does not know these for MFMAs, whose results take a while
    constexpr int kTN = S::TN, kTM = S::TM, kBefore = kTM == 4 ? kTN - 2 : kTN - 1;  // the last five
    asm volatile("s_nop 15\n s_nop 15"
                 : "+a"(acc[kBefore][kTM == 4 ? 3 : kTM - 5]), "+a"(acc[kTN - 1][kTM - 4]), "+a"(acc[kTN - 1][kTM - 3]),
                   "+a"(acc[kTN - 1][kTM - 2]), "+a"(acc[kTN - 1][kTM - 1])
                 :
                 : "memory");
    behind = done(tile, acc, lds + spare);
    if constexpr (LONG) {
#pragma unroll
      for (int i = 0; i < kReads; ++i) read(step_at(w_rows, w_part, Layout::kW, false), step_at(x_rows, x_part, Layout::kX, false), i, a);
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitAll0);
}

}  // namespace rlk
