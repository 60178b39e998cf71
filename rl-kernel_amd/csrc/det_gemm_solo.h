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
// Same MFMA chain per output element as every other loop. Needs the native layouts, 16-byte aligned rows, K % 64 == 0 and
// rows whose byte offsets inside a tile stay below 4 GiB (solo_offsets_fit()).
#pragma once

#include "det_gemm_tile.h"

namespace rlk {

using SoloShape = TileShape<256, 256, 2, 2>;
constexpr int kSoloPartBytes = 256 * kRowBytes;
constexpr int kSoloParts = 5;
constexpr int kSoloLdsBytes = kSoloParts * kSoloPartBytes;
constexpr int kSoloLoads = 8;  // load instructions of a wave per part

// `rows`: from the first row of a tile to its last.
inline bool solo_offsets_fit(const MatView& v, int64_t rows = SoloShape::BN) {
  return v.row_stride >= 0 && v.row_stride < ((int64_t)1 << 31) && rows * v.row_stride * 2 + 8192 < ((int64_t)1 << 32);
}

// Which weight row, counted from the first one of the tile's features, LDS row r of the weight part holds.
// Plain: a wave's 128 features are two spans of 64, and in each of them a lane owns 16 consecutive ones, as with the four MFMA
// tiles of a 64-feature wave column (weight_row_of_lds_row):
//   acc[4 h + jn][jm][q] is feature 128 wave_n + 64 h + 16 (lane >> 4) + 4 jn + q of token 128 wave_m + 16 jm + (lane & 15).
// Gated: 128 features of both halves of a packed gate/up weight [2 I, K],
//   acc[jn][jm][q] the gate and acc[4 + jn][jm][q] the up projection of feature 64 wave_n + 16 (lane >> 4) + 4 jn + q.
struct SoloPlainRows {
  static __device__ __forceinline__ int feature(int r) { return (r & ~63) + ((r & 15) >> 2) * 16 + ((r >> 4) & 3) * 4 + (r & 3); }
  static __device__ __forceinline__ int64_t row(int r, int last, int) { return min(feature(r), last); }
  static __device__ __forceinline__ int features(const MatView& W) { return W.rows; }
};
struct SoloGatedRows {
  static __device__ __forceinline__ int64_t row(int r, int last, int half_rows) {
    const int f = (r >> 7) * 64 + ((r & 15) >> 2) * 16 + ((r >> 4) & 3) * 4 + (r & 3);
    return min(f, last) + ((r >> 6) & 1) * half_rows;
  }
  static __device__ __forceinline__ int features(const MatView& W) { return W.rows / 2; }
};

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

// One result out of its accumulator register, where it is wanted: the compiler brings all of them into others first, which in a long
// epilogue it does not have.
__device__ __forceinline__ float solo_result(float accumulator) {
  float value;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(value) : "a"(accumulator));
  return value;
}

typedef f32x4_t SoloAcc[SoloShape::TN][SoloShape::TM];

// Runs the tiles first, first + step, ... < total (at least one). tile_at(i, n0, m0) says where tile i lies; done(i, acc, scratch)
// takes its results, may use the spare part of the LDS if it ends on a barrier then, and returns whether this wave has issued STORES
// vector memory instructions, no fewer: so many more may then be in flight at the first wait of the next tile. LONG: done() wants
// the registers of the next tile's first fragments, which are read again behind it. keep() runs once per K tile: an empty asm with the
// values that done() carries from tile to tile as its operands keeps them in registers.
struct SoloKeepsNothing {
  __device__ __forceinline__ void operator()() const {}
};
template <class Rows, int STORES, bool LONG = false, class TileAt, class Done, class Keep = SoloKeepsNothing>
__device__ __forceinline__ void solo_tiles(const MatView& W, const MatView& X, int K, int first, int step, int total, char* lds,
                                           TileAt tile_at, Done done, Keep keep = Keep()) {
  using S = SoloShape;
  constexpr int kBehind = STORES + kSoloLoads < 63 ? STORES + kSoloLoads : 63;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int grp = lane >> 4;
  const int nk = K / kTileK;

  // The load stream: the next K tile of its output tile, at w_at and x_at. A wave loads LDS rows [64 wave, + 64) of either part in eight
  // blocks of eight rows; block j adds (j & 3) KiB as the instruction's offset, which counts for the LDS address and the global one.
  constexpr int kBlockBytes = 1024, kBlocksPerBase = 4;
  uint32_t off_w[kSoloLoads], off_x[kSoloLoads];
  const char *w_at, *x_at;
  int load_tile = first, load_left = nk;
  auto aim = [&]() __attribute__((always_inline)) {
    int n0, m0;
    tile_at(load_tile, n0, m0);
    w_at = reinterpret_cast<const char*>(W.ptr + (int64_t)n0 * W.row_stride) - kBlocksPerBase * kBlockBytes;
    x_at = reinterpret_cast<const char*>(X.ptr + (int64_t)m0 * X.row_stride) - kBlocksPerBase * kBlockBytes;
    const int lane = solo_lane();
#pragma unroll
    for (int j = 0; j < kSoloLoads; ++j) {
      const int r = wave * 64 + j * 8 + (lane >> 3);
      // rows past the edge: computed, never stored
      const uint32_t row_w = (uint32_t)Rows::row(r, Rows::features(W) - n0 - 1, W.rows / 2), row_x = min(r, X.rows - m0 - 1);
      const uint32_t in_row = ((lane & 7) ^ (lane >> 3)) * 16 + (kBlocksPerBase - j % kBlocksPerBase) * kBlockBytes;
      off_w[j] = row_w * (uint32_t)W.row_stride * 2 + in_row;
      off_x[j] = row_x * (uint32_t)X.row_stride * 2 + in_row;
      asm volatile("" : "+v"(off_w[j]), "+v"(off_x[j]));  // 32 bits each: as halves of 64-bit products they took two registers
    }
  };
  aim();
  auto advance = [&]() __attribute__((always_inline)) {
    w_at += kRowBytes;
    x_at += kRowBytes;
    if (--load_left > 0) return;
    load_left = nk;
    load_tile = load_tile + step < total ? load_tile + step : load_tile;  // past the last tile: its first K tiles again, never read
    aim();
  };
  auto load = [&](auto weight, auto block, char* part) __attribute__((always_inline)) {
    constexpr int j = decltype(block)::value;
    constexpr bool kWeight = decltype(weight)::value != 0;
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kWeight ? w_at : x_at), 0, 0xffffffff, 0x00027000);
    lds_ptr_t to = (lds_ptr_t)(part + (wave * kSoloLoads + j / kBlocksPerBase * kBlocksPerBase) * kBlockBytes);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, to, 16, kWeight ? off_w[j] : off_x[j], 0, j % kBlocksPerBase * kBlockBytes, 0);
  };
  auto for_blocks = [](auto f) __attribute__((always_inline)) {
    f(IntTag<0>{}), f(IntTag<1>{}), f(IntTag<2>{}), f(IntTag<3>{}), f(IntTag<4>{}), f(IntTag<5>{}), f(IntTag<6>{}), f(IntTag<7>{});
  };

  SoloAcc acc;
  struct Frags {
    u32x4_t w[S::TN], x[S::TM];
  };
  const int frag = (grp ^ (l16 & 7)) << 4;  // of the first K step of a K tile; the second one flips bit 6
  typedef const __attribute__((address_space(3))) char* lds_bytes_t;  // 32 bits whatever the compiler knows of `lds`
  typedef const __attribute__((address_space(3))) u32x4_t* lds_chunk_t;
  const lds_bytes_t w_rows = (lds_bytes_t)lds + ((wave % S::WN) * 128 + l16) * kRowBytes;
  const lds_bytes_t x_rows = (lds_bytes_t)lds + ((wave / S::WN) * 128 + l16) * kRowBytes;
  auto read = [&](lds_bytes_t w, lds_bytes_t x, int i, Frags& f) __attribute__((always_inline)) {  // in the order of their use
    if (i == 0) f.w[0] = *(lds_chunk_t)w;
    else if (i <= S::TM) f.x[i - 1] = *(lds_chunk_t)(x + (i - 1) * 16 * kRowBytes);
    else f.w[i - S::TM] = *(lds_chunk_t)(w + (i - S::TM) * 16 * kRowBytes);
  };

  auto next_part = [](int at) { return at + kSoloPartBytes < kSoloLdsBytes ? at + kSoloPartBytes : 0; };
  int w_part = 0, x_part = kSoloPartBytes, spare = 4 * kSoloPartBytes;  // of the K tile at hand
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    for_blocks([&](auto j) __attribute__((always_inline)) { load(IntTag<1>{}, j, lds + 2 * t * kSoloPartBytes); });
    for_blocks([&](auto j) __attribute__((always_inline)) { load(IntTag<0>{}, j, lds + (2 * t + 1) * kSoloPartBytes); });
    advance();
  }
  __builtin_amdgcn_s_waitcnt(wait_vmcnt(2 * kSoloLoads));  // my part of the first K tile has landed
  wg_barrier();
  Frags a, b;
#pragma unroll
  for (int i = 0; i < S::TN + S::TM; ++i) read(w_rows + w_part + frag, x_rows + x_part + frag, i, a);

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
        __builtin_amdgcn_s_waitcnt(wait_vmcnt(kSoloLoads) & kWaitLgkm0);
      wg_barrier();
      to = lds + w_part;
      spare = x_part;
      w_part = next_part(x_part);
      x_part = next_part(w_part);
    } else {
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      to = lds + spare;
    }
    const lds_bytes_t w = w_rows + w_part + (kSecond ? frag : frag ^ 64);
    const lds_bytes_t x = x_rows + x_part + (kSecond ? frag : frag ^ 64);
    __builtin_amdgcn_sched_barrier(0);
    for_blocks([&](auto row) __attribute__((always_inline)) {
      constexpr int jn = decltype(row)::value;
#pragma unroll
      for (int jm = 0; jm < S::TM; ++jm) {
        if constexpr (kFirst && !kSecond)
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[jn][jm]) : "v"(now.w[jn]), "v"(now.x[jm]));
        if (jm % 4 == 0 && jn < 7) read(w, x, 2 * jn + jm / 4, next);
        if (jm < 2 && jn == 7) read(w, x, 14 + jm, next);
        if (jm == 2) load(IntTag<kSecond ? 0 : 1>{}, row, to);
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    if constexpr (kSecond) advance();
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
    asm volatile("s_nop 15\n s_nop 15"
                 : "+a"(acc[7][3]), "+a"(acc[7][4]), "+a"(acc[7][5]), "+a"(acc[7][6]), "+a"(acc[7][7])
                 :
                 : "memory");
    behind = done(tile, acc, lds + spare);
    if constexpr (LONG) {
#pragma unroll
      for (int i = 0; i < S::TN + S::TM; ++i) read(w_rows + w_part + frag, x_rows + x_part + frag, i, a);
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitAll0);
}

}  // namespace rlk
