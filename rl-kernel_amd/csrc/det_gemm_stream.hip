// det_gemm for up to 64 tokens against few, long weight panels: one workgroup streams a
// 16-feature weight panel through a deep LDS ring while one wave per 16-token tile runs the
// MFMA chain.
//
// With M <= 64 the GEMM is a read of W at HBM speed. The contract allows no split-K, so the
// K/32 MFMA steps of an output element run one after the other in one wave, and a 16-row
// panel is the finest unit of work (N / 16 workgroups: 256 for the Qwen3-8B down projection,
// one per CU). To keep enough bytes in flight with one workgroup per CU, four producer waves
// issue direct-to-LDS loads several stages ahead; the consumer waves only read fragments and
// issue the dependent MFMA chain, which is short (K/32 steps of ~21 cycles). Measured on this
// part: L2 hits feed a CU's direct-to-LDS path at 64 bytes per clock (135 GB/s, two issuing
// waves suffice), data that comes through the fabric (infinity cache / HBM) arrives at about
// 6 TB/s chip-wide, i.e. 23 GB/s per CU: the weight panel is the slow stream, the activations
// (re-read by every workgroup, L2 hits) the wide one. Same instruction, same ascending K order,
// same zero start as every other det_gemm kernel, so the bits match.
#include "linear_logp_common.h"
#include "rlk_host.h"

namespace rlk {

// MT token tiles of 16 rows. Wave t < MT is the consumer of token tile t (its own MFMA chain
// over the shared weight fragments), the next four waves are the producers. A stage holds KT
// weight sub-tiles (64 K values each), then KT sub-tiles per token tile; a producer always
// fetches the same 8-row half (producer & 1) of the (tile, sub-tile) pairs
// (producer >> 1) + 2 j. Rows past M or N are clamped to the last valid row: computed, never
// stored (MFMA columns and rows are independent).
//
// GATED: W is a packed gate/up weight [2 I, K] (N = 2 I). The panel of workgroup b holds the gate
// rows of features 8 b .. 8 b + 7 in its first half and their up rows in the second, so gate and
// up of an output element sit 32 lanes apart in one accumulator; the epilogue brings them
// together, rounds both to bf16 as the unfused projection would, and stores swiglu(gate, up) into
// C[M, I] (bf16).
// WSTREAM: the weight is read past the caches (streamed_weight() in rlk_host.h).
template <int KT, int RING, int MT, bool OUT_F32, bool GATED = false, bool WSTREAM = false>
__global__ __launch_bounds__(64 * (MT + 4)) void det_gemm_stream_kernel(MatView W, MatView X,
                                                                              void* __restrict__ C, int64_t ldc, int M,
                                                                              int N, int K) {
  static_assert(!(GATED && OUT_F32), "the gated projection stores bf16");
  constexpr int kSubBytes = 16 * kRowBytes;
  constexpr int kPairs = KT * (1 + MT);
  constexpr int kStageBytes = kPairs * kSubBytes;
  constexpr int kLoads = kPairs / 2;  // per producer wave per stage
  static_assert(RING >= 2 && kPairs % 2 == 0 && KT % 2 == 0 && MT >= 1 && MT <= 4, "ring geometry");
  constexpr int kWLoads = KT / 2;  // the first of a producer's loads of a stage are its weight halves
  extern __shared__ __attribute__((aligned(16))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // [0, MT): consumers, then 4 producers
  const int producer = wave - MT;
  const int n0 = blockIdx.x * (GATED ? 8 : 16);  // GATED: first feature of the workgroup
  const int nsub = K / kTileK;  // K % 64 == 0 on this path
  const int nstage = (nsub + KT - 1) / KT;

  // Producer: this lane's row inside a 16-row tile and its 16-byte chunk.
  const int rib = lane >> 3;
  const int chunk_elems = ((lane & 7) ^ rib) * kChunkElems;
  const int half = producer & 1;
  const int r16 = half * 8 + rib;
  int wr = n0 + r16 < N ? n0 + r16 : N - 1;  // rows past an edge are computed, never stored
  if constexpr (GATED) {
    const int features = N / 2;
    const int f = n0 + rib < features ? n0 + rib : features - 1;
    wr = half * features + f;  // producers with half == 0 fetch gate rows, the others up rows
  }
  const bf16_bits* w_base = W.ptr + (int64_t)wr * W.row_stride + chunk_elems;
  const bf16_bits* x_base[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int xr = t * 16 + r16 < M ? t * 16 + r16 : M - 1;
    x_base[t] = X.ptr + (int64_t)xr * X.row_stride + chunk_elems;
  }

  // Load j of this producer for a stage: its half of the pair (producer >> 1) + 2 j.
  auto load = [&](int j, const bf16_bits* src, int slot) {
    const lds_ptr_t dst = (lds_ptr_t)(lds + slot + (2 * ((producer >> 1) + 2 * j) + half) * 1024);
    if (WSTREAM && j < kWLoads)
      __builtin_amdgcn_global_load_lds((global_ptr_t)src, dst, 16, 0, kLoadNonTemporal);
    else
      __builtin_amdgcn_global_load_lds((global_ptr_t)src, dst, 16, 0, 0);
  };
  auto next_slot = [](int slot) { return slot == (RING - 1) * kStageBytes ? 0 : slot + kStageBytes; };
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  const int l16 = lane & 15;
  const int grp = lane >> 4;
  const int frag_lo = l16 * kRowBytes + ((grp ^ (l16 & 7)) << 4);  // K step 0 of a sub-tile
  const int frag_hi = frag_lo ^ 64;                                 // K step 1

  // Both kinds of waves meet at one barrier per stage and do little else there. With the stage's fragments read in front of
  // their MFMAs, and the refills' clamps and addresses in every stage, one took 0.18 us, which is what bounds panels that HBM
  // does not; now about 0.1. Weights from HBM, us, K -> outputs: 4096 -> 1536 at one token 7.8 -> 5.2, 6144 -> 2048 10.7 -> 8.3,
  // 1024 -> 4096 4.5 -> 4.0, 4096 -> 6144 13.0 -> 12.2, 4096 -> 24576 at 1 / 16 tokens 35.7 / 40.8 -> 33.8 / 38.0.
  if (wave >= MT) {
    // Stage t, of which the sub-tiles behind the reduction's end fetch the last one again (never consumed). Behind the last
    // stage one lane of each load goes on, for the counts that the wait relies on (whole loads there took the CU's load path
    // from its next workgroup: 4096 -> 24576 at 16 tokens 39.7 us, with one lane 38.0; no loads and a wait by the number of
    // stages left cost more in the short panels).
    auto issue_last = [&](int t, int slot) {
      if (t >= nstage && lane != 0) return;
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        const int q = (producer >> 1) + 2 * j;  // pair: [0, KT) weights, then KT per token tile
        const int ks = t * KT + q % KT;
        load(j, (j < kWLoads ? w_base : x_base[(2 * j - KT) / KT]) + (ks < nsub ? ks : nsub - 1) * kTileK, slot);
      }
    };
    auto step = [&] {
      __builtin_amdgcn_s_waitcnt(wait_vmcnt((RING - 2) * kLoads));  // my loads of stage s have landed
      wg_barrier();  // stage s is complete; the consumers hold the fragments of stage s - 1
    };
    int64_t k = (producer >> 1) * kTileK;
    int slot = 0;
    auto issue_whole = [&] {  // the next stage, all of it inside the reduction
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        load(j, (j < kWLoads ? w_base : x_base[(2 * j - KT) / KT]) + k + 2 * j % KT * kTileK, slot);
      k += KT * kTileK;
      slot = next_slot(slot);
    };
    const int whole = nsub / KT - (RING - 1);  // stages of the loop whose refill is a whole one
    if (whole >= 0) {
#pragma unroll
      for (int t = 0; t < RING - 1; ++t) issue_whole();
    } else {
#pragma nounroll
      for (int t = 0; t < RING - 1; ++t) {
        issue_last(t, slot);
        slot = next_slot(slot);
      }
    }
    int s = 0;
    for (; s < whole; ++s) {
      step();
      issue_whole();
    }
    for (; s < nstage; ++s) {
      step();
      issue_last(s + RING - 1, slot);
      slot = next_slot(slot);
    }
  } else {
    // The fragments of stage s are read under the MFMAs of stage s - 1.
    struct Fragments {
      u32x4_t w[2 * KT], x[2 * KT];
    };
    auto multiply = [&](const Fragments& f, int steps) {
#pragma unroll
      for (int i = 0; i < 2 * KT; ++i)
        if (i < steps) acc = mfma_16x16x32(f.w[i], f.x[i], acc);
    };
    int slot = 0;
    auto stage = [&](Fragments& next, const Fragments& now) {
      wg_barrier();
      const char* base = lds + slot;
#pragma unroll
      for (int sub = 0; sub < KT; ++sub) {
        const char* wt = base + sub * kSubBytes;
        const char* xt = base + (KT + wave * KT + sub) * kSubBytes;
        next.w[2 * sub] = *reinterpret_cast<const u32x4_t*>(wt + frag_lo);
        next.x[2 * sub] = *reinterpret_cast<const u32x4_t*>(xt + frag_lo);
        next.w[2 * sub + 1] = *reinterpret_cast<const u32x4_t*>(wt + frag_hi);
        next.x[2 * sub + 1] = *reinterpret_cast<const u32x4_t*>(xt + frag_hi);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(now, 2 * KT);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
      slot = next_slot(slot);
    };
    Fragments even, odd = {};  // (the first stage multiplies zeros: the accumulator stays +0)
    int s = 0;
    for (; s + 1 < nstage; s += 2) {
      stage(even, odd);
      stage(odd, even);
    }
    const int last_steps = 2 * (nsub - (nstage - 1) * KT);
    if (s < nstage) {
      stage(even, odd);
      multiply(even, last_steps);
    } else {
      multiply(odd, last_steps);
    }
  }
  __builtin_amdgcn_s_waitcnt(kWaitAll0);
  wg_barrier();

  const int m = wave * 16 + l16;
  if constexpr (GATED) {
    if (wave < MT) {
      // accumulator rows 4 grp + q: lane groups 0, 1 hold gate features n0 + 4 grp + q, groups 2, 3
      // the up projection of features n0 + 4 (grp - 2) + q
      float up[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        up[q] = __int_as_float(__builtin_amdgcn_ds_bpermute((lane ^ 32) << 2, __float_as_int(acc[q])));
      const int f = n0 + grp * 4;
      if (grp < 2 && m < M) {
        bf16_bits* row = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc;
        uint32_t packed[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
          packed[h] = pack_bf16x2(swiglu_f32(round_through_bf16(acc[2 * h]), round_through_bf16(up[2 * h])),
                                  swiglu_f32(round_through_bf16(acc[2 * h + 1]), round_through_bf16(up[2 * h + 1])));
        if (f + 4 <= N / 2 && (reinterpret_cast<uintptr_t>(row + f) & 7) == 0) {
          *reinterpret_cast<u32x2_t*>(row + f) = u32x2_t{packed[0], packed[1]};
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (f + q < N / 2) row[f + q] = (bf16_bits)((packed[q >> 1] >> ((q & 1) * 16)) & 0xffffu);
        }
      }
    }
    return;
  }
  if (wave < MT && m < M) {
    const int n = n0 + grp * 4;
    if (OUT_F32) {
      float* row = reinterpret_cast<float*>(C) + (int64_t)m * ldc;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < N) row[n + q] = acc[q];
    } else {
      bf16_bits* row = reinterpret_cast<bf16_bits*>(C) + (int64_t)m * ldc;
      const uint32_t lo = pack_bf16x2(acc[0], acc[1]);
      const uint32_t hi = pack_bf16x2(acc[2], acc[3]);
      if (n + 4 <= N && (reinterpret_cast<uintptr_t>(row + n) & 7) == 0) {
        *reinterpret_cast<u32x2_t*>(row + n) = u32x2_t{lo, hi};
      } else {
        const uint32_t packed[2] = {lo, hi};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < N) row[n + q] = (bf16_bits)((packed[q >> 1] >> ((q & 1) * 16)) & 0xffffu);
      }
    }
  }
}

template <int KT, int RING, int MT, bool OUT_F32, bool WSTREAM = false>
static hipError_t launch_stream(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                                      hipStream_t stream) {
  // Two to four token tiles gain nothing (down at 32 / 64 tokens 26.0 / 36.6 us either way: the activations, four times
  // the weight's loads there, set the pace).
  if constexpr (MT == 1 && !OUT_F32 && !WSTREAM) {
    if (streamed_weight(N, K, M, 16)) return launch_stream<KT, RING, MT, OUT_F32, true>(W, X, C, ldc, M, N, K, stream);
  }
  auto kernel = det_gemm_stream_kernel<KT, RING, MT, OUT_F32, false, WSTREAM>;
  constexpr int kLds = RING * KT * (1 + MT) * 16 * kRowBytes;
  static_assert(kLds <= 160 * 1024, "ring exceeds the LDS");
  static PerDeviceOnce once;
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((N + 15) / 16), dim3(64 * (MT + 4)), kLds, stream, W, X, C, ldc, M, N, K);
  return hipGetLastError();
}

// Packed gate/up projection with the SwiGLU epilogue for up to 16 tokens (W.rows = 2 I, Y[M, I]):
// the two-workgroups-per-CU geometry, I / 8 workgroups.
hipError_t det_gemm_stream_gated_launch(const MatView& W, const MatView& X, void* Y, int64_t ldy, int M, int I, int K,
                                        hipStream_t stream) {
  const bool streamed = streamed_weight(2 * (int64_t)I, K, M, 16);
  auto kernel = streamed ? det_gemm_stream_kernel<2, 8, 1, false, true, true> : det_gemm_stream_kernel<2, 8, 1, false, true>;
  constexpr int kLds = 8 * 2 * 2 * 16 * kRowBytes;
  static PerDeviceOnce once[2];
  hipError_t err = allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLds, once[streamed]);
  if (err != hipSuccess) return err;
  hipLaunchKernelGGL(kernel, dim3((I + 7) / 8), dim3(64 * 5), kLds, stream, W, X, Y, ldy, M, 2 * I, K);
  return hipGetLastError();
}

// One to four token tiles; the ring takes 128 - 144 KiB (one workgroup per CU). `shallow`
// (M <= 16 only) halves the stage so that two workgroups share a CU.
hipError_t det_gemm_stream_launch(const MatView& W, const MatView& X, void* C, int64_t ldc, int M, int N, int K,
                                  bool out_f32, bool shallow, hipStream_t stream) {
  if (M <= 16 && shallow)
    return out_f32 ? launch_stream<2, 8, 1, true>(W, X, C, ldc, M, N, K, stream)
                   : launch_stream<2, 8, 1, false>(W, X, C, ldc, M, N, K, stream);
  if (M <= 16)
    return out_f32 ? launch_stream<4, 8, 1, true>(W, X, C, ldc, M, N, K, stream)
                   : launch_stream<4, 8, 1, false>(W, X, C, ldc, M, N, K, stream);
  if (M <= 32)
    return out_f32 ? launch_stream<4, 6, 2, true>(W, X, C, ldc, M, N, K, stream)
                   : launch_stream<4, 6, 2, false>(W, X, C, ldc, M, N, K, stream);
  if (M <= 48)
    return out_f32 ? launch_stream<2, 9, 3, true>(W, X, C, ldc, M, N, K, stream)
                   : launch_stream<2, 9, 3, false>(W, X, C, ldc, M, N, K, stream);
  return out_f32 ? launch_stream<2, 7, 4, true>(W, X, C, ldc, M, N, K, stream)
                 : launch_stream<2, 7, 4, false>(W, X, C, ldc, M, N, K, stream);
}

}  // namespace rlk
