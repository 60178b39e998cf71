// GRPO ratio / k3-KL / clipped-surrogate epilogue on per-token log-probs.
//
// Restates compute_policy_ratio, compute_reference_kl and masked_mean
// (reference rl_engine/reference/definitions.py:50-106) and the surrogate of
// NativeGRPOLossOp.apply (rl_engine/reference/loss/grpo_loss.py:114-125, 162-168)
// with the fixed summation order the reference names SEQUENCE_MAJOR_FIXED
// (rl_engine/contracts/operators/loss.py:7-12): tokens are summed per sequence
// over the fixed padded length, then sequences are combined in ascending index.
//
// Per-sequence order: thread i of a 256-thread workgroup adds tokens
// i, i+256, i+512, ... ascending; the 256 partials are combined by a balanced
// binary tree over adjacent lanes (xor 1, 2, 4, ... 32), then the four waves in
// ascending order. Sequence partials are added ascending by one thread.
#include "rlk_host.h"

namespace rlk {

constexpr int kGrpoThreads = 256;
constexpr int kGrpoBackwardTokens = 1024;  // tokens of one sequence per workgroup of the backward

struct GrpoArgs {
  const float* logp;
  const float* old_logp;
  const float* ref_logp;
  const float* advantages;  // [rollouts]
  const uint8_t* mask;      // [rollouts * tokens] or null (all active)
  float* ratio;             // [rollouts * tokens] or null
  float* k3;                // [rollouts * tokens] or null
  float* seq_part;          // [3][rollouts]: policy sum, kl sum, active count
  int rollouts;
  int tokens;
  float clip_lo, clip_hi;
};

__device__ __forceinline__ float wave_tree_sum(float v) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) v = v + __shfl_xor(v, off, 64);
  return v;
}

__global__ __launch_bounds__(kGrpoThreads) void grpo_sequence_kernel(GrpoArgs a) {
  const int seq = blockIdx.x;
  const float adv = a.advantages[seq];
  const int64_t base = (int64_t)seq * a.tokens;
  float pol = 0.f, kl = 0.f, cnt = 0.f;
  // Four tokens of a thread are loaded before the first of them is used (a sequence has one workgroup, so what bounds
  // it is the latency of its loads: 8 sequences of 8192 tokens 27.4 -> 16.3 us, 64 of 1024 within 0.6 us); they are added in ascending order as before.
  constexpr int kAhead = 4;
  for (int t0 = threadIdx.x; t0 < a.tokens; t0 += kAhead * kGrpoThreads) {
    float lp[kAhead], old_lp[kAhead], ref_lp[kAhead];
    bool act[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int t = t0 + i * kGrpoThreads;
      if (t < a.tokens) {
        lp[i] = a.logp[base + t];
        old_lp[i] = a.old_logp[base + t];
        ref_lp[i] = a.ref_logp[base + t];
        act[i] = a.mask ? (a.mask[base + t] != 0) : true;
      }
    }
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int t = t0 + i * kGrpoThreads;
      if (t >= a.tokens) break;
      const bool active = act[i];
      float r = expf(lp[i] - old_lp[i]);
      const float d = ref_lp[i] - lp[i];
      float k = expf(d) - d - 1.0f;
      r = active ? r : 0.f;
      k = active ? k : 0.f;
      const float adv_t = active ? adv : 0.f;
      const float unclipped = r * adv_t;
      const float clipped = fminf(fmaxf(r, a.clip_lo), a.clip_hi) * adv_t;
      float term = -fminf(unclipped, clipped);
      term = active ? term : 0.f;
      if (a.ratio) a.ratio[base + t] = r;
      if (a.k3) a.k3[base + t] = k;
      pol = pol + term;
      kl = kl + k;
      cnt = cnt + (active ? 1.f : 0.f);
    }
  }
  pol = wave_tree_sum(pol);
  kl = wave_tree_sum(kl);
  cnt = wave_tree_sum(cnt);
  __shared__ float sh[3][kGrpoThreads / 64];
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sh[0][wave] = pol;
    sh[1][wave] = kl;
    sh[2][wave] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    float p = sh[0][0], k = sh[1][0], c = sh[2][0];
    for (int w = 1; w < kGrpoThreads / 64; ++w) {
      p = p + sh[0][w];
      k = k + sh[1][w];
      c = c + sh[2][w];
    }
    a.seq_part[seq] = p;
    a.seq_part[a.rollouts + seq] = k;
    a.seq_part[2 * a.rollouts + seq] = c;
  }
}

// The three sums over sequences, ascending, by one thread each: the partials come in through LDS, 256 sequences at a
// time (a single thread that reads them from memory itself waits for every one of them: 64 sequences 4.5 -> 2.1 us,
// 512 sequences 32.4 -> 5.0 us).
__global__ __launch_bounds__(kGrpoThreads) void grpo_finish_kernel(const float* __restrict__ seq_part, int rollouts,
                                                                   float beta, float* __restrict__ out3) {
  __shared__ float part[3][kGrpoThreads];
  __shared__ float total[3];
  const int tid = threadIdx.x;
  float sum = 0.f;
  for (int s0 = 0; s0 < rollouts; s0 += kGrpoThreads) {
    const int n = rollouts - s0 < kGrpoThreads ? rollouts - s0 : kGrpoThreads;
    if (tid < n) {
#pragma unroll
      for (int i = 0; i < 3; ++i) part[i][tid] = seq_part[(int64_t)i * rollouts + s0 + tid];
    }
    __syncthreads();
    if (tid < 3)
      for (int s = 0; s < n; ++s) sum = sum + part[tid][s];
    __syncthreads();
  }
  if (tid < 3) total[tid] = sum;
  __syncthreads();
  if (tid != 0) return;
  const float denom = fmaxf(total[2], 1e-8f);
  const float policy = total[0] / denom;
  const float klm = total[1] / denom;
  out3[0] = policy + beta * klm;
  out3[1] = policy;
  out3[2] = klm;
}

// d(out3 . weights) / d(logp), one pass: with r = exp(logp - old), d = ref - logp,
//   d policy / d logp = -A r where the unclipped branch is the minimum or ties it, else 0;  d k3 / d logp = 1 - exp(d)
// times the incoming weights, the mask and 1 / active. As elementwise tensor operations this was 36 launches, and the
// host's time for them bounded the loss (64 x 1024 tokens forward and backward 258 -> 120 us); the kernel takes 5.2 us
// there, 8.3 us at 512 x 2048 (17 bytes per token, 2.1 TB/s). The expressions and their order are those
// of the elementwise form, so the gradient keeps its bits.
__global__ __launch_bounds__(kGrpoThreads) void grpo_backward_kernel(GrpoArgs a, const float* __restrict__ g_loss,
                                                                     const float* __restrict__ g_policy,
                                                                     const float* __restrict__ g_kl, float beta,
                                                                     float* __restrict__ grad, int chunks) {
  const int seq = blockIdx.x / chunks;
  const int t0 = (blockIdx.x - seq * chunks) * kGrpoBackwardTokens + threadIdx.x;
  const float gl = g_loss ? *g_loss : 0.f;
  const float w_policy = gl + (g_policy ? *g_policy : 0.f);
  const float w_kl = beta * gl + (g_kl ? *g_kl : 0.f);
  const float adv = a.advantages[seq];
  // the active tokens of all sequences, from the forward's counts: whole numbers, so the order does not matter
  float cnt = 0.f;
  for (int s = threadIdx.x; s < a.rollouts; s += kGrpoThreads) cnt = cnt + a.seq_part[(int64_t)2 * a.rollouts + s];
  cnt = wave_tree_sum(cnt);
  __shared__ float wave_count[kGrpoThreads / 64];
  if ((threadIdx.x & 63) == 0) wave_count[threadIdx.x >> 6] = cnt;
  __syncthreads();
  const float active = fmaxf((wave_count[0] + wave_count[1]) + (wave_count[2] + wave_count[3]), 1e-8f);
  const int64_t base = (int64_t)seq * a.tokens;
#pragma unroll
  for (int i = 0; i < kGrpoBackwardTokens / kGrpoThreads; ++i) {
    const int t = t0 + i * kGrpoThreads;
    if (t < a.tokens) {
      const float keep = a.mask ? (a.mask[base + t] != 0 ? 1.f : 0.f) : 1.f;
      const float lp = a.logp[base + t];
      const float r = expf(lp - a.old_logp[base + t]);
      const bool flows = (r >= a.clip_lo && r <= a.clip_hi) || (r > a.clip_hi && adv < 0.f) || (r < a.clip_lo && adv > 0.f);
      const float d_policy = -(adv * r) * (flows ? 1.f : 0.f);
      const float d_kl = 1.0f - expf(a.ref_logp[base + t] - lp);
      grad[base + t] = (w_policy * d_policy + w_kl * d_kl) * keep / active;
    }
  }
}

hipError_t grpo_launch(const float* logp, const float* old_logp, const float* ref_logp, const float* advantages,
                       const uint8_t* mask, int rollouts, int tokens, float clip_eps, float beta, float* ratio,
                       float* k3, float* out3, float* workspace, hipStream_t stream) {
  GrpoArgs a;
  a.logp = logp;
  a.old_logp = old_logp;
  a.ref_logp = ref_logp;
  a.advantages = advantages;
  a.mask = mask;
  a.ratio = ratio;
  a.k3 = k3;
  a.seq_part = workspace;
  a.rollouts = rollouts;
  a.tokens = tokens;
  a.clip_lo = 1.0f - clip_eps;
  a.clip_hi = 1.0f + clip_eps;
  if (rollouts > 0) {
    hipLaunchKernelGGL(grpo_sequence_kernel, dim3(rollouts), dim3(kGrpoThreads), 0, stream, a);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  hipLaunchKernelGGL(grpo_finish_kernel, dim3(1), dim3(kGrpoThreads), 0, stream, workspace, rollouts, beta, out3);
  return hipGetLastError();
}

hipError_t grpo_backward_launch(const float* logp, const float* old_logp, const float* ref_logp, const float* advantages,
                                const uint8_t* mask, float* workspace, const float* g_loss, const float* g_policy,
                                const float* g_kl, int rollouts, int tokens, float clip_lo, float clip_hi, float beta,
                                float* grad, hipStream_t stream) {
  if (rollouts <= 0 || tokens <= 0) return hipSuccess;
  GrpoArgs a = {};
  a.logp = logp;
  a.old_logp = old_logp;
  a.ref_logp = ref_logp;
  a.advantages = advantages;
  a.mask = mask;
  a.seq_part = workspace;
  a.rollouts = rollouts;
  a.tokens = tokens;
  a.clip_lo = clip_lo;
  a.clip_hi = clip_hi;
  const int chunks = (tokens + kGrpoBackwardTokens - 1) / kGrpoBackwardTokens;
  if ((int64_t)rollouts * chunks > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(grpo_backward_kernel, dim3(rollouts * chunks), dim3(kGrpoThreads), 0, stream, a, g_loss,
                     g_policy, g_kl, beta, grad, chunks);
  return hipGetLastError();
}

}  // namespace rlk
