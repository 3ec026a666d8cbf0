// GSPO scoring: per-token log-probabilities of the sampled tokens, the sequence-level importance ratio,
// the clipped objective and its gradient with respect to the logits, plus group-normalised advantages.
//
// Semantics: scripts/gspo.py:340-353 (token_logprobs: log_softmax over the fp32 logits, gathered at the
// PAD-clamped targets) and scripts/gspo.py:446-477 (advantages; s = exp(sum of masked (lp - old) /
// n_bases); pg = -min(s A, clamp(s, 1 - eps, 1 + eps) A); loss = sum(pg) / N). The gradient is the
// closed form of autograd through those ops:
//   dL/dz[b,t,v] = (1/N) g_b s_b mask[b,t] / n_bases[b] (onehot(y)[v] - softmax(z[b,t])[v]),
//   g_b = d pg_b / d s_b, with torch.minimum splitting ties evenly and clamp passing its gradient on
//   the closed interval.
// Every reduction runs in a fixed order, so results are bitwise reproducible.
#include <math.h>

#include "common.h"

namespace vk {

constexpr int GS_THREADS = 256;

template <bool BF16>
__device__ __forceinline__ float logit_at(const void *p, int64_t i) {
  if (BF16) return bf2f(static_cast<const bf16_t *>(p)[i]);
  return static_cast<const float *>(p)[i];
}

// log-sum-exp and max of one token's logits, computed by one thread
template <bool BF16>
__device__ __forceinline__ void lse_thread(const void *lg, int64_t base, int V, float &mx, float &lse) {
  mx = -INFINITY;
  for (int v = 0; v < V; ++v) mx = fmaxf(mx, logit_at<BF16>(lg, base + v));
  float s = 0.f;
  for (int v = 0; v < V; ++v) s += expf(logit_at<BF16>(lg, base + v) - mx);
  lse = mx + logf(s);
}

// ... by one wavefront (every lane gets the result)
template <bool BF16>
__device__ __forceinline__ void lse_wave(const void *lg, int64_t base, int V, int lane, float &mx, float &lse) {
  mx = -INFINITY;
  for (int v = lane; v < V; v += 64) mx = fmaxf(mx, logit_at<BF16>(lg, base + v));
  mx = wave_max(mx);
  float s = 0.f;
  for (int v = lane; v < V; v += 64) s += expf(logit_at<BF16>(lg, base + v) - mx);
  s = wave_sum(s);
  lse = mx + logf(s);
}

__device__ __forceinline__ float block_sum(float v, float *scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float t = 0.f;
  for (int w = 0; w < GS_THREADS / 64; ++w) t += scratch[w];
  return t;
}

// From a sequence's ratio: its objective, and (returned) the factor of its logits' gradient.
__device__ __forceinline__ float ratio_terms(float s, float nb, float A, float eps_lo, float eps_hi, float inv_n,
                                             float &pg) {
  const float lo = 1.0f - eps_lo, hi = 1.0f + eps_hi;
  const float sc = fminf(fmaxf(s, lo), hi);
  const float a1 = s * A, a2 = sc * A;
  pg = -fminf(a1, a2);
  // d min(a1, a2) / ds: a1 branch slope A, a2 branch slope A * [lo <= s <= hi]; ties split evenly
  const float d2 = (s >= lo && s <= hi) ? A : 0.f;
  float dmin;
  if (a1 < a2)
    dmin = A;
  else if (a2 < a1)
    dmin = d2;
  else
    dmin = 0.5f * (A + d2);
  const float g = -dmin;
  return inv_n * g * s / nb;
}

// Vocabularies of at most GS_V logits and T <= GS_THREADS * GS_TPT: a token per thread and round, its logits in
// registers from the log-probs to the gradient. Bound by memory: rows of V elements are no vectors (V = 7), so a
// round's logits and gradients go through LDS and its global accesses are consecutive over the lanes. 512 x 1024
// tokens of 7 bf16 logits with the gradient: 31 us (every token's logits read and exponentiated twice by strided
// 2-byte loads) -> 24 us.
constexpr int GS_V = 8, GS_TPT = 4;
template <bool BF16>
__global__ __launch_bounds__(GS_THREADS) void gspo_score_few_kernel(
    const void *__restrict__ logits, const int64_t *__restrict__ targets, const uint8_t *__restrict__ mask,
    const float *__restrict__ old_lp, const float *__restrict__ n_bases, const float *__restrict__ adv, float eps_lo,
    float eps_hi, float inv_n, float *__restrict__ lp_out, float *__restrict__ s_out, float *__restrict__ pg_out,
    float *__restrict__ dlogits, int T, int V) {
  __shared__ float scratch[GS_THREADS / 64];
  __shared__ float coef_sh;
  __shared__ float stage[GS_THREADS * GS_V];
  const int64_t b = blockIdx.x;
  const int tid = threadIdx.x;
  const bool ratio = old_lp != nullptr && adv != nullptr && n_bases != nullptr;
  float z[GS_TPT][GS_V], lse[GS_TPT];
  int yv[GS_TPT];
  bool on[GS_TPT];
  float part = 0.f;
#pragma unroll
  for (int c = 0; c < GS_TPT; ++c) {
    const int t0 = c * GS_THREADS, t = t0 + tid;
    if (t0 >= T) break;  // uniform
    const int n = min(GS_THREADS, T - t0) * V;
    __syncthreads();  // the previous round's readers are done
    for (int i = tid; i < n; i += GS_THREADS) stage[i] = logit_at<BF16>(logits, (b * T + t0) * V + i);
    __syncthreads();
    on[c] = false;
    if (t >= T) continue;
    const int64_t row = b * T + t;
    int64_t y = targets[row];
    y = (y < 0 || y >= V) ? 0 : y;
    yv[c] = static_cast<int>(y);
    float mx = -INFINITY, s = 0.f;
#pragma unroll
    for (int v = 0; v < GS_V; ++v) {
      z[c][v] = v < V ? stage[tid * V + v] : -INFINITY;
      if (v < V) mx = fmaxf(mx, z[c][v]);
    }
#pragma unroll
    for (int v = 0; v < GS_V; ++v)
      if (v < V) s += expf(z[c][v] - mx);
    lse[c] = mx + logf(s);
    const float lp = stage[tid * V + yv[c]] - lse[c];
    lp_out[row] = lp;
    if (ratio) {
      on[c] = mask[row] != 0;
      if (on[c]) part += lp - old_lp[row];
    }
  }
  if (!ratio) return;
  const float tot = block_sum(part, scratch);
  if (tid == 0) {
    const float nb = n_bases[b], sr = expf(tot / nb);
    float pg;
    coef_sh = ratio_terms(sr, nb, adv[b], eps_lo, eps_hi, inv_n, pg);
    s_out[b] = sr;
    pg_out[b] = pg;
  }
  if (dlogits == nullptr) return;
  __syncthreads();
  const float coef = coef_sh;
  // dL/dz = coef * mask * (onehot - softmax)
#pragma unroll
  for (int c = 0; c < GS_TPT; ++c) {
    const int t0 = c * GS_THREADS;
    if (t0 >= T) break;
    const int n = min(GS_THREADS, T - t0) * V;
    const float k = on[c] ? coef : 0.f;
    if (t0 + tid < T) {
#pragma unroll
      for (int v = 0; v < GS_V; ++v)
        if (v < V) stage[tid * V + v] = k * ((v == yv[c] ? 1.f : 0.f) - expf(z[c][v] - lse[c]));
    }
    __syncthreads();
    for (int i = tid; i < n; i += GS_THREADS) dlogits[(b * T + t0) * V + i] = stage[i];
    __syncthreads();
  }
}

// Larger vocabularies or longer rows: a token per wavefront (V > 32; GS_TW tokens of a wavefront at once) or per thread,
// over the whole batch. (A workgroup per sequence, its four wavefronts taking every fourth token twice, left most CUs
// idle and waited for each token's round trips. Loss and gradient of 64 x 1024 tokens of 343 bf16 logits: 2176 -> 135
// us, of them 90 in these three kernels; of 8 x 512: 674 -> 98.) A token's logits stay in registers (V <= 64 GS_VR)
// between its max, sum and gradient.
constexpr int GS_VR = 8, GS_TW = 2;

// z[k] = logit lane + 64 k of a row (-inf past V), its max and log-sum-exp
template <bool BF16>
__device__ __forceinline__ void row_regs(const void *lg, int64_t base, int V, int lane, float (&z)[GS_VR]) {
#pragma unroll
  for (int k = 0; k < GS_VR; ++k) z[k] = lane + 64 * k < V ? logit_at<BF16>(lg, base + lane + 64 * k) : -INFINITY;
}
__device__ __forceinline__ float lse_regs(const float (&z)[GS_VR], int V, int lane) {
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < GS_VR; ++k) mx = fmaxf(mx, z[k]);
  mx = wave_max(mx);
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < GS_VR; ++k)
    if (lane + 64 * k < V) s += expf(z[k] - mx);
  return mx + logf(wave_sum(s));
}

template <bool BF16, bool WAVE_PER_TOKEN>
__global__ __launch_bounds__(GS_THREADS) void gspo_lp_kernel(const void *__restrict__ logits,
                                                            const int64_t *__restrict__ targets,
                                                            float *__restrict__ lp_out, int64_t n, int V) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  auto target = [&](int64_t row) {
    const int64_t y = targets[row];
    return (y < 0 || y >= V) ? int64_t(0) : y;
  };
  if (!WAVE_PER_TOKEN) {
    const int64_t row = static_cast<int64_t>(blockIdx.x) * GS_THREADS + tid;
    if (row >= n) return;
    float mx, lse;
    lse_thread<BF16>(logits, row * V, V, mx, lse);
    lp_out[row] = logit_at<BF16>(logits, row * V + target(row)) - lse;
    return;
  }
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * (GS_THREADS / 64) + wid) * GS_TW;
  if (V > 64 * GS_VR) {
    for (int i = 0; i < GS_TW && r0 + i < n; ++i) {
      float mx, lse;
      lse_wave<BF16>(logits, (r0 + i) * V, V, lane, mx, lse);
      if (lane == 0) lp_out[r0 + i] = logit_at<BF16>(logits, (r0 + i) * V + target(r0 + i)) - lse;
    }
    return;
  }
  float z[GS_TW][GS_VR], zy[GS_TW];
#pragma unroll
  for (int i = 0; i < GS_TW; ++i) {
    const int64_t row = min(r0 + i, n - 1);
    row_regs<BF16>(logits, row * V, V, lane, z[i]);
    zy[i] = logit_at<BF16>(logits, row * V + target(row));
  }
#pragma unroll
  for (int i = 0; i < GS_TW; ++i) {
    const float lse = lse_regs(z[i], V, lane);
    if (lane == 0 && r0 + i < n) lp_out[r0 + i] = zy[i] - lse;
  }
}

// A workgroup per sequence: the masked sum of (lp - old), the ratio and the objective.
__global__ __launch_bounds__(GS_THREADS) void gspo_ratio_kernel(const float *__restrict__ lp, const uint8_t *__restrict__ mask,
                                                               const float *__restrict__ old_lp,
                                                               const float *__restrict__ n_bases,
                                                               const float *__restrict__ adv, float eps_lo, float eps_hi,
                                                               float inv_n, float *__restrict__ s_out,
                                                               float *__restrict__ pg_out, int64_t T) {
  __shared__ float scratch[GS_THREADS / 64];
  const int64_t b = blockIdx.x;
  float part = 0.f;
  for (int64_t t = threadIdx.x; t < T; t += GS_THREADS)
    if (mask[b * T + t]) part += lp[b * T + t] - old_lp[b * T + t];
  const float tot = block_sum(part, scratch);
  if (threadIdx.x == 0) {
    const float nb = n_bases[b], s = expf(tot / nb);
    float pg;
    ratio_terms(s, nb, adv[b], eps_lo, eps_hi, inv_n, pg);
    s_out[b] = s;
    pg_out[b] = pg;
  }
}

// dL/dz = coef * mask * (onehot - softmax)
template <bool BF16, bool WAVE_PER_TOKEN>
__global__ __launch_bounds__(GS_THREADS) void gspo_grad_kernel(const void *__restrict__ logits,
                                                              const int64_t *__restrict__ targets,
                                                              const uint8_t *__restrict__ mask,
                                                              const float *__restrict__ s_in,
                                                              const float *__restrict__ n_bases,
                                                              const float *__restrict__ adv, float eps_lo, float eps_hi,
                                                              float inv_n, float *__restrict__ dlogits, int64_t n,
                                                              int64_t T, int V) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  auto factor = [&](int64_t row) {
    if (!mask[row]) return 0.f;
    const int64_t b = row / T;
    float pg;
    return ratio_terms(s_in[b], n_bases[b], adv[b], eps_lo, eps_hi, inv_n, pg);
  };
  auto target = [&](int64_t row) {
    const int64_t y = targets[row];
    return (y < 0 || y >= V) ? int64_t(0) : y;
  };
  if (!WAVE_PER_TOKEN) {
    const int64_t row = static_cast<int64_t>(blockIdx.x) * GS_THREADS + tid;
    if (row >= n) return;
    const float c = factor(row);
    const int64_t y = target(row);
    float mx, lse;
    lse_thread<BF16>(logits, row * V, V, mx, lse);
    for (int v = 0; v < V; ++v)
      dlogits[row * V + v] = c * ((v == y ? 1.f : 0.f) - expf(logit_at<BF16>(logits, row * V + v) - lse));
    return;
  }
  const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * (GS_THREADS / 64) + wid) * GS_TW;
  if (V > 64 * GS_VR) {
    for (int i = 0; i < GS_TW && r0 + i < n; ++i) {
      const int64_t row = r0 + i, y = target(row);
      const float c = factor(row);
      float mx, lse;
      lse_wave<BF16>(logits, row * V, V, lane, mx, lse);
      for (int v = lane; v < V; v += 64)
        dlogits[row * V + v] = c * ((v == y ? 1.f : 0.f) - expf(logit_at<BF16>(logits, row * V + v) - lse));
    }
    return;
  }
  float z[GS_TW][GS_VR], c[GS_TW];
  int64_t y[GS_TW];
#pragma unroll
  for (int i = 0; i < GS_TW; ++i) {
    const int64_t row = min(r0 + i, n - 1);
    row_regs<BF16>(logits, row * V, V, lane, z[i]);
    y[i] = target(row);
    c[i] = factor(row);
  }
#pragma unroll
  for (int i = 0; i < GS_TW; ++i) {
    const float lse = lse_regs(z[i], V, lane);
    if (r0 + i >= n) break;
#pragma unroll
    for (int k = 0; k < GS_VR; ++k) {
      const int v = lane + 64 * k;
      if (v < V) dlogits[(r0 + i) * V + v] = c[i] * ((v == y[i] ? 1.f : 0.f) - expf(z[i][k] - lse));
    }
  }
}

// loss = inv_n * sum_b pg[b], one workgroup, fixed order
__global__ __launch_bounds__(GS_THREADS) void gspo_loss_kernel(const float *__restrict__ pg, int64_t B, float inv_n,
                                                               float *__restrict__ loss) {
  __shared__ float scratch[GS_THREADS / 64];
  float part = 0.f;
  for (int64_t b = threadIdx.x; b < B; b += GS_THREADS) part += pg[b];
  const float tot = block_sum(part, scratch);
  if (threadIdx.x == 0) loss[0] = tot * inv_n;
}

__global__ void group_advantage_kernel(const float *__restrict__ reward, int64_t groups, int n, int mode, float param,
                                       float *__restrict__ adv, uint8_t *__restrict__ live) {
  const int64_t gi = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gi >= groups) return;
  const float *r = reward + gi * n;
  float mean = 0.f;
  for (int i = 0; i < n; ++i) mean += r[i];
  mean /= static_cast<float>(n);
  float var = 0.f;
  for (int i = 0; i < n; ++i) var += (r[i] - mean) * (r[i] - mean);
  const float sd = sqrtf(var / static_cast<float>(n));
  const float den = mode == 0 ? fmaxf(sd, param) : sd + param;
  for (int i = 0; i < n; ++i) adv[gi * n + i] = (r[i] - mean) / den;
  if (live) live[gi] = sd > 1e-6f ? 1 : 0;
}

}  // namespace vk

using namespace vk;

extern "C" int vk_gspo_score(const void *logits, int32_t logits_dtype, const int64_t *targets, const uint8_t *mask,
                             const float *old_lp, const float *n_bases, const float *adv, float eps_lo, float eps_hi,
                             float inv_n, float *lp, float *s, float *pg, float *loss, float *dlogits, int64_t B,
                             int64_t T, int32_t V, void *stream) {
  VK_CHECK_ARG(logits && targets && lp, "gspo_score: null pointer");
  VK_CHECK_ARG(logits_dtype == VK_DTYPE_BF16 || logits_dtype == VK_DTYPE_F32, "gspo_score: bad logits dtype");
  VK_CHECK_ARG(B >= 0 && B < (int64_t(1) << 31) && T >= 0 && V > 0, "gspo_score: bad sizes");
  const bool ratio = old_lp != nullptr || adv != nullptr;
  VK_CHECK_ARG(!ratio || (old_lp && adv && n_bases && mask && s && pg && loss),
               "gspo_score: the ratio / loss needs mask, old_lp, n_bases, adv, s, pg and loss");
  VK_CHECK_ARG(dlogits == nullptr || ratio, "gspo_score: dlogits needs the ratio inputs");
  if (B == 0 || T == 0) return VK_OK;
  hipStream_t st = VK_STREAM(stream);
  const bool wave = V > 32;
  const dim3 grid(static_cast<unsigned>(B));
  // few logits per token and rows short enough to stay in registers; longer rows read their logits twice
  if (V <= GS_V && T <= GS_THREADS * GS_TPT) {
    auto kern = logits_dtype == VK_DTYPE_BF16 ? gspo_score_few_kernel<true> : gspo_score_few_kernel<false>;
    kern<<<grid, GS_THREADS, 0, st>>>(logits, targets, mask, ratio ? old_lp : nullptr, n_bases, ratio ? adv : nullptr,
                                      eps_lo, eps_hi, inv_n, lp, s, pg, dlogits, static_cast<int>(T), V);
  } else {
    const bool bf = logits_dtype == VK_DTYPE_BF16;
    const int64_t n = B * T, per = wave ? GS_THREADS / 64 * GS_TW : GS_THREADS, blocks = (n + per - 1) / per;
    VK_CHECK_ARG(blocks < (int64_t(1) << 31), "gspo_score: too many tokens");
    auto lpk = bf ? (wave ? gspo_lp_kernel<true, true> : gspo_lp_kernel<true, false>)
                  : (wave ? gspo_lp_kernel<false, true> : gspo_lp_kernel<false, false>);
    lpk<<<static_cast<unsigned>(blocks), GS_THREADS, 0, st>>>(logits, targets, lp, n, V);
    if (ratio) {
      int rc = launch_status("gspo_score log-probs");
      if (rc != VK_OK) return rc;
      gspo_ratio_kernel<<<grid, GS_THREADS, 0, st>>>(lp, mask, old_lp, n_bases, adv, eps_lo, eps_hi, inv_n, s, pg, T);
      rc = launch_status("gspo_score ratio");
      if (rc != VK_OK) return rc;
    }
    if (ratio && dlogits != nullptr) {
      auto gk = bf ? (wave ? gspo_grad_kernel<true, true> : gspo_grad_kernel<true, false>)
                   : (wave ? gspo_grad_kernel<false, true> : gspo_grad_kernel<false, false>);
      gk<<<static_cast<unsigned>(blocks), GS_THREADS, 0, st>>>(logits, targets, mask, s, n_bases, adv, eps_lo, eps_hi,
                                                              inv_n, dlogits, n, T, V);
    }
  }
  int rc = launch_status("gspo_score");
  if (rc != VK_OK || !ratio) return rc;
  gspo_loss_kernel<<<1, GS_THREADS, 0, st>>>(pg, B, inv_n, loss);
  return launch_status("gspo_loss");
}

extern "C" int vk_group_advantage(const float *reward, int64_t groups, int32_t n, int32_t mode, float param, float *adv,
                                  uint8_t *live, void *stream) {
  VK_CHECK_ARG(reward && adv && groups >= 0 && n > 0, "group_advantage: bad arguments");
  VK_CHECK_ARG(mode == 0 || mode == 1, "group_advantage: mode must be 0 (std floor) or 1 (std + eps)");
  if (groups == 0) return VK_OK;
  group_advantage_kernel<<<static_cast<unsigned>((groups + 255) / 256), 256, 0, VK_STREAM(stream)>>>(
      reward, groups, n, mode, param, adv, live);
  return launch_status("group_advantage");
}
