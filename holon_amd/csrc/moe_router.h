// A mixture's router for steps of few rows, by a block of 16 waves a token: a launch of its own (ffn_kinds.hip) or blocks of another one
// (gemm_skinny.hip).
#pragma once
#include "common.h"

namespace moe_router {
constexpr int BLOCK_WAVES = 16;
struct Lds {
  float z[WAVE + 1], choice[WAVE], group[WAVE];
};

__device__ __forceinline__ float dot4(float x0, float x1, float x2, float x3, const float4& w) {
  return fmaf(x3, w.w, fmaf(x2, w.z, fmaf(x1, w.y, x0 * w.x)));
}

// The choice for one token by one wave, an expert a lane, from the logits in lds.z; its weights go to `to`. (The wave's lanes read back what
// its lanes wrote.)
__device__ __forceinline__ void choose(Lds& lds, const float* __restrict__ bias, float* __restrict__ to, int experts, int rows_r, int top,
                                       int groups, int keep, int score, float scale) {
  float(&z)[WAVE + 1] = lds.z;
  float(&choice)[WAVE] = lds.choice;
  float(&group)[WAVE] = lds.group;
  const int lane = threadIdx.x % WAVE;
  const auto settle = []() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
  settle();
  const bool in = lane < experts;
  float mine = -INFINITY, own = 0.f;                        // the choice score; the score or logit a weight is made of
  if (in) {
    own = z[lane];
    if (score < 0) {
      own = 1.0f / (1.0f + expf(-own));
      mine = bias ? own + bias[lane] : own;
    } else {
      own = bias ? own + bias[lane] : own;
      mine = own;
    }
    choice[lane] = mine;
  }
  settle();
  if (groups > 1) {
    const int size = experts / groups, g = in ? lane / size : 0;
    float best = -INFINITY, next = -INFINITY;               // the group's two largest
    for (int i = 0; i < size; ++i) {
      const float v = choice[g * size + i];
      if (v > best) { next = best; best = v; } else if (v > next) { next = v; }
    }
    const float rank = score < 0 && size > 1 ? best + next : best;
    if (in && lane % size == 0) group[g] = rank;
    settle();
    int before = 0;
    for (int o = 0; o < groups; ++o) before += (group[o] > rank) || (group[o] == rank && o < g);
    if (before >= keep) mine = -INFINITY;
    if (in) choice[lane] = mine;
    settle();
  }
  int ahead = 0;
  for (int o = 0; o < experts; ++o) {
    const float other = choice[o];
    ahead += (other > mine) || (other == mine && o < lane);
  }
  const bool chosen = in && ahead < top && mine > -INFINITY;
  if (score != 0) {
    float s = 0.f;
    if (chosen) s = score < 0 ? own * scale : 1.0f / (1.0f + expf(-own));
    if (in) to[lane] = score == 2 ? s * s : s;
  } else {
    const float top_z = wave_max(mine);                     // the largest logit is always chosen
    const float v = chosen ? expf(mine - top_z) : 0.f;
    const float sum = wave_sum(v);
    if (in) to[lane] = v / sum;
  }
  if (rows_r > experts && lane == 0) to[experts] = 1.0f / (1.0f + expf(-z[experts]));
}

// The router of up to 64 experts for steps of few rows, both kinds: float32 logits z_e = x . router[e] (+ bias[e]), then the choice by one wave with
// an expert a lane. `score` -1: the scores are s = sigmoid(z), experts are chosen by s + bias (a correction; none: by s), a
// group's rank is the sum of its two best, and a chosen expert's weight is s * scale; otherwise as moe_router_top_kernel.
// Equal ones: the lower index first. A logit is added up as the kernels for other sizes do it: PARTS 1 as 64 lanes of a wave,
// PARTS 4 as 256 threads whose waves' sums are added in order, here four sums a lane; so neither the number of rows nor the
// kernel changes a choice.
// A block of 16 waves a token, a wave an expert (all its loads under way at once: one round of memory latency instead of one for
// every few experts): at one row of 2,048 over 8 experts 6.0 us (PARTS 1) and 6.8 (PARTS 4), 8.7 and 10.7 with a block of four
// waves a token.
template <typename T, int PARTS>
__device__ __forceinline__ void few_token(Lds& lds, int64_t t, const T* __restrict__ x, const float* __restrict__ router,
                                          const float* __restrict__ bias, float* __restrict__ weights, int width, int experts, int rows_r,
                                          int top, int groups, int keep, int score, float scale) {
  float(&z)[WAVE + 1] = lds.z;
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const T* row = x + t * width;
  const bool wide = width % 4 == 0 && (uintptr_t)router % 16 == 0;      // (wherever x lies: the order of a sum may not follow it)
  struct Four { T v[4]; };                                  // (aligned as T is; one load all the same)
  for (int e = wave; e < rows_r; e += BLOCK_WAVES) {
    const float* w = router + (int64_t)e * width;
    float acc[PARTS];
#pragma unroll
    for (int q = 0; q < PARTS; ++q) acc[q] = 0.f;
    if (wide) {
#pragma unroll(8 / PARTS)
      for (int i0 = lane * 4; i0 < width; i0 += PARTS * WAVE * 4) {
#pragma unroll
        for (int q = 0; q < PARTS; ++q) {
          const int i = i0 + q * WAVE * 4;
          if (PARTS > 1 && i >= width) break;
          const Four r = *reinterpret_cast<const Four*>(row + i);
          const float4 v = *reinterpret_cast<const float4*>(w + i);
          acc[q] += dot4(Elem<T>::load(r.v[0]), Elem<T>::load(r.v[1]), Elem<T>::load(r.v[2]), Elem<T>::load(r.v[3]), v);
        }
      }
    } else {
      for (int i0 = lane; i0 < width; i0 += PARTS * WAVE) {
#pragma unroll
        for (int q = 0; q < PARTS; ++q) {
          const int i = i0 + q * WAVE;
          if (PARTS > 1 && i >= width) break;
          acc[q] = fmaf(Elem<T>::load(row[i]), w[i], acc[q]);
        }
      }
    }
    float sum = wave_sum(acc[0]);
#pragma unroll
    for (int q = 1; q < PARTS; ++q) sum += wave_sum(acc[q]);
    if (lane == 0) z[e] = sum;
  }
  __syncthreads();
  if (wave == 0) choose(lds, bias, weights + t * rows_r, experts, rows_r, top, groups, keep, score, scale);
}
}  // namespace moe_router
