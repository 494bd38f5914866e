// Routing of one row of logits by one wave, shared by the kernels of moe.hip and route_rows.hip.
#pragma once
#include "seqmix.h"

namespace lumen {

constexpr int kMaxPerLane = 16;   // experts <= 1024

// wave-wide arg-max of (value, index) pairs, ties to the lowest index; every lane gets the result
__device__ __forceinline__ void wave_argmax(float& bv, int& bi) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
  }
}

constexpr int kNone = 0x7fffffff;

// Lane e < E <= 64 holds entry e: how many of them come before it, larger ones and equal ones at lower places.  A choice of the
// largest by counting costs three instructions an entry (0.041 us at 1 - 64 rows), where a round of a wave-wide arg-max is six
// exchanges (0.93 us): it is taken up to kCountPer entries a choice (16 logits, 4 chosen 5.6 -> 2.5 us; 64, 6: 7.6 -> 4.6; 60 of
// which 2 are chosen would be 4.1 us instead of 3.6).
constexpr int kCountPer = 20;
__device__ __forceinline__ int rank_of(float v, int E, int lane) {
  int r = 0;
  for (int j = 0; j < E; ++j) {
    const float o = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), j));
    r += o > v || (o == v && j < lane);
  }
  return r;
}
// the sum of p over the lanes that won, by rank r
__device__ __forceinline__ float sum_by_rank(float p, bool won, int r, int top) {
  float den = 0.f;
  for (int q = 0; q < top; ++q) {
    const unsigned long long at = __ballot(won && r == q);
    if (at == 0) break;
    den += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), __builtin_ctzll(at)));
  }
  return den;
}

// s = sigmoid(z) or the softmax of z over all experts, c = s + corr; see route_groups_kernel.  `c` [E] and
// `rank` [n_groups] are this wave's LDS: the choice ranks (-inf once an expert is chosen or its group dropped) and
// the groups' (-inf once a group is kept)
__device__ __forceinline__ void route_groups_row(const float* zr, const float* __restrict__ corr,
                                                 float* __restrict__ orow, float* c, float* rank, int lane,
                                                 int E, int top, int n_groups, int keep, int rank_top,
                                                 float scale, float sum_eps, int softmax, int normalize) {
  // the scores: sigmoids, or the softmax over all experts (maximum and sum wave-wide, fp32)
  float smax = 0.f, sinv = 1.f;
  if (softmax) {
    smax = -INFINITY;
    for (int e = lane; e < E; e += 64) smax = fmaxf(smax, zr[e]);
    smax = wave_max(smax);
    float ssum = 0.f;
    for (int e = lane; e < E; e += 64) ssum += expf(zr[e] - smax);
    sinv = 1.f / wave_sum(ssum);
  }
  const auto score = [&](int e) {
    return softmax ? expf(zr[e] - smax) * sinv : sigmoid_f(zr[e]);
  };
  for (int e = lane; e < E; e += 64) {
    c[e] = score(e) + (corr != nullptr ? corr[e] : 0.f);
    orow[e] = 0.f;
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  if (n_groups > 1 && keep < n_groups) {
    const int per = E / n_groups;
    // a group's rank: its `rank_top` largest c summed, one lane per group
    for (int g = lane; g < n_groups; g += 64) {
      float sum = 0.f;
      int taken[4] = {-1, -1, -1, -1};               // rank_top <= 4
      for (int r = 0; r < rank_top && r < per; ++r) {
        float bv = -INFINITY;
        int bi = -1;
        for (int k = 0; k < per; ++k) {
          bool used = false;
          for (int q = 0; q < r; ++q) used |= taken[q] == k;
          if (!used && (bi < 0 || c[g * per + k] > bv)) { bv = c[g * per + k]; bi = k; }
        }
        taken[r] = bi;
        sum += bv;
      }
      rank[g] = sum;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    for (int it = 0; it < keep; ++it) {
      float bv = -INFINITY;
      int bi = kNone;
      for (int g = lane; g < n_groups; g += 64)
        if (rank[g] > bv || (rank[g] == bv && g < bi && rank[g] != -INFINITY)) { bv = rank[g]; bi = g; }
      wave_argmax(bv, bi);
      if (bi == kNone) break;
      if (lane == 0) rank[bi] = -INFINITY;           // kept: marked by -inf
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    }
    for (int e = lane; e < E; e += 64)
      if (rank[e / per] != -INFINITY) c[e] = -INFINITY;   // its group was not kept
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  }
  if (E <= 64 && E <= kCountPer * top) {             // a lane an expert; NaN and -inf are never chosen
    const float v = lane < E ? c[lane] : -INFINITY;
    const int r = rank_of(v, E, lane);
    const bool won = v > -INFINITY && r < top;
    const float p = won ? score(lane) : 0.f, den = sum_by_rank(p, won, r, top);
    if (won) orow[lane] = p * (normalize ? scale / (den + sum_eps) : scale);
    return;
  }
  float den = 0.f;
  int mine[16];                                      // top <= E <= 1024: a lane wins <= 16 rounds
  int n_mine = 0;
  for (int it = 0; it < top; ++it) {
    float bv = -INFINITY;
    int bi = kNone;
    for (int e = lane; e < E; e += 64)
      if (c[e] > bv) { bv = c[e]; bi = e; }          // ascending e: ties keep the lowest index
    wave_argmax(bv, bi);
    if (bi == kNone) break;                          // fewer than `top` eligible experts
    den += score(bi);
    if ((bi & 63) == lane) {
      c[bi] = -INFINITY;
      if (n_mine < 16) mine[n_mine++] = bi;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  }
  const float k = normalize ? scale / (den + sum_eps) : scale;
  for (int q = 0; q < n_mine; ++q) orow[mine[q]] = score(mine[q]) * k;
}

// the softmax over the row's `top` largest logits at their places, zero elsewhere
__device__ __forceinline__ void route_topk_row(const float* zr, float* __restrict__ orow, int lane, int E, int top) {
  if (E <= 64 && E <= kCountPer * top) { // a lane an expert; NaN is never chosen
    const float v = lane < E ? zr[lane] : 0.f;
    const int r = rank_of(v, E, lane);
    const bool on = lane < E && v == v, won = on && r < top;
    const unsigned long long first = __ballot(on && r == 0);
    const float m0 = first ? __shfl(v, __builtin_ctzll(first), 64) : 0.f, p = won ? expf(v - m0) : 0.f;
    const float den = sum_by_rank(p, won, r, top);
    if (lane < E) orow[lane] = won ? p / den : 0.f;
    return;
  }
  float val[kMaxPerLane];
  unsigned sel = 0;
#pragma unroll
  for (int q = 0; q < kMaxPerLane; ++q) {
    const int e = lane + 64 * q;
    val[q] = e < E ? zr[e] : -INFINITY;
  }
  float m0 = 0.f, den = 0.f;
  for (int it = 0; it < top; ++it) {
    float bv = -INFINITY;
    int bi = 0x7fffffff;
#pragma unroll
    for (int q = 0; q < kMaxPerLane; ++q) {
      const int e = lane + 64 * q;
      if (e < E && !((sel >> q) & 1u) && (val[q] > bv || (val[q] == bv && e < bi))) {
        bv = val[q];
        bi = e;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
    }
    if (bi == 0x7fffffff) break;         // fewer than `top` finite candidates
    if (it == 0) m0 = bv;
    den += expf(bv - m0);
    if ((bi & 63) == lane) sel |= 1u << (bi >> 6);
  }
#pragma unroll
  for (int q = 0; q < kMaxPerLane; ++q) {
    const int e = lane + 64 * q;
    if (e < E) orow[e] = ((sel >> q) & 1u) ? expf(val[q] - m0) / den : 0.f;
  }
}

}  // namespace lumen
