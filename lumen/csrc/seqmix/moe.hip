// Mixture-of-experts helpers around the two stacked library GEMMs of a hybrid layer's
// feed-forward:
//   sm_route_topk  router logits [T, E] fp32 -> dense routing weights [T, E] fp32 (softmax over
//                  the row's `top` largest logits at their places, zero elsewhere).  One wave per
//                  row: each lane keeps E / 64 logits in registers, `top` rounds of a wave-wide
//                  arg-max (ties: lowest index).
//   sm_route_groups  router with a choice correction and a limit to the best groups of
//                  experts: s = sigmoid(z) (or the softmax of z over all experts; weights then
//                  optionally un-normalised), the choice ranks c = s + correction, a group of
//                  neighbouring experts ranks by the sum of its largest c, only experts of the
//                  `keep` best groups are eligible, the `top` eligible experts with the largest c
//                  get s / (sum of the chosen s + eps) * scale.  One wave per row, the row's c in
//                  LDS; every arg-max breaks ties towards the lowest index.
//   sm_gated_act   act(gate) * up over stacked [gate | up] blocks (act: SiLU, ReLU, tanh-GELU or
//                  squared ReLU; or clamped: g sigmoid(slope g) (u + shift) with g = min(gate, limit),
//                  u = clamp(up, -limit, limit)), expert e's block scaled by the row's routing weight
//                  -- the activation's result, or with weigh_in the gate and up values that enter it
//                  (an expert whose INPUT is weighted); fp32 math.
//   sm_scaled_act  act(up) over stacked up blocks of experts without a gate, scaled the same way.
//   sm_write_k     rows of the key projection into the paged key cache by slot.
#include "route.h"

using namespace lumen;

namespace {

__global__ void __launch_bounds__(256)
route_groups_kernel(const float* __restrict__ z, const float* __restrict__ corr,
                    float* __restrict__ out, int T, int E, int top, int n_groups, int keep,
                    int rank_top, float scale, float sum_eps, int softmax, int normalize) {
  extern __shared__ float s_all[];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int row = blockIdx.x * 4 + wv;
  if (row >= T) return;                              // whole waves leave; no block barrier below
  float* c = s_all + wv * (E + n_groups);
  route_groups_row(z + (long long)row * E, corr, out + (long long)row * E, c, c + E, lane, E, top, n_groups, keep,
                   rank_top, scale, sum_eps, softmax, normalize);
}

template <typename T>
__global__ void scaled_act_kernel(const T* __restrict__ u, const float* __restrict__ wts,
                                  T* __restrict__ out, int Tn, int E, int ff, int ffs, int act) {
  const int width = E * ff + ffs;
  const long long n = (long long)Tn * width;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int t = (int)(i / width), col = (int)(i % width);
    const float w = col < E * ff ? wts[(long long)t * E + col / ff] : 1.f;
    out[i] = from_f32<T>(w == 0.f ? 0.f : gate_act(to_f32(u[i]), act) * w);
  }
}

// eight outputs per thread (16-byte accesses): block sizes multiples of 8, 16-bit dtypes
template <typename T>
__global__ void __launch_bounds__(256)
scaled_act_v8(const T* __restrict__ u, const float* __restrict__ wts, T* __restrict__ out, int Tn,
              int E, int ff, int ffs, int act) {
  const int width = E * ff + ffs;
  const int col = 8 * (blockIdx.x * 256 + threadIdx.x);
  if (col >= width) return;
  const int e = col < E * ff ? col / ff : -1;
  for (int t = blockIdx.y; t < Tn; t += gridDim.y) {
    const float w = e >= 0 ? wts[(long long)t * E + e] : 1.f;
    float v[8], o[8];
    if (w == 0.f) {
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = 0.f;
    } else {
      load8<T>(u + (long long)t * width + col, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = gate_act(v[j], act) * w;
    }
    store8<T>(out + (long long)t * width + col, o);
  }
}

__global__ void __launch_bounds__(256)
route_topk_kernel(const float* __restrict__ z, float* __restrict__ out, int T, int E, int top) {
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= T) return;
  route_topk_row(z + (long long)row * E, out + (long long)row * E, threadIdx.x & 63, E, top);
}

template <typename T>
__global__ void gated_act_kernel(const T* __restrict__ gu, const float* __restrict__ wts,
                                 T* __restrict__ out, int Tn, int E, int ff, int ffs,
                                 const GateForm form) {
  const int in_w = E * 2 * ff + 2 * ffs, out_w = E * ff + ffs;
  const long long n = (long long)Tn * out_w;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int t = (int)(i / out_w), c = (int)(i % out_w);
    const T* row = gu + (long long)t * in_w;
    float g, u, w = 1.f;
    if (c < E * ff) {
      const int e = c / ff, q = c % ff;
      w = wts[(long long)t * E + e];
      g = to_f32(row[e * 2 * ff + q]);
      u = to_f32(row[e * 2 * ff + ff + q]);
    } else {
      const int q = c - E * ff;
      g = to_f32(row[E * 2 * ff + q]);
      u = to_f32(row[E * 2 * ff + ffs + q]);
    }
    out[i] = from_f32<T>(w == 0.f ? 0.f : gated_f(g, u, w, c >= E * ff, form));
  }
}

// eight outputs per thread (16-byte accesses): every block size a multiple of 8, 16-bit dtypes
template <typename T>
__global__ void __launch_bounds__(256)
gated_act_v8(const T* __restrict__ gu, const float* __restrict__ wts, T* __restrict__ out, int Tn,
             int E, int ff, int ffs, const GateForm form) {
  const int in_w = E * 2 * ff + 2 * ffs, out_w = E * ff + ffs;
  const int c = 8 * (blockIdx.x * 256 + threadIdx.x);
  if (c >= out_w) return;
  int e = -1, goff, uoff;
  if (c < E * ff) {
    e = c / ff;
    goff = e * 2 * ff + (c - e * ff);
    uoff = goff + ff;
  } else {
    goff = E * 2 * ff + (c - E * ff);
    uoff = goff + ffs;
  }
  for (int t = blockIdx.y; t < Tn; t += gridDim.y) {
    const T* row = gu + (long long)t * in_w;
    const float w = e >= 0 ? wts[(long long)t * E + e] : 1.f;
    float g[8], u[8], o[8];
    if (w == 0.f) {
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = 0.f;
    } else {
      load8<T>(row + goff, g);
      load8<T>(row + uoff, u);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = gated_f(g[j], u[j], w, e < 0, form);
    }
    store8<T>(out + (long long)t * out_w + c, o);
  }
}

template <typename T>
__global__ void write_k_kernel(const T* __restrict__ k, long long ld, T* __restrict__ cache,
                               const long long* __restrict__ slots, int Tn, int GD) {
  const long long n = (long long)Tn * GD;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    const int t = (int)(i / GD), c = (int)(i % GD);
    const long long s = slots[t];
    if (s >= 0) cache[s * GD + c] = k[(long long)t * ld + c];
  }
}

inline int grid_for(long long n, int block = 256) {
  long long g = (n + block - 1) / block;
  return (int)(g < 1 ? 1 : (g > 65536 ? 65536 : g));
}

}  // namespace

extern "C" {

hipError_t sm_route_topk(const float* z, float* out, int T, int E, int top, hipStream_t st) {
  if (T == 0) return hipSuccess;
  if (E < 1 || E > 64 * kMaxPerLane || top < 1 || top > E) return hipErrorInvalidValue;
  route_topk_kernel<<<(T + 3) / 4, 256, 0, st>>>(z, out, T, E, top);
  return hipGetLastError();
}

// z, out [T, E] fp32; corr [E] fp32.  4 * (E + n_groups) * 4 bytes of LDS per workgroup.
hipError_t sm_route_groups(const float* z, const float* corr, float* out, int T, int E, int top,
                           int n_groups, int keep, int rank_top, float scale, float sum_eps,
                           int softmax, int normalize, hipStream_t st) {
  if (T == 0) return hipSuccess;
  if (E < 1 || E > 64 * kMaxPerLane || n_groups < 1 || E % n_groups || keep < 1 ||
      keep > n_groups || top < 1 || top > keep * (E / n_groups) || rank_top < 1 || rank_top > 4)
    return hipErrorInvalidValue;
  const size_t lds = 4 * (size_t)(E + n_groups) * sizeof(float);
  route_groups_kernel<<<(T + 3) / 4, 256, lds, st>>>(z, corr, out, T, E, top, n_groups, keep,
                                                     rank_top, scale, sum_eps, softmax, normalize);
  return hipGetLastError();
}

hipError_t sm_scaled_act(int dt, const void* u, const float* wts, void* out, int T, int E, int ff,
                         int ffs, int act, hipStream_t st) {
  const long long n = (long long)T * (E * ff + ffs);
  if (n == 0) return hipSuccess;
  if (E > 0 && wts == nullptr) return hipErrorInvalidValue;
  if (ff % 8 == 0 && ffs % 8 == 0 && (dt == kBF16 || dt == kF16)) {
    const dim3 grid(((E * ff + ffs) / 8 + 255) / 256, T < 65535 ? T : 65535);
    if (dt == kBF16)
      scaled_act_v8<bf16><<<grid, 256, 0, st>>>((const bf16*)u, wts, (bf16*)out, T, E, ff, ffs, act);
    else
      scaled_act_v8<fp16><<<grid, 256, 0, st>>>((const fp16*)u, wts, (fp16*)out, T, E, ff, ffs, act);
    return hipGetLastError();
  }
#define CALL(TT) scaled_act_kernel<TT><<<grid_for(n), 256, 0, st>>>((const TT*)u, wts, (TT*)out, T, E, ff, ffs, act)
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

hipError_t sm_gated_act(int dt, const void* gu, const float* wts, void* out, int T, int E, int ff,
                        int ffs, int act, int weigh_in, float limit, float limit_s, float slope,
                        float shift, hipStream_t st) {
  const long long n = (long long)T * (E * ff + ffs);
  if (n == 0) return hipSuccess;
  if (act < 0 || act > 4) return hipErrorInvalidValue;
  const GateForm form{act, weigh_in, limit, limit_s, slope, shift};
  if (E > 0 && wts == nullptr) return hipErrorInvalidValue;
  if (ff % 8 == 0 && ffs % 8 == 0 && (dt == kBF16 || dt == kF16)) {
    const dim3 grid(((E * ff + ffs) / 8 + 255) / 256, T < 65535 ? T : 65535);
    if (dt == kBF16)
      gated_act_v8<bf16><<<grid, 256, 0, st>>>((const bf16*)gu, wts, (bf16*)out, T, E, ff, ffs,
                                                 form);
    else
      gated_act_v8<fp16><<<grid, 256, 0, st>>>((const fp16*)gu, wts, (fp16*)out, T, E, ff, ffs,
                                                 form);
    return hipGetLastError();
  }
#define CALL(TT) gated_act_kernel<TT><<<grid_for(n), 256, 0, st>>>((const TT*)gu, wts, (TT*)out, T, E, ff, ffs, form)
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

hipError_t sm_write_k(int dt, const void* k, long long ld, void* cache, const long long* slots,
                      int T, int GD, hipStream_t st) {
  if ((long long)T * GD == 0) return hipSuccess;
#define CALL(TT) write_k_kernel<TT><<<grid_for((long long)T * GD), 256, 0, st>>>((const TT*)k, ld, (TT*)cache, slots, T, GD)
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

}  // extern "C"
