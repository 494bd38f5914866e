// Shared pieces of the sequence-mixing kernels (hybrid models): dtype dispatch and the fp32
// scalar functions every kernel here uses.  All arithmetic is fp32; 16-bit types only appear at
// loads and stores.  Launchers are `extern "C"`, take raw pointers and a stream, never allocate
// or synchronise (safe under hipGraph capture) and return hipGetLastError().
#pragma once
#include "../kernels/common.h"

namespace lumen {

__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.f + expf(-x)); }
__device__ __forceinline__ float gelu_tanh_f(float z) {
  return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
__device__ __forceinline__ float dyt_f(float x, float alpha, float w, float b) {
  return tanhf(alpha * x) * w + b;
}

// four consecutive elements as one vector access (16 bytes of fp32, 8 bytes of a 16-bit type)
template <typename T> __device__ __forceinline__ void load4(const T* __restrict__ p, float (&o)[4]) {
  const uint2 raw = *reinterpret_cast<const uint2*>(p);
  const T* e = reinterpret_cast<const T*>(&raw);
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = to_f32(e[j]);
}
template <> __device__ __forceinline__ void load4<float>(const float* __restrict__ p, float (&o)[4]) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w;
}
template <typename T> __device__ __forceinline__ void store4(T* __restrict__ p, const float (&v)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
}
template <> __device__ __forceinline__ void store4<float>(float* __restrict__ p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

// the gate's activation: 0 SiLU, 1 ReLU, 2 tanh-GELU, 3 squared ReLU
__device__ __forceinline__ float gate_act(float g, int act) {
  if (act == 3) {
    const float r = fmaxf(g, 0.f);
    return r * r;
  }
  return act == 0 ? silu_f(g) : act == 1 ? fmaxf(g, 0.f) : gelu_tanh_f(g);
}

struct GateForm {
  int act;                                  // as above; 4: clamped, with the constants below
  int weigh_in;                             // the weight multiplies gate and up, not the result
  float limit, limit_s, slope, shift;       // limit: experts; limit_s: the unweighted block
};

// the gated activation of one (gate, up) pair with routing weight w
__device__ __forceinline__ float gated_f(float g, float u, float w, bool shared,
                                         const GateForm& f) {
  if (f.weigh_in) { g *= w; u *= w; }
  float y;
  if (f.act == 4) {
    const float lim = shared ? f.limit_s : f.limit;
    g = fminf(g, lim);
    u = fminf(fmaxf(u, -lim), lim);
    y = g * sigmoid_f(f.slope * g) * (u + f.shift);
  } else {
    y = gate_act(g, f.act) * u;
  }
  return f.weigh_in ? y : y * w;
}

// Workgroup `b` of `n` = tiles x heads -> (tile, head).  Tiles are listed in row order, so the later ones of a
// prompt see more keys: they go first.  Two workgroups share a CU, b and b + 256 as they are handed out:
// every second round of 256 runs backwards, or equal prompts would put two of their last tiles on one CU
// and two first ones on another (16 heads x 8 prompts of 512: 16 key steps against 4).
__device__ __forceinline__ void heavy_first(unsigned b, unsigned n, int heads, int& tile, int& head) {
  const unsigned r = b >> 8;
  if (r & 1) b = (r << 8) + min(256u, n - (r << 8)) - 1 - (b & 255);
  tile = (int)(n / heads) - 1 - (int)(b / heads);
  head = (int)(b % heads);
}

}  // namespace lumen

// run `CALL(T)` with T = float / fp16 / bf16 for dtype code `dt`
#define SM_DISPATCH(dt, CALL)                          \
  switch (dt) {                                        \
    case lumen::kF32: { CALL(float); break; }          \
    case lumen::kF16: { CALL(lumen::fp16); break; }    \
    case lumen::kBF16: { CALL(lumen::bf16); break; }   \
    default: return hipErrorInvalidValue;              \
  }
