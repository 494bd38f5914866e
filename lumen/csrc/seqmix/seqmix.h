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

// expf, logf, tanhf and an exact division from the hardware's 2^t, log2 and reciprocal with their roundings made good,
// at a third of the instructions, for the inner loops that those bound.  Largest error in units of the last place,
// the library's -> here (4 M values each): e^x, -80 .. 5: 0.85 -> 1.25 (the hardware's form as it is 62); ln, 1 .. 500: 2.3 -> 2.1;
// tanh 1.4 -> 2.2; sigmoid, -60 .. 60: 2.5 -> 3.4 (58).
// e^x for x up to 88 (more: as 88; below -200: 0)
__device__ __forceinline__ float exp_near(float x) {
  constexpr float kL = 1.44269502f, kLlo = 1.92596299e-8f;     // log2(e) = kL + kLlo
  x = x < -200.f ? -200.f : x > 88.f ? 88.f : x;               // (NaN stays)
  const float t = x * kL, lo = fmaf(x, kLlo, fmaf(x, kL, -t));
  const float r = __builtin_amdgcn_exp2f(t);
  return fmaf(r, lo * 0.693147182f, r);
}
// 1 / d for 1 <= d < 2^127
__device__ __forceinline__ float recip_near(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, r, 1.f), r, r);
}
__device__ __forceinline__ float sigmoid_near(float x) { return recip_near(1.f + exp_near(-x)); }
// g / (1 + e^-z) as expf and a division give it, in the half of their instructions: e^-z from the hardware's 2^f, |f| <= 1/2, the
// quotient from its reciprocal and one remainder.  Largest error in units of the last place (mean square) over 16 M values, |g| up to 88, silu_f -> here:
// 2.72 (0.441) -> 2.72 (0.442); g sigmoid_f(1.7 g) -> here 2.65 (0.473) -> 2.18 (0.401).  KEEP: NaN z with a g that is none.
template <bool KEEP>
__device__ __forceinline__ float logistic_gate(float g, float z) {
  constexpr float kL = 1.44269502f, kLlo = 1.92596299e-8f;     // log2(e) = kL + kLlo
  float x = -z;                                                // beyond +-200 as there: e^x is 0 or infinite
  x = !KEEP ? __builtin_amdgcn_fmed3f(x, -200.f, 200.f) : x < -200.f ? -200.f : x > 200.f ? 200.f : x;
  const float n = rintf(x * kL), f = fmaf(x, kLlo, fmaf(x, kL, -n));
  const float e = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
  const float d = fmaf(e, 0.25f, 0.25f), r = __builtin_amdgcn_rcpf(d), g4 = 0.25f * g;     // (a quarter: the reciprocal is no denormal)
  const float q = g4 * r, rest = fmaf(-d, q, g4);
  return rest == rest ? fmaf(rest, r, q) : q;                  // (no remainder where g or d is infinite)
}
// ln x for normal x
__device__ __forceinline__ float log_near(float x) {
  constexpr float kL = 0.693147182f, kLlo = -1.90465421e-9f;   // ln 2 = kL + kLlo
  const float y = __builtin_amdgcn_logf(x), r = y * kL;
  return r + fmaf(y, kLlo, fmaf(y, kL, -r));
}
// tanh x: near 0 an odd polynomial (least squares in x^2, weighted to an even relative error of 3e-10), else through
// one exponential of |x|
__device__ __forceinline__ float tanh_near(float x) {
  const float z = x * x;
  float p = fmaf(z, -0.00665356684f, 0.0213016998f);
  p = fmaf(z, p, -0.0538999699f);
  p = fmaf(z, p, 0.133329704f);
  p = fmaf(z, p, -0.333333284f);
  return z < 0.25f ? fmaf(x, z * p, x) : copysignf(1.f - 2.f * recip_near(1.f + exp_near(2.f * fabsf(x))), x);
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
// the same asked for now and converted where it is used: a conversion waits for its load, also under a branch not yet left
template <typename T> struct Raw4 {
  uint2 v;
  __device__ __forceinline__ void ask(const T* __restrict__ p) { v = *reinterpret_cast<const uint2*>(p); }
  __device__ __forceinline__ void put(T* __restrict__ p) const { *reinterpret_cast<uint2*>(p) = v; }
  __device__ __forceinline__ void get(float (&o)[4]) const { load4<T>(reinterpret_cast<const T*>(&v), o); }
};
template <> struct Raw4<float> {
  float4 v;
  __device__ __forceinline__ void ask(const float* __restrict__ p) { v = *reinterpret_cast<const float4*>(p); }
  __device__ __forceinline__ void put(float* __restrict__ p) const { *reinterpret_cast<float4*>(p) = v; }
  __device__ __forceinline__ void get(float (&o)[4]) const { o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w; }
};
template <typename T> __device__ __forceinline__ void store4(T* __restrict__ p, const float (&v)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
}
template <> __device__ __forceinline__ void store4<float>(float* __restrict__ p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

// infinities and NaN among 16-bit values
template <typename T> struct OddBits {            // exponents of all ones and their lowest bit, in both halves
  static constexpr unsigned E = 0x7c007c00u, one = 0x04000400u;
};
template <> struct OddBits<bf16> { static constexpr unsigned E = 0x7f807f80u, one = 0x00800080u; };
template <typename T> __device__ __forceinline__ unsigned odd2(unsigned v) {      // bits 15 and 31
  return ((v & OddBits<T>::E) + OddBits<T>::one) & 0x80008000u;
}
template <typename T> __device__ __forceinline__ bool odd8(const uint4& v) {
  return (odd2<T>(v.x) | odd2<T>(v.y) | odd2<T>(v.z) | odd2<T>(v.w)) != 0;
}
template <typename T> __device__ __forceinline__ unsigned finite2(unsigned v) { return v & ~((odd2<T>(v) >> 15) * 0xffffu); }
template <typename T> __device__ __forceinline__ uint4 finite8(const uint4& v) {
  return make_uint4(finite2<T>(v.x), finite2<T>(v.y), finite2<T>(v.z), finite2<T>(v.w));
}
// the infinities and NaN of four consecutive 16-bit values, 0 elsewhere
template <typename T> __device__ __forceinline__ void odd4(const T* p, float (&o)[4]) {
  load4<T>(p, o);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = fabsf(o[e]) < INFINITY ? 0.f : o[e];
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
