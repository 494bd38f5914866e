// One decoded row: y = act(W rms_norm(x + r) + b), the norm formed in the projection's prologue and the gated activation in
// its epilogue -- a batch-1 step's q|k|v, gate|up and head projections.
//
// A step of one row is a chain of weight streams with small kernels between them, 3 - 4 us each where their work is
// nothing (norm of one row: 24 KB).  Here every wave asks for its first weight rows, then the workgroup forms the normed
// row for itself while those are under way (24 KB from L2, met in LDS), and every wave keeps all of it in registers:
//  * a wave streams whole weight rows, lane = one 16-byte chunk, 1 KiB per instruction, D rows in flight, no barrier;
//  * gated: a wave's rows are a gate row and its up row in turn, so silu(gate) * up leaves the kernel from the fp32 sums;
//  * the sum x + r (rounded, the next residual) is stored by the first workgroup, into a buffer of its own.
// The rounding of the normed row is that of the norm kernel.  STREAM: x, the norm's weight and the sum are fp32, the
// residual stream of a stack of mixers, which the sublayer's output r joins.  (Tazulix, one stream, width 2048: 284 -> 274
// us a step with the norms before the mixers, a dense feed-forward and the head in their projections.)
// Bound by HBM (6.3 TB/s and ~5 us of start and drain).  Measured in a graph, weights rotated, norm + projection (+
// activation) -> here, us, one bf16 row: 3072 x 2048 8.0 -> 5.5, 11264 x 2048 gated 15.8 -> 11.2, 32000 x 2048 28.0 -> 22.9,
// 16896 x 3072 gated 27.9 -> 20.1, 12288 x 4096 19.6 -> 18.4, 22016 x 4096 gated 33.4 -> 30.7, 32000 x 4096 43.1 -> 42.5, 8192 x
// 8192 28.6 -> 25.4, 1536 x 1024 5.6 -> 4.0.  (A quarter of K per wave, four rows at a time and a barrier each: 19.0 - 31.6.)
#include "seqmix.h"

using namespace lumen;

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
template <typename T> __device__ __forceinline__ float dot2(unsigned a, unsigned b, float c);
template <> __device__ __forceinline__ float dot2<bf16>(unsigned a, unsigned b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
template <> __device__ __forceinline__ float dot2<fp16>(unsigned a, unsigned b, float c) {
  return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
}
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <typename T> __device__ __forceinline__ uint4 ntload(const T* p) {
  return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)));
}
template <int CTRL> __device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float sum64(float v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  v += dpp<0x140>(v);
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

template <typename T> struct RowGemvArgs {
  const T *x, *r, *wn;      // the row, the residual (nullable), the norm's weight
  T* s;                     // x + r (written when r is given)
  const T* W;
  T* y;
  int K, F;                 // F: result columns (gated: half of W's rows)
  float eps;
  const float *xs, *ws;     // STREAM: the row and the norm's weight; ss takes the sum
  float* ss;
  const T* bias;            // [F] or null
  int act;                  // of the result: -1 none, else gate_act's
  float* y32;               // takes the result in fp32 instead of y
};

// KS: 512-element steps of K; D: weight rows in flight per wave
template <typename T, bool GATED, int KS, int D, bool STREAM>
__global__ void __launch_bounds__(256, 2) row_gemv_kernel(const RowGemvArgs<T> a) {
  static_assert(!GATED || D % 2 == 0, "rows come in pairs");
  __shared__ float s_ss[4];
  __shared__ __attribute__((aligned(16))) T s_x[KS * 512];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = gridDim.x * 4, wave = blockIdx.x * 4 + w;
  // the wave's n-th row: plain row wave + n waves; gated: gate and up row of column wave + (n / 2) waves
  const int mine = wave < a.F ? (a.F - 1 - wave) / waves + 1 : 0, rows = GATED ? 2 * mine : mine;
  const uint4 z = make_uint4(0, 0, 0, 0);
  uint4 wv[D][KS];
  const auto load = [&](int n, uint4 (&o)[KS]) __attribute__((always_inline)) {
    const long long row = GATED ? wave + (long long)(n >> 1) * waves + (n & 1 ? a.F : 0) : wave + (long long)n * waves;
    const T* p = a.W + row * a.K;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      // (the last step that K reaches may end within it, and need not be the last of KS)
      if (512 * (u + 1) <= a.K) o[u] = ntload(p + 512 * u + 8 * lane);
      else o[u] = 512 * u + 8 * lane < a.K ? ntload(p + 512 * u + 8 * lane) : z;
    }
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (d < rows) load(d, wv[d]);
  // the normed row: a quarter per wave, met in LDS
  {
    constexpr int Q = (KS + 3) / 4;
    float v[Q][8], g[Q][8], ss = 0.f;
#pragma unroll
    for (int u = 0; u < Q; ++u) {
      const int at0 = 512 * (4 * u + w) + 8 * lane;
      const bool ok = 4 * u + w < KS && at0 < a.K;
      const int at = ok ? at0 : 0;
      if constexpr (STREAM) {
        load8<float>(a.xs + at, v[u]);
        load8<float>(a.ws + at, g[u]);
        if (a.r) {
          float rr[8];
          load8<T>(a.r + at, rr);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[u][e] += rr[e];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[u][e] = ok ? v[u][e] : 0.f;
          ss += v[u][e] * v[u][e];
        }
        if (ok && a.r && blockIdx.x == 0) store8<float>(a.ss + at, v[u]);
      } else {
        const Vec8<T> xr = *reinterpret_cast<const Vec8<T>*>(a.x + at);
        const Vec8<T> rr = *reinterpret_cast<const Vec8<T>*>((a.r ? a.r : a.x) + at);
        const Vec8<T> wr = *reinterpret_cast<const Vec8<T>*>(a.wn + at);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          float t = to_f32(xr.v[e]);
          if (a.r) t += to_f32(rr.v[e]);
          v[u][e] = ok ? t : 0.f;
          g[u][e] = to_f32(wr.v[e]);
          ss += v[u][e] * v[u][e];
        }
        if (ok && a.r && blockIdx.x == 0)
          *reinterpret_cast<uint4*>(a.s + at) = make_uint4(pk2<T>(v[u][0], v[u][1]), pk2<T>(v[u][2], v[u][3]),
                                                           pk2<T>(v[u][4], v[u][5]), pk2<T>(v[u][6], v[u][7]));
      }
    }
    ss = sum64(ss);
    if (lane == 0) s_ss[w] = ss;
    __syncthreads();
    const float ms = (s_ss[0] + s_ss[1] + s_ss[2] + s_ss[3]) / (float)a.K + a.eps;
    const float rs = STREAM ? 1.f / sqrtf(ms) : rsqrtf(ms);
#pragma unroll
    for (int u = 0; u < Q; ++u) {
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = v[u][e] * rs * g[u][e];
      if (4 * u + w < KS)
        *reinterpret_cast<uint4*>(s_x + 512 * (4 * u + w) + 8 * lane) =
            make_uint4(pk2<T>(o[0], o[1]), pk2<T>(o[2], o[3]), pk2<T>(o[4], o[5]), pk2<T>(o[6], o[7]));
    }
    __syncthreads();
  }
  uint4 xn[KS];
#pragma unroll
  for (int u = 0; u < KS; ++u) xn[u] = *reinterpret_cast<const uint4*>(s_x + 512 * u + 8 * lane);
  float gate = 0.f;
  for (int n0 = 0; n0 < rows; n0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int n = n0 + d;
      if (n >= rows) break;
      if (n + D - 1 < rows) load(n + D - 1, wv[(d + D - 1) % D]);
      float acc[2] = {0.f, 0.f};
#pragma unroll
      for (int u = 0; u < KS; ++u) {
        acc[u & 1] = dot2<T>(wv[d][u].x, xn[u].x, acc[u & 1]);
        acc[u & 1] = dot2<T>(wv[d][u].y, xn[u].y, acc[u & 1]);
        acc[u & 1] = dot2<T>(wv[d][u].z, xn[u].z, acc[u & 1]);
        acc[u & 1] = dot2<T>(wv[d][u].w, xn[u].w, acc[u & 1]);
      }
      const float o = sum64(acc[0] + acc[1]);
      if constexpr (GATED) {
        if (d % 2 == 0) gate = o;
        else if (lane == 0) a.y[wave + (long long)(n >> 1) * waves] = from_f32<T>(silu_f(gate) * o);
      } else {
        if constexpr (STREAM) {          // (in the other form these branches cost a batch-1 Llama step 19 of 377 us)
          if (lane == 0) {
            const long long c = wave + (long long)n * waves;
            float z = o + (a.bias ? to_f32(a.bias[c]) : 0.f);
            if (a.act >= 0) z = gate_act(z, a.act);
            if (a.y32) a.y32[c] = z;
            else a.y[c] = from_f32<T>(z);
          }
        } else {
          if (lane == 0) a.y[wave + (long long)n * waves] = from_f32<T>(o);
        }
      }
    }
  }
}

// as many workgroups as stay on the chip: two per CU with the rows of a pair in flight, three without where there are
// rows for them (22016 x 4096 gated 30.7 us with 512, 33.3 with 768; 32000 x 4096 44.3 and 42.5)
template <typename T, bool GATED, bool STREAM = false>
hipError_t launch(const RowGemvArgs<T>& a, hipStream_t st) {
  const int wgs = (a.F + 3) / 4, most = !GATED && a.F >= 12288 ? 768 : 512;
  const dim3 grid(wgs < most ? wgs : most);
  const int ks = (a.K + 511) / 512;
#define GO(KS, D) row_gemv_kernel<T, GATED, KS, D, STREAM><<<grid, 256, 0, st>>>(a)
  if (ks <= 2) GO(2, 8);
  else if (ks <= 3) GO(3, 8);
  else if (ks <= 4) GO(4, 8);
  else if (ks <= 6) GO(6, 4);
  else if (ks <= 8) GO(8, 4);
  else if (ks <= 12) GO(12, 2);
  else if (ks <= 16) GO(16, 2);
  else return hipErrorInvalidValue;
#undef GO
  return hipGetLastError();
}

}  // namespace

extern "C" {

// y = W rms_norm(x + r) for one row: x, r (or null), wn [K], W [F or, gated, 2 F][K] contiguous, y [F]; gated: y =
// silu(W[:F] n) * (W[F:] n).  s [K] takes x + r.  K <= 8192, K % 8 == 0, F % 4 == 0 (gated % 2), 16-byte bases.
hipError_t sm_row_gemv(int dt, const void* x, const void* r, const void* wn, void* s, const void* W, void* y, int K,
                       int F, int gated, float eps, hipStream_t st) {
  if (F == 0) return hipSuccess;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (K < 8 || K > 8192 || K % 8 || F < 0 || F % (gated ? 2 : 4) || !al(x) || !al(r) || !al(wn) || !al(s) || !al(W) ||
      (r != nullptr && (s == nullptr || s == x || s == r)) || (dt != kBF16 && dt != kF16))
    return hipErrorInvalidValue;
#define GO(T)                                                                                       \
  {                                                                                                 \
    const RowGemvArgs<T> a{(const T*)x, (const T*)r, (const T*)wn, (T*)s, (const T*)W, (T*)y, K, F, eps, \
                              nullptr, nullptr, nullptr, nullptr, -1, nullptr};                    \
    return gated ? launch<T, true>(a, st) : launch<T, false>(a, st);                                \
  }
  if (dt == kBF16) GO(bf16)
  GO(fp16)
#undef GO
}

// y = act(W rms_norm(x + r) + b) of one row of an fp32 stream: x, wn [K] fp32, r [K] (or null) and W [F][K] 16-bit; s [K] fp32 takes
// x + r (with r; not x itself).  bias [F] or null; act -1 (none) .. 3; y [F] in the type dt, or fp32 with out32.  K, F and
// bases as above (bias and y need no alignment).
hipError_t sm_row_stream(int dt, const float* x, const void* r, const float* wn, float* s, const void* W, const void* bias,
                         void* y, int K, int F, int act, int out32, float eps, hipStream_t st) {
  if (F == 0) return hipSuccess;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (K < 8 || K > 8192 || K % 8 || F < 0 || !al(x) || !al(r) || !al(wn) || !al(s) || !al(W) || !x || !wn || !W || !y ||
      (r != nullptr && (s == nullptr || s == x)) || act < -1 || act > 3 || (dt != kBF16 && dt != kF16))
    return hipErrorInvalidValue;
#define GO(T)                                                                                                         \
  {                                                                                                                   \
    const RowGemvArgs<T> a{nullptr, (const T*)r, nullptr, nullptr, (const T*)W, (T*)y, K, F, eps, x, wn, s, (const T*)bias, \
                           act, out32 ? (float*)y : nullptr};                                                         \
    return launch<T, false, true>(a, st);                                                                             \
  }
  if (dt == kBF16) GO(bf16)
  GO(fp16)
#undef GO
}

}  // extern "C"
