// The router of a decode step's rows in one launch: what joins the residual stream, the norm before the experts, the
// router's logits and the routing.
//
//   sm_route_rows   kind 0: the normed rows h are given
//                   kind 1: x += y;  h = x / sqrt(mean(x^2) + eps) * w             (as sm_stream_rms)
//                   kind 2: x += DyT_post(y);  h = DyT_pre(x)                      (as sm_dyt_residual)
//                   then z = h R^T (+ bias) in fp32 from the 16-bit rows, and the routing weights of z as
//                   sm_route_topk (groups = 0) or sm_route_groups form them.
//
// For a few rows each of these was a launch of 4 - 6 us for a few KB.  A workgroup of eight waves takes a row; a wave
// takes every eighth expert, whose first rows (two up to width 4096) it asks for before the norm, as it does for all that the norm
// takes; the logits meet in LDS and one wave routes.
// Every row reads the router again (64 KB from L2), which 64 rows still hide.
// All of the norm's operands are asked for before its sum, and few experts are ranked by counting (route.h): one row of 2048, 8
// experts 5.2 -> 4.1 us, 16 experts 5.6 -> 4.7.
// Measured as a decode step's time (bf16, width 2048): one row, three layers of 16 experts 296.6 -> 284.0 us; eight rows,
// two layers of 8 experts 375.8 -> 368.6.
#include "route.h"

using namespace lumen;

namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kMaxE = 64, kMaxW = 8192;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// 8 products of 16-bit values, fp32 (fp16 by mixed fmas: the dot instruction need not keep subnormals)
template <typename T>
__device__ __forceinline__ float dot8(const uint4& a, const uint4& b, float s) {
  if constexpr (sizeof(T) == 2 && __is_same(T, bf16)) {
    const unsigned x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x[j]), __builtin_bit_cast(bf16x2, y[j]), s, false);
  } else {
    const T *x = reinterpret_cast<const T*>(&a), *y = reinterpret_cast<const T*>(&b);
#pragma unroll
    for (int j = 0; j < 8; ++j) s = fmaf(to_f32(x[j]), to_f32(y[j]), s);
  }
  return s;
}

template <typename T> struct RouteArgs {
  float* x; const T* y;                     // kinds 1, 2
  T* h; long long ldh;                      // kind 0: read; else written (rows of W)
  const float *w, *b, *alpha;               // the norm before the experts (kind 1: w alone)
  const float *pw, *pb, *pa;                // kind 2: DyT of y
  const T *R, *bias;                        // [E, W]; bias [E] or null
  float* out;                               // [T, E]
  int W, E;
  float eps;
  int top, groups, keep, rank_top, softmax, normalize;
  float scale, sum_eps; const float* corr;
};

// KS: 512-column steps of a row
template <typename T, int KIND, int KS>
__global__ void __launch_bounds__(kThreads) route_rows_kernel(const RouteArgs<T> a) {
  __shared__ __attribute__((aligned(16))) T s_h[KS * 512];
  __shared__ float s_z[kMaxE], s_c[2 * kMaxE], s_red[kWaves];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = a.W;
  const long long row = blockIdx.x;
  constexpr int B = KS <= 8 && (KS <= 4 || std::is_same<T, bf16>::value) ? 2 : 1;   // a wave's experts at a time: what registers hold
  uint4 r[B][KS];
  const auto ask = [&](int e, uint4 (&o)[KS]) __attribute__((always_inline)) {
    if (e >= a.E) return;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      const int c = 512 * u + 8 * lane;
      o[u] = c < W ? *reinterpret_cast<const uint4*>(a.R + (long long)e * W + c) : make_uint4(0, 0, 0, 0);
    }
  };
#pragma unroll
  for (int b = 0; b < B; ++b) ask(w + b * kWaves, r[b]);
  if constexpr (KIND > 0) {
    constexpr int N = (KS * 512 + 4 * kThreads - 1) / (4 * kThreads);
    float v[N][4], y[N][4], nw[N][4], nb[N][4], pw[N][4], pb[N][4], sq = 0.f;
    Raw4<T> y4[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {                        // (no branch: past the row's end, its first channels again)
      const int c0 = 4 * (threadIdx.x + i * kThreads), c = c0 < W ? c0 : 0;
      load4<float>(a.x + row * W + c, v[i]);
      y4[i].ask(a.y + row * W + c);
      load4<float>(a.w + c, nw[i]);
      if constexpr (KIND == 2) {
        load4<float>(a.pw + c, pw[i]);
        load4<float>(a.pb + c, pb[i]);
        load4<float>(a.b + c, nb[i]);
      }
    }
    const float ap = KIND == 2 ? *a.pa : 0.f, an = KIND == 2 ? *a.alpha : 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = 4 * (threadIdx.x + i * kThreads);
      if (c >= W) break;
      y4[i].get(y[i]);
      if constexpr (KIND == 2) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[i][e] = dyt_f(y[i][e], ap, pw[i][e], pb[i][e]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[i][e] += y[i][e];
        sq += v[i][e] * v[i][e];
      }
      store4<float>(a.x + row * W + c, v[i]);
    }
    float inv = 0.f;
    if constexpr (KIND == 1) inv = 1.f / sqrtf(block_sum<kThreads>(sq, s_red) / (float)W + a.eps);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = 4 * (threadIdx.x + i * kThreads);
      if (c >= W) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[i][e] = KIND == 1 ? v[i][e] * inv * nw[i][e] : dyt_f(v[i][e], an, nw[i][e], nb[i][e]);
      store4<T>(a.h + row * a.ldh + c, v[i]);
      store4<T>(s_h + c, v[i]);
    }
    __syncthreads();
  }
  uint4 x[KS];
#pragma unroll
  for (int u = 0; u < KS; ++u) {
    const int c = 512 * u + 8 * lane;
    x[u] = make_uint4(0, 0, 0, 0);
    if (c < W) x[u] = *reinterpret_cast<const uint4*>(KIND > 0 ? s_h + c : a.h + row * a.ldh + c);
  }
  for (int e = w; e < a.E; e += B * kWaves) {
    float z[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      float s[2] = {0.f, 0.f};
      if (e + b * kWaves < a.E) {
#pragma unroll
        for (int u = 0; u < KS; ++u) s[u & 1] = dot8<T>(r[b][u], x[u], s[u & 1]);
      }
      z[b] = s[0] + s[1];
      ask(e + (B + b) * kWaves, r[b]);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int f = e + b * kWaves;
      z[b] = wave_sum(z[b]);
      if (lane == 0 && f < a.E) s_z[f] = z[b] + (a.bias != nullptr ? to_f32(a.bias[f]) : 0.f);
    }
  }
  __syncthreads();
  if (w != 0) return;
  float* o = a.out + row * a.E;
  if (a.groups == 0) route_topk_row(s_z, o, lane, a.E, a.top);
  else route_groups_row(s_z, a.corr, o, s_c, s_c + kMaxE, lane, a.E, a.top, a.groups, a.keep, a.rank_top, a.scale,
                        a.sum_eps, a.softmax, a.normalize);
}

template <typename T, int KIND>
hipError_t launch(const RouteArgs<T>& a, int rows, hipStream_t st) {
#define GO(KS) route_rows_kernel<T, KIND, KS><<<rows, kThreads, 0, st>>>(a)
  if (a.W <= 1024) GO(2);
  else if (a.W <= 2048) GO(4);
  else if (a.W <= 4096) GO(8);
  else GO(16);
#undef GO
  return hipGetLastError();
}

}  // namespace

extern "C" {

// 16-bit rows, W % 8 == 0, W <= 8192, E <= 64; x, y, h (kinds 1, 2) contiguous rows, all bases 16-byte aligned.
hipError_t sm_route_rows(int dt, int kind, float* x, const void* y, void* h, long long ldh, const float* w,
                         const float* b, const float* alpha, const float* pw, const float* pb, const float* pa,
                         const void* R, const void* bias, float* out, int rows, int W, int E, float eps, int top,
                         int groups, int keep, int rank_top, int softmax, int normalize, float scale, float sum_eps,
                         const float* corr, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (rows < 0 || W < 8 || W % 8 || W > kMaxW || E < 1 || E > kMaxE || ldh < W || ldh % 8 || top < 1 || !h || !R ||
      !out || !al(x) || !al(y) || !al(h) || !al(w) || !al(b) || !al(pw) || !al(pb) || !al(R) || kind < 0 || kind > 2 ||
      (kind > 0 && (!x || !y || !w)) || (kind == 2 && (!b || !alpha || !pw || !pb || !pa)) ||
      (groups == 0 ? top > E
                   : groups < 1 || E % groups || keep < 1 || keep > groups || top > keep * (E / groups) ||
                         rank_top < 1 || rank_top > 4) ||
      (dt != kBF16 && dt != kF16))
    return hipErrorInvalidValue;
#define GO(T)                                                                                                      \
  {                                                                                                                \
    const RouteArgs<T> a{x, (const T*)y, (T*)h, ldh, w, b, alpha, pw, pb, pa, (const T*)R, (const T*)bias, out, W, \
                         E, eps, top, groups, keep, rank_top, softmax, normalize, scale, sum_eps, corr};           \
    return kind == 0 ? launch<T, 0>(a, rows, st) : kind == 1 ? launch<T, 1>(a, rows, st)                           \
                                                             : launch<T, 2>(a, rows, st);                          \
  }
  if (dt == kBF16) GO(bf16)
  GO(fp16)
#undef GO
}

}  // extern "C"
