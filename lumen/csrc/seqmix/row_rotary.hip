// Whole-projection q / k norm, rotation and cache writes of an attention layer in one pass:
//
//   sm_row_norm_rotary  a fused projection's row [q heads | k heads | values]: q and k are RMS-normed
//                       over ALL their entries at once (every head together) with weights of that
//                       size and turned on the first `dims` entries of every head in the half layout
//                       (entry i with entry i + dims / 2) by position * inv_freq[i], cosine and sine
//                       carrying the factor `amp`; q in place, k and the values as projected into
//                       their paged caches.
//
// One workgroup of four waves per row.  The sums of squares of the two parts are reduced in a fixed
// order; the row's dims / 2 sines and cosines are computed once, in LDS, for all heads.  A work item is
// V consecutive entries and, where they turn, their V partners: it is read, normed, turned and stored
// by one lane, so nothing is exchanged and nothing is read after it was replaced.  Norms, angles and
// the rotation are fp32; only a stored q or k is rounded.
#include "seqmix.h"

using namespace lumen;

namespace {

constexpr int kThreads = 256;
constexpr int kMaxHead = 512;

template <typename T>
struct RowRotArgs {
  T* z; long long ld;
  const float* wq; const float* wk;
  const int* positions; const long long* slots;
  T* kc; T* vc;
  const float* inv_freq;
  int H, G, D, vw, dims;                     // vw: value columns (G * Dv)
  float amp, eps;
};

template <typename T, int V>
__device__ __forceinline__ void load_v(const T* p, float (&o)[V]) {
  if constexpr (V == 8) load8<T>(p, o);
  else if constexpr (V == 4) load4<T>(p, o);
  else o[0] = to_f32(p[0]);
}
template <typename T, int V>
__device__ __forceinline__ void store_v(T* p, const float (&o)[V]) {
  if constexpr (V == 8) store8<T>(p, o);
  else if constexpr (V == 4) store4<T>(p, o);
  else p[0] = from_f32<T>(o[0]);
}

template <typename T, int V>
__global__ void __launch_bounds__(kThreads) row_norm_rotary_kernel(const RowRotArgs<T> a) {
  __shared__ float s_cs[kMaxHead / 2], s_sn[kMaxHead / 2];
  __shared__ float s_red[2][kThreads / 64];
  const int t = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int half = a.dims / 2, HD = a.H * a.D, GD = a.G * a.D;
  const long long slot = a.slots[t];
  T* row = a.z + (long long)t * a.ld;
  const float pos = (float)a.positions[t];
  for (int i = threadIdx.x; i < half; i += kThreads) {
    float sn, cs;
    sincosf(pos * a.inv_freq[i], &sn, &cs);
    s_sn[i] = sn * a.amp;
    s_cs[i] = cs * a.amp;
  }
  float sq = 0.f, sk = 0.f;
  for (int c = threadIdx.x * V; c < HD; c += kThreads * V) {
    float v[V];
    load_v<T, V>(row + c, v);
#pragma unroll
    for (int e = 0; e < V; ++e) sq += v[e] * v[e];
  }
  for (int c = threadIdx.x * V; c < GD; c += kThreads * V) {
    float v[V];
    load_v<T, V>(row + HD + c, v);
#pragma unroll
    for (int e = 0; e < V; ++e) sk += v[e] * v[e];
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) {
    s_red[0][w] = sq;
    s_red[1][w] = sk;
  }
  __syncthreads();
  sq = (s_red[0][0] + s_red[0][1]) + (s_red[0][2] + s_red[0][3]);
  sk = (s_red[1][0] + s_red[1][1]) + (s_red[1][2] + s_red[1][3]);
  const float iq = 1.f / sqrtf(sq / (float)HD + a.eps), ik = 1.f / sqrtf(sk / (float)GD + a.eps);
  const int turning = half / V, per = turning + (a.D - a.dims) / V;     // items of a head
  for (int it = threadIdx.x; it < (a.H + a.G) * per; it += kThreads) {
    const int hd = it / per, j = it - hd * per;
    const bool is_q = hd < a.H, turns = j < turning;
    const int c = turns ? j * V : a.dims + (j - turning) * V;           // first entry in the head
    const T* src = row + hd * a.D + c;
    const float* wt = is_q ? a.wq + hd * a.D + c : a.wk + (hd - a.H) * a.D + c;
    const float inv = is_q ? iq : ik;
    T* dst = is_q ? row + hd * a.D + c
                  : (slot < 0 ? nullptr : a.kc + slot * GD + (hd - a.H) * a.D + c);
    float u[V], ww[V];
    load_v<T, V>(src, u);
    load_v<float, V>(wt, ww);
#pragma unroll
    for (int e = 0; e < V; ++e) u[e] = u[e] * inv * ww[e];
    if (turns) {
      float v[V];
      load_v<T, V>(src + half, v);
      load_v<float, V>(wt + half, ww);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float y = v[e] * inv * ww[e], x = u[e], cs = s_cs[c + e], sn = s_sn[c + e];
        u[e] = x * cs - y * sn;
        v[e] = y * cs + x * sn;
      }
      if (dst != nullptr) store_v<T, V>(dst + half, v);
    }
    if (dst != nullptr) store_v<T, V>(dst, u);
  }
  if (slot < 0) return;
  const T* vs = row + HD + GD;
  T* vd = a.vc + slot * a.vw;
  for (int c = threadIdx.x * V; c < a.vw; c += kThreads * V) {
    if constexpr (V == 8 && sizeof(T) == 2) {
      *reinterpret_cast<uint4*>(vd + c) = *reinterpret_cast<const uint4*>(vs + c);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) vd[c + e] = vs[c + e];
    }
  }
}

// The same with a thread's N items held in registers from the sums on: everything that a row takes is asked for at once (a
// decoded row costs its chain of loads: 16 + 4 heads of 128, one row 3.24 -> 3.09 us, 64 rows 3.52 -> 3.34; 32 + 8 heads 3.97 -> 3.52,
// 4.23 -> 3.88).  Many rows hide each other's chains, and threads without an item or its registers then cost more (us, 512 / 768 / 1024 /
// 2048 rows, above -> here: 8 + 2 heads of 64 3.5 -> 3.5 / 3.6 -> 3.7 / 3.7 -> 3.9 / 4.9 -> 5.5, 16 + 4 of 128 3.9 -> 3.9 / 4.3 -> 4.3 / 4.7 -> 4.9 /
// 6.8 -> 7.1, 32 + 8 of 128 5.1 -> 5.0 / 5.8 -> 5.7 / 6.5 -> 6.9 / 11.2 -> 12.4), unless every thread has its two items (32 + 32 of 128, 4096 rows
// 38.5 -> 30.9) or there are rows enough to read them once (4096 rows of 32 + 8 19.6 -> 18.9, 8192 of 16 + 4 0.98; 3072 1.03).
template <typename T, int N>
__global__ void __launch_bounds__(kThreads) row_norm_rotary_held(const RowRotArgs<T> a) {
  __shared__ float s_cs[kMaxHead / 2], s_sn[kMaxHead / 2];
  __shared__ float s_red[2][kThreads / 64];
  const int t = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int half = a.dims / 2, HD = a.H * a.D, GD = a.G * a.D;
  const long long slot = a.slots[t];
  T* row = a.z + (long long)t * a.ld;
  const float pos = (float)a.positions[t];
  const int turning = half / 8, per = turning + (a.D - a.dims) / 8, items = (a.H + a.G) * per;
  Raw4<T> u4[N][2], v4[N][2], val[2];
  Raw4<float> wu[N][2], wv[N][2];
  float sq = 0.f, sk = 0.f;
  int at[N];                                 // first entry of the item; a key's from HD on
  bool turns[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int it = threadIdx.x + n * kThreads, hd = it / per, j = it - hd * per;
    turns[n] = j < turning;
    at[n] = hd * a.D + (turns[n] ? j * 8 : a.dims + (j - turning) * 8);
    if (it >= items) at[n] = 0;              // (no branch: the first item again, left out of the sums)
    const float* wt = at[n] < HD ? a.wq + at[n] : a.wk + (at[n] - HD);
    const int up = turns[n] ? half : 0;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      u4[n][p].ask(row + at[n] + 4 * p);
      wu[n][p].ask(wt + 4 * p);
      v4[n][p].ask(row + at[n] + up + 4 * p);
      wv[n][p].ask(wt + up + 4 * p);
    }
  }
  const T* vs = row + HD + GD;
  const int c0 = threadIdx.x * 8 < a.vw ? threadIdx.x * 8 : 0;
  val[0].ask(vs + c0);
  val[1].ask(vs + c0 + 4);
  for (int i = threadIdx.x; i < half; i += kThreads) {
    float sn, cs;
    sincosf(pos * a.inv_freq[i], &sn, &cs);
    s_sn[i] = sn * a.amp;
    s_cs[i] = cs * a.amp;
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    float s = 0.f;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      float u[4], v[4];
      u4[n][p].get(u);
      v4[n][p].get(v);
#pragma unroll
      for (int e = 0; e < 4; ++e) s += u[e] * u[e] + (turns[n] ? v[e] * v[e] : 0.f);
    }
    const bool in = (int)threadIdx.x + n * kThreads < items;
    sq += in && at[n] < HD ? s : 0.f;
    sk += in && at[n] >= HD ? s : 0.f;
  }
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if (lane == 0) {
    s_red[0][w] = sq;
    s_red[1][w] = sk;
  }
  __syncthreads();
  sq = (s_red[0][0] + s_red[0][1]) + (s_red[0][2] + s_red[0][3]);
  sk = (s_red[1][0] + s_red[1][1]) + (s_red[1][2] + s_red[1][3]);
  const float iq = 1.f / sqrtf(sq / (float)HD + a.eps), ik = 1.f / sqrtf(sk / (float)GD + a.eps);
#pragma unroll
  for (int n = 0; n < N; ++n) {
    if ((int)threadIdx.x + n * kThreads >= items) continue;
    const bool is_q = at[n] < HD;
    const float inv = is_q ? iq : ik;
    T* dst = is_q ? row + at[n] : (slot < 0 ? nullptr : a.kc + slot * GD + (at[n] - HD));
    const int c = at[n] % a.D;                 // (HD is a multiple of D)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      float u[4], v[4], w1[4], w2[4];
      u4[n][p].get(u);
      wu[n][p].get(w1);
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = u[e] * inv * w1[e];
      if (turns[n]) {
        v4[n][p].get(v);
        wv[n][p].get(w2);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float y = v[e] * inv * w2[e], x = u[e], cs = s_cs[c + 4 * p + e], sn = s_sn[c + 4 * p + e];
          u[e] = x * cs - y * sn;
          v[e] = y * cs + x * sn;
        }
        if (dst != nullptr) store4<T>(dst + half + 4 * p, v);
      }
      if (dst != nullptr) store4<T>(dst + 4 * p, u);
    }
  }
  if (slot < 0) return;
  T* vd = a.vc + slot * a.vw;
  for (int c = threadIdx.x * 8; c < a.vw; c += kThreads * 8) {
    if (c != (int)threadIdx.x * 8) {
      val[0].ask(vs + c);
      val[1].ask(vs + c + 4);
    }
    val[0].put(vd + c);
    val[1].put(vd + c + 4);
  }
}

}  // namespace

extern "C" {

// z [T][>= (H + G) D + vw] (row stride ld); kc / vc rows of G D / vw entries by slot.
hipError_t sm_row_norm_rotary(int dt, void* z, long long ld, const float* wq, const float* wk,
                              const int* positions, const long long* slots, void* kc, void* vc,
                              const float* inv_freq, int T, int H, int G, int D, int vw, int dims,
                              float amp, float eps, hipStream_t st) {
  if (T == 0) return hipSuccess;
  if (H < 1 || G < 1 || D < 1 || D > kMaxHead || vw < 1 || dims < 0 || dims % 2 || dims > D ||
      (dims > 0 && !inv_freq) || ld < (long long)(H + G) * D + vw)
    return hipErrorInvalidValue;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  const int half = dims / 2;
  const auto fits = [&](int v) {
    return half % v == 0 && D % v == 0 && (D - dims) % v == 0 && vw % v == 0 && ld % v == 0 &&
           al(z) && al(kc) && al(vc) && al(wq) && al(wk);
  };
  const int items = (H + G) * ((D - half) / 8);                     // eight entries, and their partners
#define CALL(TT)                                                                                  \
  {                                                                                               \
    RowRotArgs<TT> a{(TT*)z, ld, wq, wk, positions, slots, (TT*)kc, (TT*)vc, inv_freq, H, G, D,   \
                     vw, dims, amp, eps};                                                         \
    if constexpr (sizeof(TT) == 2) {                                                              \
      if (fits(8) && items <= 2 * kThreads && (T <= 512 || items == 2 * kThreads ||             \
                                               (T > 3072 && items > kThreads / 2))) {             \
        if (items <= kThreads) row_norm_rotary_held<TT, 1><<<T, kThreads, 0, st>>>(a);            \
        else row_norm_rotary_held<TT, 2><<<T, kThreads, 0, st>>>(a);                              \
        return hipGetLastError();                                                                 \
      }                                                                                           \
    }                                                                                             \
    if (fits(8)) row_norm_rotary_kernel<TT, 8><<<T, kThreads, 0, st>>>(a);                        \
    else if (fits(4)) row_norm_rotary_kernel<TT, 4><<<T, kThreads, 0, st>>>(a);                   \
    else row_norm_rotary_kernel<TT, 1><<<T, kThreads, 0, st>>>(a);                                \
  }
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

}  // extern "C"
