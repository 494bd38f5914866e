// What a decode step's latent-attention layer does around its attention, three launches instead of six.
//
//   sm_latent_in     a row of z = [query latent Q | latent R | rotated key part Dr]: the cache row as sm_latent_write
//                    forms it, and rms(z[:Q]) * wq.  One workgroup for each of the two, per row: as a wave of a
//                    four-row workgroup the write took 10 us for 64 rows, most of it one wave's chain of loads.
//   sm_latent_query  the query in the latent space, qa[h] = q[h, :D] uk[h] (uk held [H][R][D], so both operands are
//                    rows along D), and the rotated part of every head turned in place.  A wave takes 16
//                    latent columns of a head and 64 rows, fragments straight from L2 (2 MB of weights, 16 KB of
//                    queries a head; nothing is worth staging for one product each), all loads in flight at once.
//   sm_latent_out    the partial sums of sm_latent_attn weighed together (or its finished rows), rounded, and expanded:
//                    o[h] = uv[h] ol[h].  A workgroup takes 16 rows of a head; a wave asks for its 16 output columns'
//                    weights (all of R), joins in the sums, which meet in LDS, and multiplies.
// Bound by latency.  64 rows x 16 heads, D = 128, R = 512, in a decode step, us: write and norm 10.1 + 4.5 -> 6.2; batched
// library product and rotation 5.1 + 4.5 -> 7.0; sums of 8 splits and library product 4.9 + 12.7 -> 6.5 (10.9 with
// 16 rows a workgroup and sums of splits without keys).
#include "mma.h"

using namespace lumen;

namespace {

constexpr int kThreads = 256;

template <typename T> struct InArgs {
  const T* z; long long ldz;
  const float *wq, *wn, *inv_freq;
  const int* positions; const long long* slots;
  T *cache, *vt, *qn;
  int bs, Q, R, Dr, dims;
  float eps;
};

template <typename T>
__global__ void __launch_bounds__(kThreads) latent_in_kernel(const InArgs<T> a) {
  __shared__ float s_red[kThreads / 64];
  const int t = blockIdx.x, tid = threadIdx.x;
  const T* zr = a.z + (long long)t * a.ldz;
  const bool query = blockIdx.y == 1;
  const long long s = query ? 0 : a.slots[t];
  if (s < 0) return;                                   // (the whole workgroup)
  const T* x = query ? zr : zr + a.Q;
  const int n = query ? a.Q : a.R;
  const float* w = query ? a.wq : a.wn;
  float ss = 0.f;
  for (int c = tid; c < n; c += kThreads) {
    const float v = to_f32(x[c]);
    ss += v * v;
  }
  const float inv = 1.f / sqrtf(block_sum<kThreads>(ss, s_red) / (float)n + a.eps);
  T* dst = query ? a.qn + (long long)t * a.Q : a.cache + s * (a.R + a.Dr);
  T* dt = !query && a.vt ? a.vt + (s / a.bs) * (long long)a.R * a.bs + s % a.bs : nullptr;
  for (int c = tid; c < n; c += kThreads) {
    const T v = from_f32<T>(to_f32(x[c]) * inv * w[c]);
    dst[c] = v;
    if (dt) dt[(long long)c * a.bs] = v;
  }
  if (query) return;
  const float pos = (float)a.positions[t];
  for (int pr = tid; pr < a.dims / 2; pr += kThreads) {
    float sn, cs;
    sincosf(pos * a.inv_freq[pr], &sn, &cs);
    const float u = to_f32(x[a.R + 2 * pr]), v = to_f32(x[a.R + 2 * pr + 1]);
    dst[a.R + 2 * pr] = from_f32<T>(u * cs - v * sn);
    dst[a.R + 2 * pr + 1] = from_f32<T>(v * cs + u * sn);
  }
  for (int c = a.dims + tid; c < a.Dr; c += kThreads) dst[a.R + c] = x[a.R + c];
}

// 16-bit rows of up to 2048 aligned entries: eight a thread, everything asked for at once (1536 + 512 + 64 entries, 64 rows
// 3.73 -> 3.12 us, 4096 rows 22.8 -> 19.0)
template <typename T>
__global__ void __launch_bounds__(kThreads) latent_in_wide(const InArgs<T> a) {
  __shared__ float s_red[kThreads / 64];
  const int t = blockIdx.x, c = 8 * threadIdx.x;
  const T* zr = a.z + (long long)t * a.ldz;
  const bool query = blockIdx.y == 1;
  const long long s = query ? 0 : a.slots[t];
  const T* x = query ? zr : zr + a.Q;
  const int n = query ? a.Q : a.R, pr = threadIdx.x;
  const bool on = c < n, turns = !query && pr < a.dims / 2;
  float v[8], w[8], ss = 0.f, u0 = 0.f, u1 = 0.f, f = 0.f;
  load8<T>(x + (on ? c : 0), v);
  load8<float>((query ? a.wq : a.wn) + (on ? c : 0), w);
  if (turns) {
    u0 = to_f32(x[a.R + 2 * pr]);
    u1 = to_f32(x[a.R + 2 * pr + 1]);
    f = (float)a.positions[t] * a.inv_freq[pr];
  }
  if (s < 0) return;                                   // (the whole workgroup)
#pragma unroll
  for (int e = 0; e < 8; ++e) ss += on ? v[e] * v[e] : 0.f;
  const float inv = 1.f / sqrtf(block_sum<kThreads>(ss, s_red) / (float)n + a.eps);
  T* dst = query ? a.qn + (long long)t * a.Q : a.cache + s * (a.R + a.Dr);
  if (on) {
    T o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = from_f32<T>(v[e] * inv * w[e]);
    *reinterpret_cast<uint4*>(dst + c) = *reinterpret_cast<const uint4*>(o);
    if (!query && a.vt) {
      T* dt = a.vt + (s / a.bs) * (long long)a.R * a.bs + s % a.bs;
#pragma unroll
      for (int e = 0; e < 8; ++e) dt[(long long)(c + e) * a.bs] = o[e];
    }
  }
  if (query) return;
  if (turns) {
    float sn, cs;
    sincosf(f, &sn, &cs);
    dst[a.R + 2 * pr] = from_f32<T>(u0 * cs - u1 * sn);
    dst[a.R + 2 * pr + 1] = from_f32<T>(u1 * cs + u0 * sn);
  }
  for (int i = a.dims + threadIdx.x; i < a.Dr; i += kThreads) dst[a.R + i] = x[a.R + i];
}

template <typename T> struct QueryArgs {
  T* q; long long ldq; int ldh;             // rows; head h of a row at column h * ldh
  const T* w;                               // [H][R][D]
  T* out;                                   // [H][Tn][R]
  int Tn, R, off, dims;                     // rotated part: columns off .. off + dims - 1 of a head
  const float* inv_freq; const int* positions;
};

// KS: steps of 32 along D
template <typename T, int KS>
__global__ void __launch_bounds__(256) latent_query_kernel(const QueryArgs<T> a) {
  constexpr int D = 32 * KS;
  const int h = blockIdx.y, t0 = blockIdx.z * 64;
  if ((int)blockIdx.x * 64 >= a.R) {                   // the last column of workgroups: the rotation
    const int half = a.dims / 2, n = min(64, a.Tn - t0) * half;
    for (int i = threadIdx.x; i < n; i += 256) {
      const int t = t0 + i / half, pr = i % half;
      float sn, cs;
      sincosf((float)a.positions[t] * a.inv_freq[pr], &sn, &cs);
      T* p = a.q + (long long)t * a.ldq + h * a.ldh + a.off + 2 * pr;
      const float u = to_f32(p[0]), v = to_f32(p[1]);
      p[0] = from_f32<T>(u * cs - v * sn);
      p[1] = from_f32<T>(v * cs + u * sn);
    }
    return;
  }
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int r0 = blockIdx.x * 64 + 16 * (threadIdx.x >> 6);
  const T* wr = a.w + ((long long)h * a.R + r0 + lr) * D + 8 * lg;
  uint4 x[KS], y[4][KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) x[s] = *reinterpret_cast<const uint4*>(wr + 32 * s);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (t0 + 16 * j < a.Tn) {
      const T* qr = a.q + (long long)min(t0 + 16 * j + lr, a.Tn - 1) * a.ldq + h * a.ldh + 8 * lg;
#pragma unroll
      for (int s = 0; s < KS; ++s) y[j][s] = *reinterpret_cast<const uint4*>(qr + 32 * s);
    }
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (t0 + 16 * j < a.Tn) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s) c = Mfma<T>::run(x[s], y[j][s], c);
      const int t = t0 + 16 * j + lr;                  // lane (lr, lg): row t, columns r0 + 4 lg ..
      if (t < a.Tn)
        *reinterpret_cast<uint2*>(a.out + ((long long)h * a.Tn + t) * a.R + r0 + 4 * lg) =
            make_uint2(pk2<T>(c[0], c[1]), pk2<T>(c[2], c[3]));
    }
}

template <typename T> struct OutArgs {
  const float *ml, *part; int nsplit;       // of sm_latent_attn; nsplit 1: x
  const T* x; long long xr, xh;             // finished rows [Tn][H][R] at these strides
  const T* gate; long long gater;
  const T* uv;                              // [H][Dv][R]
  T* o; long long orow, oh;
  int Tn, H, Dv, rows;                      // rows: of a workgroup
};

// KS: steps of 32 along R; a wave per 16 of Dv
template <typename T, int KS>
__global__ void __launch_bounds__(1024) latent_out_kernel(const OutArgs<T> a) {
  constexpr int R = 32 * KS, LD = R + 8;               // (16-byte pieces of 16 rows: no bank conflicts)
  __shared__ __attribute__((aligned(16))) T s_x[16 * LD];
  __shared__ float s_w[16][64];
  __shared__ int s_n[16];
  const int h = blockIdx.y, t0 = blockIdx.x * a.rows, n = min(a.rows, a.Tn - t0);
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4, w = tid >> 6;
  uint4 u[KS];
  const T* ur = a.uv + ((long long)h * a.Dv + 16 * w + lr) * R + 8 * lg;
#pragma unroll
  for (int s = 0; s < KS; ++s) u[s] = *reinterpret_cast<const uint4*>(ur + 32 * s);
  if (a.nsplit > 1) {
    for (int i = w; i < n; i += (int)blockDim.x >> 6) {    // lane s weighs split s
      const long long base = ((long long)(t0 + i) * a.H + h) * a.nsplit;
      const float ms = lane < a.nsplit ? a.ml[2 * (base + lane)] : -INFINITY;
      const float ls = lane < a.nsplit ? a.ml[2 * (base + lane) + 1] : 0.f;
      const int live = __popcll(__ballot(lane < a.nsplit && !(ls < 0.f)));   // (the last ones had no key: no sums)
      if (lane == 0) s_n[i] = live;
      const float M = wave_max(ms);
      const float e = ms == -INFINITY ? 0.f : expf(ms - M);
      float L = wave_sum(ls * e);
      if (a.gate != nullptr) L *= 1.f + expf(-to_f32(a.gate[(long long)(t0 + i) * a.gater + h]));   // / sigmoid
      s_w[i][lane] = e / L;
    }
    __syncthreads();
  }
  for (int x = tid; x < n * (R / 4); x += blockDim.x) {
    const int i = x / (R / 4), c = 4 * (x % (R / 4));
    if (a.nsplit > 1) {
      const float* p = a.part + ((long long)(t0 + i) * a.H + h) * a.nsplit * R + c;
      float v[4] = {0.f, 0.f, 0.f, 0.f};
      const auto add = [&](const float4& y, float k) {
        v[0] += y.x * k; v[1] += y.y * k; v[2] += y.z * k; v[3] += y.w * k;
      };
      const int live = s_n[i];
      int s = 0;
      for (; s + 4 <= live; s += 4) {
        float4 y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) y[q] = *reinterpret_cast<const float4*>(p + (long long)(s + q) * R);
#pragma unroll
        for (int q = 0; q < 4; ++q) add(y[q], s_w[i][s + q]);
      }
      for (; s < live; ++s) add(*reinterpret_cast<const float4*>(p + (long long)s * R), s_w[i][s]);
      store4<T>(s_x + i * LD + c, v);
    } else {
      *reinterpret_cast<uint2*>(s_x + i * LD + c) =
          *reinterpret_cast<const uint2*>(a.x + (long long)(t0 + i) * a.xr + h * a.xh + c);
    }
  }
  __syncthreads();
  f32x4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
  const T* xr = s_x + min(lr, n - 1) * LD + 8 * lg;
#pragma unroll
  for (int s = 0; s < KS; s += 2) {
    c0 = Mfma<T>::run(u[s], *reinterpret_cast<const uint4*>(xr + 32 * s), c0);
    c1 = Mfma<T>::run(u[s + 1], *reinterpret_cast<const uint4*>(xr + 32 * s + 32), c1);
  }
  c0 += c1;
  if (lr < n)                                          // lane (lr, lg): row t0 + lr, columns 16 w + 4 lg ..
    *reinterpret_cast<uint2*>(a.o + (long long)(t0 + lr) * a.orow + h * a.oh + 16 * w + 4 * lg) =
        make_uint2(pk2<T>(c0[0], c0[1]), pk2<T>(c0[2], c0[3]));
}

}  // namespace

extern "C" {

// z [rows][>= Q + R + Dr] at stride ldz, any 16-bit or fp32 type; qn [rows][Q]; the rest as sm_latent_write.
hipError_t sm_latent_in(int dt, const void* z, long long ldz, const float* wq, void* qn, const float* wn,
                        const float* inv_freq, const int* positions, const long long* slots, void* cache, void* vt,
                        int bs, int rows, int Q, int R, int Dr, int dims, float eps, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (rows < 0 || Q < 1 || R < 1 || Dr < 0 || dims < 0 || dims % 2 || dims > Dr || bs < 1 || ldz < Q + R + Dr)
    return hipErrorInvalidValue;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  const bool wide = dt != kF32 && Q % 8 == 0 && R % 8 == 0 && Dr % 8 == 0 && Q <= 8 * kThreads && R <= 8 * kThreads &&
                    dims / 2 <= kThreads && ldz % 8 == 0 && al(z) && al(wq) && al(wn) && al(qn) && al(cache);
  if (wide) {
#define WIDE(T)                                                                                                 \
  latent_in_wide<T><<<dim3(rows, 2), kThreads, 0, st>>>(InArgs<T>{(const T*)z, ldz, wq, wn, inv_freq, positions, \
                                                          slots, (T*)cache, (T*)vt, (T*)qn, bs, Q, R, Dr, dims, eps})
    if (dt == kBF16) WIDE(bf16);
    else if (dt == kF16) WIDE(fp16);
    else return hipErrorInvalidValue;
#undef WIDE
    return hipGetLastError();
  }
#define CALL(T)                                                                                                 \
  latent_in_kernel<T><<<dim3(rows, 2), kThreads, 0, st>>>(InArgs<T>{(const T*)z, ldz, wq, wn, inv_freq, positions, \
                                                            slots, (T*)cache, (T*)vt, (T*)qn, bs, Q, R, Dr, dims, eps})
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

// q [rows] at stride ldq, heads at stride ldh (both % 8); w [H][R][D]; out [H][rows][R].  16-bit, D in 64, 128, 192 or
// 256, R % 64 == 0, 16-byte bases; the rotated part, if any, lies behind a head's first D columns.
hipError_t sm_latent_query(int dt, void* q, long long ldq, int ldh, const void* w, void* out, int rows, int H, int D,
                           int R, int off, int dims, const float* inv_freq, const int* positions, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (rows < 0 || rows > 64 * 65535 || H < 1 || H > 65535 || R < 64 || R % 64 || ldh < D || ldh % 8 || ldq % 8 ||
      ldq < (long long)(H - 1) * ldh + D || dims < 0 || dims % 2 ||
      (dims > 0 && (off < D || off + dims > ldh || !inv_freq || !positions ||
                    ldq < (long long)(H - 1) * ldh + off + dims)) ||
      ((uintptr_t)q | (uintptr_t)w | (uintptr_t)out) % 16 || (dt != kBF16 && dt != kF16))
    return hipErrorInvalidValue;
  const dim3 grid(R / 64 + (dims > 0), H, (rows + 63) / 64);
#define GO(T, KS)                                                                                                   \
  latent_query_kernel<T, KS><<<grid, 256, 0, st>>>(QueryArgs<T>{(T*)q, ldq, ldh, (const T*)w, (T*)out, rows, R, off, \
                                                                 dims, inv_freq, positions})
#define GO_T(T)                            \
  if (D == 64) GO(T, 2);                   \
  else if (D == 128) GO(T, 4);             \
  else if (D == 192) GO(T, 6);             \
  else if (D == 256) GO(T, 8);             \
  else return hipErrorInvalidValue
  if (dt == kBF16) { GO_T(bf16); } else { GO_T(fp16); }
#undef GO_T
#undef GO
  return hipGetLastError();
}

// The rows of sm_latent_attn: ml, part of nsplit > 1 splits (gate as there), or with nsplit 1 x at strides xr, xh (% 4, 8-byte
// base).  uv [H][Dv][R], Dv % 16 == 0 up to 256, R 64, 128, 256 or 512; o at strides orow, oh (% 4, 8-byte base).
hipError_t sm_latent_out(int dt, const float* ml, const float* part, int nsplit, const void* x, long long xr,
                         long long xh, const void* gate, long long gater, const void* uv, void* o, long long orow,
                         long long oh, int rows, int H, int Dv, int R, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (rows < 0 || H < 1 || H > 65535 || Dv < 16 || Dv % 16 || Dv > 256 || nsplit < 1 || nsplit > 64 || !uv || !o ||
      (uintptr_t)uv % 16 || (uintptr_t)o % 8 || orow % 4 || oh % 4 || (dt != kBF16 && dt != kF16) ||
      (nsplit > 1 ? !ml || !part || (uintptr_t)part % 16 : !x || (uintptr_t)x % 8 || xr % 4 || xh % 4))
    return hipErrorInvalidValue;
  // rows of a workgroup: 16, fewer while all of them have a CU each, as the sums of 16 rows and a head's weights are 300 KB to
  // fetch for one (16 rows -> fewer, us with the attention: 8 rows of 16 heads 16.7 -> 14.1, 16 of 8 18.8 -> 13.8, 48 of 16 23.2 -> 19.3; more than
  // one a CU fetch a head's weights again: two of 4 rows 48 of 16 22.8, 48 rows of 32 heads over 128, 40 keys, 8.5 -> 10.6)
  int per = 16;
  while (per > 1 && (long long)((rows + per / 2 - 1) / (per / 2)) * H <= 256) per /= 2;
  const dim3 grid((rows + per - 1) / per, H);
#define GO(T, KS)                                                                                                 \
  latent_out_kernel<T, KS><<<grid, 4 * Dv, 0, st>>>(OutArgs<T>{ml, part, nsplit, (const T*)x, xr, xh, (const T*)gate, \
                                                               gater, (const T*)uv, (T*)o, orow, oh, rows, H, Dv, per})
#define GO_T(T)                            \
  if (R == 64) GO(T, 2);                   \
  else if (R == 128) GO(T, 4);             \
  else if (R == 256) GO(T, 8);             \
  else if (R == 512) GO(T, 16);            \
  else return hipErrorInvalidValue
  if (dt == kBF16) { GO_T(bf16); } else { GO_T(fp16); }
#undef GO_T
#undef GO
  return hipGetLastError();
}

}  // extern "C"
