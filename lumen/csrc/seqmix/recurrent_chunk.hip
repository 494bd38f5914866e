// The `wkv` and generalised-delta recurrences of recurrent.hip over a step's prompt portions, sixteen
// tokens at a time.  With w_t the decays of token t (one per key channel), P_t = w_1 ... w_t within the
// chunk, Q_t = w_(t+1) ... w_16, S_0 the state before it, and for the delta rule b_t = a_t un_t:
//   delta  c_t = un_t^T S_(t-1),   S_t = diag(w_t) S_(t-1) - b_t c_t^T + k_t v_t^T,   o_t = S_t^T r_t
//   wkv    o_t = S_(t-1)^T r_t + (sum_i r u k) v_t,   S_t = diag(w_t) S_(t-1) + k_t v_t^T
// and the scaled rows  U_t = un_t P_(t-1),  R_t = r_t P_t (wkv: r_t P_(t-1)),  K_t = k_t Q_t,  B_t = b_t Q_t
// and their quotients U' = U / P_16, R' = R / P_16, all of it is matrix products:
//   C = (I + strict(U' B^T))^-1 (U S_0 + strict(U' K^T) V)
//   O = R S_0 + lower(R' K^T) V - lower(R' B^T) C      (wkv: strict, its diagonal the bonus; no C)
//   S' = P_16 S_0 + K^T V - B^T C
// Rows past a chunk's end (or a portion's) enter with w = 1 and zeros, so they change nothing.
//
// What bounded the token-by-token kernel: every lane re-read its slice of five vectors from LDS for
// every token (40 16-byte reads per wave and token at head size 128, ~2 us a token whatever else it did)
// on segments x heads workgroups.  Here a workgroup owns 64 value columns of a (segment, head), a wave
// 16 of them with its [D x 16] slice of the state in accumulator registers for the whole portion: the
// 16x16x4 product's accumulator register e of lane group g holds row 4 g + e, which IS the right operand
// of a product over the inner rows {4 g + e}, so S, V, C and U S_0 never pass through LDS; the left
// operands are staged there once for the four waves and read 16 bytes at a time.  All products are
// fp32 matrix instructions; decays are fp32, their products fp64.
// The read-outs leave in fp32; the per-head norm and gate follow in gated_rms (rms_group.hip).
// Measured (8 portions of 512 tokens, width 2048, bf16; the norm kernel's 17 us included): delta, 16 heads
// of 128: 1000 -> 310 us; wkv, 32 heads of 64: 460 -> 119 us.  A chunk is now a chain of three barriers
// -- decays and sums, scaled rows, products -- with one wave per SIMD at this size.
// Error against float64 (512 tokens, heads of 32 - 256): the read-outs are as far off as the serial walk's
// (1.66e-3, the bf16 result's rounding), the state a little less (delta 0.86e-7, serial 0.88e-7; wkv 0.60e-7,
// serial 0.62e-7).  That takes the decays' products in float64 (in fp32: + 0.1e-7) and care with the sums
// (see the state's update; term by term 1.4e-7 and 0.9e-7), which cost 20 us of the delta scan.
//
// Range: P_t and 1 / P_16 must stay finite, and so must the masked entries' factors.  A wkv chunk ends
// before the token that would take some channel's P below 2^-100, so a decay beyond that (0 too) is alone in
// its chunk, where nothing is divided by it; the delta rule's decays, at least e^-decay_scale per token,
// stay above 2^-70.  r and k that scaled rows could not hold as normal numbers (kLarge, kTiny*), infinities and
// NaN run one token at a time, so that earlier tokens stay as they are; wkv values below kSmall make the
// chunk end at 2^-40.  A chunk of one token costs what one of sixteen does: decays up to e^-50 a token (wkv,
// 8 x 512 tokens, 32 heads of 64, log decays -e^N(1, 1) at the fast end) take 770 us, the
// serial walk 460.
#include "seqmix.h"

using namespace lumen;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kC = 16;                 // tokens per chunk
constexpr int LP = 20;                 // row stride of the chunk matrices in LDS
constexpr float kMinP = 0x1p-100f;     // smallest product of a chunk's decays, and a group's share of it
template <int NG> constexpr float kGroupP() {
  return NG == 1 ? 0x1p-100f : NG == 2 ? 0x1p-50f : NG == 4 ? 0x1p-25f : 0x1p-12f;
}

// |x| as bits, whose order is that of the values (infinities and NaN last)
__device__ __forceinline__ unsigned mag(float x) { return __builtin_bit_cast(unsigned, x) & 0x7fffffffu; }
// The scaled rows of r and k have to stay normal numbers (2^-126), and their products finite.  Values above
// kLarge, or (0 apart) below the smallest that a chunk's decays leave normal, go one token at a time;
// wkv values below kSmall (2^-24, the end of fp16) let the decays reach kSmallP only.
constexpr unsigned kInf = 0x7f800000u, kLarge = 0x49800000u;       // 2^20
constexpr unsigned kSmall = 0x33800000u;                           // 2^-24: x 2^-100 = 2^-124
constexpr unsigned kTinyWkv = 0x15000000u, kTinyDelta = 0x24000000u;   // 2^-85 x 2^-40, 2^-55 x 2^-70
constexpr float kSmallP = 0x1p-40f;

template <typename T> struct ScanArgs {
  const T *r, *k, *v, *wl, *al;        // rows of H * D; al: removal rates (delta)
  long long ldr, ldk, ldv, ldw, lda;
  const float *w0, *ub;                // decay offsets; u (wkv) / removal-rate bias (delta) [H * D]
  float* state;                        // [slots][H][D][D]
  float* out;                          // [T][H * D]
  const int *cu, *slot, *start;
  int H, D;
  float decay_scale, key_eps;
};

template <int CTRL> __device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL,
                                                               0xF, 0xF, false));
}
__device__ __forceinline__ float lane_f(float v, int l) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ float sum16(float v) {        // over the 16 lanes of a row
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  v += dpp<0x141>(v);
  return v + dpp<0x140>(v);
}

// KB: key channels in blocks of 16
template <typename T, int KB, bool DELTA>
__global__ void __launch_bounds__(256)
scan_chunk_kernel(const ScanArgs<T> a) {
  constexpr int DKP = 16 * KB, LK = DKP + 4;
  constexpr int NG = 256 / DKP, TG = kC / NG;            // staging: token groups, tokens of each
  constexpr int NM = DELTA ? 4 : 1;
  __shared__ __attribute__((aligned(16))) float s_r[kC * LK], s_k[kC * LK];
  __shared__ __attribute__((aligned(16))) float s_u[DELTA ? kC * LK : 4], s_b[DELTA ? kC * LK : 4];
  __shared__ __attribute__((aligned(16))) float s_m[NM][kC * LP];
  __shared__ __attribute__((aligned(16))) float s_P[DKP], s_iP[DKP], s_red[kC][KB];
  __shared__ double s_gp[NG][DKP];
  __shared__ float s_tok[kC];
  __shared__ int s_n[2], s_low[2], s_small[2];
  const int sg = blockIdx.x, hd = blockIdx.y;
  const int r0 = a.cu[sg], len = a.cu[sg + 1] - r0;
  if (len <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lg = lane >> 4;
  const int D = a.D, col0 = hd * D;
  const int j = (blockIdx.z * 4 + w) * 16 + lr;                  // this lane's value column
  const bool on = j < D;
  const int ch = tid % DKP, tg = tid / DKP;                      // staging: channel, token group
  const bool chan = ch < D;
  const float w0 = chan ? a.w0[col0 + ch] : 0.f, ub = chan ? a.ub[col0 + ch] : 0.f;

  f32x4 S[KB];
  float* st = a.state + ((long long)a.slot[sg] * a.H + hd) * D * D + j;
  const bool fresh = a.start[sg] == 0;
#pragma unroll
  for (int b = 0; b < KB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 16 * b + 4 * lg + e;
      S[b][e] = (!fresh && on && i < D) ? st[(long long)i * D] : 0.f;
    }

  // the chunk at t0, as loaded: this thread's channel of its tokens, this lane's values (4 lg + e).  Rows
  // past the portion repeat its last one, channels past D the last one: blanked where they are used.
  T pr[TG], pk[TG], pw[TG], pa[TG], pv[4];
  const int chc = min(ch, D - 1), jc = min(j, D - 1);
  // the token of a lane's e-th value: an inner index of every product with V
  const auto tok_of = [&](int e) { return DELTA ? 4 * lg + e : 4 * e + lg; };
  // row t + i of `base`'s chunk at t0, column c (uniform base, 32-bit byte offset from the chunk's first row,
  // so the rows that are left count up to a chunk's; i known when compiled)
  const auto get = [&](const T* base, long long ld, int t0, int t, int i, int c)
                       __attribute__((always_inline)) {
    const unsigned step = (unsigned)ld, last = (unsigned)min(len - 1 - t0, kC - 1) * step;
    const unsigned at = min((unsigned)t * step + (unsigned)i * step, last) + (unsigned)c;
    return *reinterpret_cast<const T*>(
        reinterpret_cast<const char*>(base + (long long)(r0 + t0) * ld + col0) + at * (unsigned)sizeof(T));
  };
  const auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < TG; ++q) {
      pr[q] = get(a.r, a.ldr, t0, tg * TG, q, chc);
      pk[q] = get(a.k, a.ldk, t0, tg * TG, q, chc);
      pw[q] = get(a.wl, a.ldw, t0, tg * TG, q, chc);
      if (DELTA) pa[q] = get(a.al, a.lda, t0, tg * TG, q, chc);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) pv[e] = get(a.v, a.ldv, t0, tok_of(0), DELTA ? e : 4 * e, jc);
  };
  if (tid < 2) { s_n[tid] = kC; s_low[tid] = s_small[tid] = 0; }
  fetch(0);
  __syncthreads();
  for (int t0 = 0, par = 0; t0 < len; par ^= 1) {
    // ---- decays, removal rates, the channel sums of every token ----
    float rv[TG], kv[TG], wv[TG], av[TG];
    {
      unsigned top = 0u, low = ~0u, lim = 0u;   // r and k: largest, smallest - 1; the others: largest
      double gp = 1.;
#pragma unroll
      for (int q = 0; q < TG; ++q) {
        const bool live = t0 + tg * TG + q < len && chan;
        rv[q] = chan ? to_f32(pr[q]) : 0.f;
        kv[q] = chan ? to_f32(pk[q]) : 0.f;
        const float zl = to_f32(pw[q]), z = zl + w0;
        const float d = DELTA ? expf(-a.decay_scale * sigmoid_f(z)) : expf(-expf(z));
        wv[q] = live ? d : 1.f;
        gp *= wv[q];
        const unsigned mr = mag(rv[q]), mk = mag(kv[q]);
        top = max(top, max(mr, mk));
        low = min(low, min(mr - 1u, mk - 1u));   // (0 is as good as large)
        lim = max(lim, mag(zl));
        if (DELTA) {
          const float al = to_f32(pa[q]);
          lim = max(lim, mag(al));
          av[q] = live ? sigmoid_f(al + ub) : 0.f;
        }
        const float s = sum16(DELTA ? kv[q] * kv[q] : rv[q] * ub * kv[q]);
        if (lr == 0) s_red[tg * TG + q][ch >> 4] = s;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) lim = max(lim, mag(to_f32(pv[e])));
      s_gp[tg][ch] = gp;
      if (top > kLarge || low < (DELTA ? kTinyDelta : kTinyWkv) - 1u || lim >= kInf)
        atomicMin(&s_n[par], 1);
      if (!DELTA && low < kSmall - 1u) s_small[par] = 1;
      // no group's product below its share of the range: no chunk product leaves it
      if (!DELTA && !(gp >= kGroupP<NG>())) s_low[par] = 1;
    }
    __syncthreads();
    // the tokens' sums, a lane for each of the wave's, handed round
    float tok[TG];
    {
      float v = 0.f;
#pragma unroll
      for (int b = 0; b < KB; ++b) v += s_red[tg * TG + lane % TG][b];
      if (DELTA) v = 1.f / sqrtf(v + a.key_eps);
#pragma unroll
      for (int q = 0; q < TG; ++q) {
        tok[q] = lane_f(v, q);
        if (DKP < 64) tok[q] = lane < 32 ? tok[q] : lane_f(v, 32 + q);
      }
    }
    if (s_n[par] < kC || s_low[par] || s_small[par]) {   // a shorter chunk (one decision for the workgroup)
      if (!DELTA) {                      // where does a channel's product leave the range?
        const float least = s_small[par] ? kSmallP : kMinP;
        double p = 1.;
        for (int g = 0; g < tg; ++g) p *= s_gp[g][ch];
#pragma unroll
        for (int q = 0; q < TG; ++q) {
          p *= wv[q];
          if (p < least && tg * TG + q > 0) atomicMin(&s_n[par], tg * TG + q);
        }
      }
      __syncthreads();
      double p = 1.;                     // the rows that are left for the next chunk decay nothing
#pragma unroll
      for (int q = 0; q < TG; ++q) {
        if (tg * TG + q >= s_n[par]) wv[q] = 1.f;
        p *= wv[q];
      }
      s_gp[tg][ch] = p;
      __syncthreads();
    }
    const int n = __builtin_amdgcn_readfirstlane(min(s_n[par], len - t0));
    if (tid == 0) { s_n[par ^ 1] = kC; s_low[par ^ 1] = s_small[par ^ 1] = 0; }
    // ---- the scaled rows ----
    double P = 1., Q = 1.;               // decay of the token groups before and after this one
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const double q = s_gp[g][ch];
      P *= g < tg ? q : 1.;
      Q *= g > tg ? q : 1.;
    }
#pragma unroll
    for (int q = TG - 1; q >= 0; --q) {  // decayed to the chunk's end
      const int at = (tg * TG + q) * LK + ch;
      const bool live = tg * TG + q < n;
      s_k[at] = live ? (float)(kv[q] * Q) : 0.f;
      if (DELTA) s_b[at] = live ? (float)(kv[q] * tok[q] * av[q] * Q) : 0.f;
      Q *= wv[q];
    }
#pragma unroll
    for (int q = 0; q < TG; ++q) {       // decayed from the chunk's start
      const int t = tg * TG + q, at = t * LK + ch;
      const bool live = t < n;
      const float P0 = (float)P;
      P *= wv[q];
      s_r[at] = live ? rv[q] * (DELTA ? (float)P : P0) : 0.f;
      if (DELTA) s_u[at] = live ? kv[q] * tok[q] * P0 : 0.f;
      else if (ch == 0) s_tok[t] = tok[q];
    }
    if (tg == NG - 1) {
      s_P[ch] = (float)P;
      s_iP[ch] = 1.f / (float)P;                // (one token: only entries that are masked out see it)
    }
    f32x4 V;
#pragma unroll
    for (int e = 0; e < 4; ++e) V[e] = tok_of(e) < n ? to_f32(pv[e]) : 0.f;
    const int next = t0 + n;
    if (next < len) fetch(next);         // in flight during the products
    __syncthreads();
    // ---- chunk matrices, one per wave: U K^T, U B^T (then inverted), R K^T, R B^T ----
    if (w < NM) {
      const float* x = (DELTA && w < 2 ? s_u : s_r) + lr * LK + 4 * lg;
      const float* y = (DELTA && (w & 1) ? s_b : s_k) + lr * LK + 4 * lg;
      f32x4 c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        const float4 xa = *reinterpret_cast<const float4*>(x + 16 * b);
        const float4 ya = *reinterpret_cast<const float4*>(y + 16 * b);
        const float4 ip = *reinterpret_cast<const float4*>(&s_iP[16 * b + 4 * lg]);
        c[0] = mma(xa.x * ip.x, ya.x, c[0]);
        c[1] = mma(xa.y * ip.y, ya.y, c[1]);
        c[2] = mma(xa.z * ip.z, ya.z, c[2]);
        c[3] = mma(xa.w * ip.w, ya.w, c[3]);
      }
      const f32x4 acc = (c[0] + c[1]) + (c[2] + c[3]);
      float* m = s_m[w];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * lg + e;        // row: token t; column lr: token s
        float z = i < n && (DELTA && w >= 2 ? lr <= i : lr < i) ? acc[e] : 0.f;
        if (!DELTA && lr == i && i < n) z = s_tok[i];
        m[i * LP + lr] = z;
      }
      if (DELTA && w == 1) {             // (I + M)^-1, a lane per column
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float t[kC];
#pragma unroll
        for (int i = 0; i < kC; ++i) {
          float s = 0.f;
#pragma unroll
          for (int q = 0; q < kC; q += 4)
            if (q < i) {
              const float4 xr = *reinterpret_cast<const float4*>(&m[i * LP + q]);
              s += xr.x * t[q];
              if (q + 1 < i) s += xr.y * t[q + 1];
              if (q + 2 < i) s += xr.z * t[q + 2];
              if (q + 3 < i) s += xr.w * t[q + 3];
            }
          t[i] = i == lr ? 1.f : i > lr ? -s : 0.f;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < 16) {
#pragma unroll
          for (int i = 0; i < kC; ++i) m[i * LP + lr] = t[i];
        }
      }
    }
    // ---- what the old state gives (four sums each: a quarter of the chain, and of its error) ----
    f32x4 O, C = {0.f, 0.f, 0.f, 0.f};
    {
      f32x4 o[4], c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = c[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        const float4 x = *reinterpret_cast<const float4*>(&s_r[lr * LK + 16 * b + 4 * lg]);
        o[0] = mma(x.x, S[b][0], o[0]);
        o[1] = mma(x.y, S[b][1], o[1]);
        o[2] = mma(x.z, S[b][2], o[2]);
        o[3] = mma(x.w, S[b][3], o[3]);
        if (DELTA) {
          const float4 u = *reinterpret_cast<const float4*>(&s_u[lr * LK + 16 * b + 4 * lg]);
          c[0] = mma(u.x, S[b][0], c[0]);
          c[1] = mma(u.y, S[b][1], c[1]);
          c[2] = mma(u.z, S[b][2], c[2]);
          c[3] = mma(u.w, S[b][3], c[3]);
        }
      }
      O = (o[0] + o[1]) + (o[2] + o[3]);
      if (DELTA) C = (c[0] + c[1]) + (c[2] + c[3]);
    }
    __syncthreads();                     // chunk matrices complete
    const auto small = [&](int m, const f32x4& x, f32x4 acc) {
      float4 y;
      if (DELTA) y = *reinterpret_cast<const float4*>(&s_m[m][lr * LP + 4 * lg]);
      else {
        const float* r = &s_m[m][lr * LP + lg];
        y = make_float4(r[0], r[4], r[8], r[12]);
      }
      acc = mma(y.x, x[0], acc);
      acc = mma(y.y, x[1], acc);
      acc = mma(y.z, x[2], acc);
      return mma(y.w, x[3], acc);
    };
    if (DELTA) {
      C = small(0, V, C);
#pragma unroll
      for (int e = 0; e < 4; ++e) C[e] = 4 * lg + e < n ? C[e] : 0.f;
      C = small(1, C, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int e = 0; e < 4; ++e) C[e] = 4 * lg + e < n ? -C[e] : 0.f;
      O = small(3, C, small(2, V, O));
    } else {
      O = small(0, V, O);
    }
    if (on) {
      float* o = a.out + (long long)(r0 + t0) * a.H * D + col0;
      const unsigned HD = (unsigned)(a.H * D);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (4 * lg + e < n) o[(unsigned)(4 * lg) * HD + (unsigned)e * HD + (unsigned)j] = O[e];
    }
    // ---- the state moves on.  wkv: decayed, then the tokens' terms in order, the last (and least decayed)
    // ones last, so that a fast channel sees few roundings.  Delta: what the chunk adds is summed apart, in
    // fours, and meets the state in one rounding; added term by term to it the error was 1.4 - 1.6 times
    // the serial walk's ----
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const float4 P = *reinterpret_cast<const float4*>(&s_P[16 * b + 4 * lg]);
      const float p[4] = {P.x, P.y, P.z, P.w};
      if (DELTA) {
        f32x4 d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          d[e] = mma(s_k[(4 * lg + e) * LK + 16 * b + lr], V[e], zero) +
                 mma(s_b[(4 * lg + e) * LK + 16 * b + lr], C[e], zero);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          S[b][e] = fmaf(p[e], S[b][e], (d[0][e] + d[1][e]) + (d[2][e] + d[3][e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[b][e] *= p[e];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          S[b] = mma(s_k[(4 * e + lg) * LK + 16 * b + lr], V[e], S[b]);
      }
    }
    t0 = next;
  }
  if (on) {
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * b + 4 * lg + e;
        if (i < D) st[(long long)i * D] = S[b][e];
      }
  }
}

template <typename T, bool DELTA>
hipError_t launch(const ScanArgs<T>& a, int n_seg, hipStream_t st) {
  const dim3 grid(n_seg, a.H, (a.D + 63) / 64);
  if (a.D <= 32) scan_chunk_kernel<T, 2, DELTA><<<grid, 256, 0, st>>>(a);
  else if (a.D <= 64) scan_chunk_kernel<T, 4, DELTA><<<grid, 256, 0, st>>>(a);
  else if (a.D <= 128) scan_chunk_kernel<T, 8, DELTA><<<grid, 256, 0, st>>>(a);
  else scan_chunk_kernel<T, 16, DELTA><<<grid, 256, 0, st>>>(a);
  return hipGetLastError();
}

}  // namespace

extern "C" {

// 16-bit rows at strides below 2^26; delta: al, the removal rates, and decay_scale <= 3 (16 tokens keep P
// above 2^-70).
// Segments [0, n_seg) of cu / slot / start; out [T][H * D] fp32, un-normalised read-outs.
hipError_t sm_scan_chunk(int dt, int delta, const void* r, long long ldr, const void* k, long long ldk,
                         const void* v, long long ldv, const void* wl, long long ldw, const void* al,
                         long long lda, const float* w0, const float* ub, float* state, float* out,
                         const int* cu, const int* slot, const int* start, int n_seg, int H, int D,
                         float decay_scale, float key_eps, hipStream_t st) {
  if (n_seg == 0) return hipSuccess;
  const auto stride = [](long long l) { return l >= 0 && l < (1 << 26); };   // (32-bit offsets in a chunk)
  if (n_seg < 0 || H < 1 || D < 1 || D > 256 || (delta && (al == nullptr || !(decay_scale <= 3.f))) ||
      !stride(ldr) || !stride(ldk) || !stride(ldv) || !stride(ldw) || !stride(lda) ||
      !stride((long long)H * D))
    return hipErrorInvalidValue;
#define GO(T)                                                                                   \
  {                                                                                             \
    const ScanArgs<T> a{(const T*)r, (const T*)k, (const T*)v, (const T*)wl, (const T*)al, ldr, ldk, \
                        ldv, ldw, lda, w0, ub, state, out, cu, slot, start, H, D,               \
                        decay_scale, key_eps};                                                  \
    return delta ? launch<T, true>(a, n_seg, st) : launch<T, false>(a, n_seg, st);              \
  }
  if (dt == kBF16) GO(bf16)
  if (dt == kF16) GO(fp16)
  return hipErrorInvalidValue;
#undef GO
}

}  // extern "C"
