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
//
// A chunk's decays and sums, its scaled rows and its small matrices do not need the state: producer waves build the
// next chunk's (three stages, a barrier after each, the rows after it in flight) while the column waves run the one
// before, in two LDS buffers.  With all of it done by the same four waves, one after the other, a step was 21 thousand
// cycles (delta, heads of 128: exponentials and divisions 5.8, scaled rows 3.3, the matrices and the 16-row
// substitution 4.9, the state's products 7); it is 16 now, bound by what
// the three waves of a SIMD issue: matrix instructions 5.6 of it.
// Measured (width 2048, bf16, the norm kernel's 17 us included), four waves -> this, us: delta, 16 heads of 128: 8
// portions of 512 tokens 305 -> 237, one of 512 281 -> 211, 32 of 128 311 -> 248; 8 heads of 256 512 -> 434; 64 of 32 185
// -> 172; wkv, 32 heads of 64 whose decays hardly ever cut a chunk: 136 -> 126, 117 -> 99, 106 -> 101; 8 heads of 256 338 ->
// 281.  (Token by token: 1000 and 460.)
// Error against float64 (512 tokens, heads of 32 - 256): the read-outs are as far off as the serial walk's
// (1.66e-3, the bf16 result's rounding), the state a little less (delta 0.86e-7, serial 0.90e-7; wkv 0.62e-7,
// serial 0.65e-7).  That takes the decays' products in float64 (in fp32: + 0.1e-7) and care with the sums
// (see the state's update; term by term 1.4e-7 and 0.9e-7), which cost 20 us of the delta scan.
// (Both products of an update in one accumulator: 0.94e-7.)
//
// Range: P_t and 1 / P_16 must stay finite, and so must the masked entries' factors.  A wkv chunk ends
// before the token that would take some channel's P below 2^-100, so a decay beyond that (0 too) is alone in
// its chunk, where nothing is divided by it; the delta rule's decays, at least e^-decay_scale per token,
// stay above 2^-70.  r and k that scaled rows could not hold as normal numbers (kLarge, kTiny*), infinities and
// NaN run one token at a time, so that earlier tokens stay as they are; wkv values below kSmall make the
// chunk end at 2^-40.
// A chunk that turns out to leave the range costs rows formed and asked for twice, and two more barriers; where the two
// before it did, its place is found before the rows (one more barrier).  us, four waves -> rows always twice, three
// more barriers -> this, 8 x 512 tokens, 32 heads of 64, the kernel alone: decays a token of -e^N(0..2, 0.6), all chunks cut,
// 478 -> 442 -> 301; a head of which 31 - 49 of 39 - 51 chunks are cut 207 -> 222 -> 180; none cut 119 -> 107 -> 109.
// Decays up to e^-50 a token, chunks of one: 770 with the four-wave form.
#include "seqmix.h"

using namespace lumen;

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kC = 16;                 // tokens per chunk
constexpr int LP = 20;                 // row stride of the chunk matrices in LDS
constexpr int kCol = 4;                 // column waves of a workgroup
constexpr float kMinP = 0x1p-100f;     // smallest product of a chunk's decays

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

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

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

// KB: key channels in blocks of 16; kProd: producer waves
template <typename T, int KB, bool DELTA, int kProd>
__global__ void __launch_bounds__(64 * (kCol + kProd))
scan_chunk_kernel(const ScanArgs<T> a) {
  constexpr int DKP = 16 * KB, LK = DKP + 4;
  constexpr int NG = 64 * kProd / DKP, TG = kC / NG;     // staging: token groups, tokens of each
  constexpr int NM = DELTA ? 4 : 1;
  static_assert(NG * TG == kC && NM <= kProd, "staging");
  struct Buf {                                           // a chunk as the column waves read it
    float r[kC * LK], k[kC * LK], u[DELTA ? kC * LK : 4], b[DELTA ? kC * LK : 4];
    float m[NM][kC * LP], P[DKP];
  };
  __shared__ __attribute__((aligned(16))) Buf s_buf[2];
  __shared__ __attribute__((aligned(16))) float s_iP[DKP], s_red[kC][KB];
  __shared__ double s_gp[NG][DKP], s_gt[DELTA ? 1 : kC][DELTA ? 1 : DKP];   // a token group's decay; up to each token (`cut`)
  __shared__ float s_tok[kC];
  __shared__ int s_n[2], s_low[2], s_small[2];
  const int sg = blockIdx.x, hd = blockIdx.y;
  const int r0 = a.cu[sg], len = a.cu[sg + 1] - r0;
  if (len <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool col = w < kCol;                                     // else: a producer
  const int D = a.D, col0 = hd * D;
  const int j = (blockIdx.z * kCol + w) * 16 + lr;               // a column wave's lane: its value column
  const bool on = col && j < D;
  // row t + i of `base`'s chunk at t0, column c (uniform base, 32-bit byte offset from the chunk's first row,
  // so the rows that are left count up to a chunk's; i known when compiled).  Rows past the portion repeat its
  // last one, channels past D the last one: blanked where they are used.
  const auto get = [&](const T* base, long long ld, int t0, int t, int i, int c)
                       __attribute__((always_inline)) {
    const unsigned step = (unsigned)ld, last = (unsigned)min(len - 1 - t0, kC - 1) * step;
    const unsigned at = min((unsigned)t * step + (unsigned)i * step, last) + (unsigned)c;
    return *reinterpret_cast<const T*>(
        reinterpret_cast<const char*>(base + (long long)(r0 + t0) * ld + col0) + at * (unsigned)sizeof(T));
  };

  // ---------------- the producers ----------------
  const int ptid = col ? 0 : tid - 64 * kCol;
  const int ch = ptid % DKP, tg = ptid / DKP;                    // channel, token group
  const bool chan = ch < D;
  const int chc = min(ch, D - 1);
  const float w0 = chan ? a.w0[col0 + ch] : 0.f, ub = chan ? a.ub[col0 + ch] : 0.f;
  T pr[TG], pk[TG], pw[TG], pa[TG];                              // the chunk to build, as loaded
  float rv[TG], kv[TG], wv[TG], av[TG], tok[TG];
  const auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < TG; ++q) {
      pr[q] = get(a.r, a.ldr, t0, tg * TG, q, chc);
      pk[q] = get(a.k, a.ldk, t0, tg * TG, q, chc);
      pw[q] = get(a.wl, a.ldw, t0, tg * TG, q, chc);
      if (DELTA) pa[q] = get(a.al, a.lda, t0, tg * TG, q, chc);
    }
  };
  // decays, removal rates, the channel sums of every token
  const auto decays = [&](int t0, int par) __attribute__((always_inline)) {
    unsigned top = 0u, low = ~0u, lim = 0u;   // r and k: largest, smallest - 1; the others: largest
    double gp = 1.;
#pragma unroll
    for (int q = 0; q < TG; ++q) {
      const bool live = t0 + tg * TG + q < len && chan;
      rv[q] = chan ? to_f32(pr[q]) : 0.f;
      kv[q] = chan ? to_f32(pk[q]) : 0.f;
      const float zl = to_f32(pw[q]), z = zl + w0;
      const float d = DELTA ? exp_near(-a.decay_scale * sigmoid_near(z)) : exp_near(-exp_near(z));
      wv[q] = live ? d : 1.f;
      gp *= wv[q];
      const unsigned mr = mag(rv[q]), mk = mag(kv[q]);
      top = max(top, max(mr, mk));
      low = min(low, min(mr - 1u, mk - 1u));   // (0 is as good as large)
      lim = max(lim, mag(zl));
      if (DELTA) {
        const float al = to_f32(pa[q]);
        lim = max(lim, mag(al));
        av[q] = live ? sigmoid_near(al + ub) : 0.f;
      }
      const float s = sum16(DELTA ? kv[q] * kv[q] : rv[q] * ub * kv[q]);
      if (lr == 0) s_red[tg * TG + q][ch >> 4] = s;
    }
    s_gp[tg][ch] = gp;
    if (top > kLarge || low < (DELTA ? kTinyDelta : kTinyWkv) - 1u || lim >= kInf)
      atomicMin(&s_n[par], 1);
    if (!DELTA && low < kSmall - 1u) s_small[par] = 1;
  };
  // the tokens' sums, a lane for each of the wave's, handed round
  const auto tokens = [&]() __attribute__((always_inline)) {
    float v = 0.f;
#pragma unroll
    for (int b = 0; b < KB; ++b) v += s_red[tg * TG + lane % TG][b];
    if (DELTA) v = 1.f / sqrtf(v + a.key_eps);
#pragma unroll
    for (int q = 0; q < TG; ++q) {
      tok[q] = lane_f(v, q);
      if (DKP < 64) tok[q] = lane < 32 ? tok[q] : lane_f(v, 32 + q);
    }
  };
  // where does a channel's product leave the range?  The chunk ends before that token
  const auto cut = [&](int par) __attribute__((always_inline)) {
    if constexpr (DELTA) return;
    const float least = s_small[par] ? kSmallP : kMinP;
    double before = 1., p = 1.;
#pragma unroll
    for (int g = 0; g < NG; ++g) before *= g < tg ? s_gp[g][ch] : 1.;
    int first = kC;
#pragma unroll
    for (int q = 0; q < TG; ++q) {
      p *= wv[q];
      s_gt[tg * TG + q][ch] = p;
      if (first == kC && before * p < least) first = tg * TG + q;
    }
    if (first < kC && !(before < least)) atomicMin(&s_n[par], max(first, 1));
  };
  // The scaled rows of a chunk of n tokens (ALL: as many as there are, at most kC); rows that are left for the next
  // chunk decay nothing.  Returns whether some channel's product leaves the range (ALL).
  const auto rows = [&](auto all, Buf& B, int n, float least) __attribute__((always_inline)) {
    constexpr bool ALL = decltype(all)::value;
    const int tc = ALL ? NG - 1 : (n - 1) / TG;          // the group that the chunk ends in
    double P = 1., Q = 1.;               // decay of the token groups before and after this one
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      P *= g < tg ? s_gp[g][ch] : 1.;
      Q *= g > tg && g <= tc ? (ALL || DELTA || g < tc ? s_gp[g][ch] : s_gt[n - 1][ch]) : 1.;
    }
#pragma unroll
    for (int q = TG - 1; q >= 0; --q) {  // decayed to the chunk's end
      const int at = (tg * TG + q) * LK + ch;
      const bool live = tg * TG + q < n;
      B.k[at] = live ? (float)(kv[q] * Q) : 0.f;
      if (DELTA) B.b[at] = live ? (float)(kv[q] * tok[q] * av[q] * Q) : 0.f;
      Q *= ALL || live ? wv[q] : 1.f;
    }
#pragma unroll
    for (int q = 0; q < TG; ++q) {       // decayed from the chunk's start
      const int t = tg * TG + q, at = t * LK + ch;
      const bool live = t < n;
      const float P0 = (float)P;
      P *= ALL || live ? wv[q] : 1.f;
      B.r[at] = live ? rv[q] * (DELTA ? (float)P : P0) : 0.f;
      if (DELTA) B.u[at] = live ? kv[q] * tok[q] * P0 : 0.f;
      else if (ch == 0) s_tok[t] = tok[q];
    }
    if (tg != tc) return false;
    B.P[ch] = (float)P;
    s_iP[ch] = 1.f / (float)P;           // (one token: only entries that are masked out see it)
    return !DELTA && ALL && !((float)P >= least);
  };
  // chunk matrices, one per wave: U K^T, U B^T (then inverted), R K^T, R B^T
  const auto matrices = [&](Buf& B, int n) __attribute__((always_inline)) {
    const int pw_ = w - kCol;
    if (pw_ >= NM) return;
    const float* x = (DELTA && pw_ < 2 ? B.u : B.r) + lr * LK + 4 * lg;
    const float* y = (DELTA && (pw_ & 1) ? B.b : B.k) + lr * LK + 4 * lg;
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
      if (KB > 8 && b % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    const f32x4 acc = (c[0] + c[1]) + (c[2] + c[3]);
    float* m = B.m[pw_];
    float z[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * lg + e;          // row: token t; column lr: token s
      z[e] = i < n && (DELTA && pw_ >= 2 ? lr <= i : lr < i) ? acc[e] : 0.f;
      if (!DELTA && lr == i && i < n) z[e] = s_tok[i];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) m[(4 * lg + e) * LP + lr] = z[e];
    if (DELTA && pw_ == 1) {
      // (I + M)^-1 = D - D C D: D the inverses of the diagonal 8 x 8 blocks (a lane per column, substitution),
      // C the block below them.  (Substitution over all sixteen rows: 3800 cycles, a fifth of the step; here 1000.)
      wave_lds_fence();
      const int hb = lr >> 3;
      const float* d = m + 8 * hb * (LP + 1);
      float4 x[8][2];
#pragma unroll
      for (int i = 1; i < 8; ++i) {
        x[i][0] = *reinterpret_cast<const float4*>(d + i * LP);
        if (i > 4) x[i][1] = *reinterpret_cast<const float4*>(d + i * LP + 4);
      }
      float4 cr = *reinterpret_cast<const float4*>(m + lr * LP + 4 * lg);
      if (!(lr >= 8 && lg < 2)) cr = make_float4(0.f, 0.f, 0.f, 0.f);
      float t[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < i; ++q) {
          const float4 r4 = x[i][q >> 2];
          v += (q % 4 == 0 ? r4.x : q % 4 == 1 ? r4.y : q % 4 == 2 ? r4.z : r4.w) * t[q];
        }
        t[i] = (i == (lr & 7) ? 1.f : 0.f) - v;      // (0 above the diagonal: every term is)
      }
      wave_lds_fence();
      if (lg < 2) {                      // lane group 0: D's blocks; 1: zeros where C was
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (lg == 0) m[(8 * hb + i) * LP + lr] = t[i];
          else if (lr < 8) m[(8 + i) * LP + lr] = 0.f;
      }
      wave_lds_fence();
      const float4 da = *reinterpret_cast<const float4*>(m + lr * LP + 4 * lg);
      f32x4 db, X = {0.f, 0.f, 0.f, 0.f}, Y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) db[e] = m[(4 * lg + e) * LP + lr];
      X = mma(cr.x, db[0], X);
      X = mma(cr.y, db[1], X);
      X = mma(cr.z, db[2], X);
      X = mma(cr.w, db[3], X);
      Y = mma(da.x, X[0], Y);
      Y = mma(da.y, X[1], Y);
      Y = mma(da.z, X[2], Y);
      Y = mma(da.w, X[3], Y);
      wave_lds_fence();
#pragma unroll
      for (int e = 0; e < 4; ++e) m[(4 * lg + e) * LP + lr] = db[e] - Y[e];
    }
  };

  // ---------------- the column waves ----------------
  f32x4 S[KB], V, O, C;
  T pv[4];
  float* st = a.state + ((long long)a.slot[sg] * a.H + hd) * D * D + j;
  const int jc = min(j, D - 1);
  // the token of a lane's e-th value: an inner index of every product with V
  const auto tok_of = [&](int e) { return DELTA ? 4 * lg + e : 4 * e + lg; };
  const auto fetch_v = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) pv[e] = get(a.v, a.ldv, t0, tok_of(0), DELTA ? e : 4 * e, jc);
  };
  // what the old state gives (four sums each: a quarter of the chain, and of its error)
  const auto old_state = [&](const Buf& B) __attribute__((always_inline)) {
    f32x4 o[4], c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = c[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      const float4 x = *reinterpret_cast<const float4*>(&B.r[lr * LK + 16 * b + 4 * lg]);
      o[0] = mma(x.x, S[b][0], o[0]);
      o[1] = mma(x.y, S[b][1], o[1]);
      o[2] = mma(x.z, S[b][2], o[2]);
      o[3] = mma(x.w, S[b][3], o[3]);
      if (DELTA) {
        const float4 u = *reinterpret_cast<const float4*>(&B.u[lr * LK + 16 * b + 4 * lg]);
        c[0] = mma(u.x, S[b][0], c[0]);
        c[1] = mma(u.y, S[b][1], c[1]);
        c[2] = mma(u.z, S[b][2], c[2]);
        c[3] = mma(u.w, S[b][3], c[3]);
      }
      if (KB > 8 && b % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
    O = (o[0] + o[1]) + (o[2] + o[3]);
    if (DELTA) C = (c[0] + c[1]) + (c[2] + c[3]);
  };
  const auto read_out = [&](const Buf& B, int t0, int n) __attribute__((always_inline)) {
    const auto small = [&](int m, const f32x4& x, f32x4 acc) {
      float4 y;
      if (DELTA) y = *reinterpret_cast<const float4*>(&B.m[m][lr * LP + 4 * lg]);
      else {
        const float* r = &B.m[m][lr * LP + lg];
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
  };
  // The state moves on.  wkv: decayed, then the tokens' terms in order, the last (and least decayed)
  // ones last, so that a fast channel sees few roundings.  Delta: what the chunk adds is summed apart, in
  // fours, and meets the state in one rounding; added term by term to it the error was 1.4 - 1.6 times
  // the serial walk's.
  const auto new_state = [&](const Buf& B, int b0, int b1) __attribute__((always_inline)) {
#pragma unroll
    for (int b = b0; b < b1; ++b) {
      const float4 P = *reinterpret_cast<const float4*>(&B.P[16 * b + 4 * lg]);
      const float p[4] = {P.x, P.y, P.z, P.w};
      if (DELTA) {
        f32x4 d[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          d[e] = mma(B.k[(4 * lg + e) * LK + 16 * b + lr], V[e], zero) +
                 mma(B.b[(4 * lg + e) * LK + 16 * b + lr], C[e], zero);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
          S[b][e] = fmaf(p[e], S[b][e], (d[0][e] + d[1][e]) + (d[2][e] + d[3][e]));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) S[b][e] *= p[e];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          S[b] = mma(B.k[(4 * e + lg) * LK + 16 * b + lr], V[e], S[b]);
      }
      if (KB > 8 && b % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Step: the producers build the chunk at tb while the column waves run the one before it, [tc, tc + nc).  Both
  // meet at the same barriers: what decides about more of them lies in LDS before the second.
  if (tid < 2) { s_n[tid] = kC; s_low[tid] = s_small[tid] = 0; }
  const auto count = [&](int par, int tb) { return __builtin_amdgcn_readfirstlane(min(s_n[par], len - tb)); };
  // A wkv chunk's rows are formed as if all of it stayed in range, and again if it does not -- unless the two before were
  // cut (a head with a fast channel cuts most of its chunks): then the place is found first.  The delta rule's length
  // is known before its rows.
  if (!col) {
    int tb = 0, par = 0, cuts = 0;
    // one step; false: it was the last
    const auto step = [&](auto cutting) __attribute__((always_inline)) {
      constexpr bool CUT = decltype(cutting)::value;
      const bool build = tb < len;
      Buf& B = s_buf[par];
      if (build) decays(tb, par);
      __syncthreads();
      int n = min(kC, len - tb);
      if (build) {
        if (CUT) {
          cut(par);
          __syncthreads();
        }
        tokens();
        if (DELTA || CUT) {
          n = count(par, tb);
          rows(std::false_type{}, B, n, 0.f);
        } else if (rows(std::true_type{}, B, n, s_small[par] ? kSmallP : kMinP)) {
          s_low[par] = 1;
        }
        if (tb + n < len) fetch(tb + n);       // in flight from here on, unless the chunk is shorter
      }
      __syncthreads();
      if (!DELTA && !CUT && build && (s_n[par] < kC || s_low[par])) {
        cut(par);
        __syncthreads();
        n = count(par, tb);
        rows(std::false_type{}, B, n, 0.f);
        if (tb + n < len) fetch(tb + n);
        __syncthreads();
      }
      cuts = !DELTA && n < min(kC, len - tb) ? cuts + 1 : 0;
      if (ptid == 0) { s_n[par ^ 1] = kC; s_low[par ^ 1] = s_small[par ^ 1] = 0; }
      if (build) matrices(B, n);
      __syncthreads();
      tb += n;
      par ^= 1;
      return build;
    };
    fetch(0);
    __syncthreads();
    for (;;) {                           // (two loops: with the choice inside, a step that is not cut took 0.2 us more)
      do
        if (!step(std::false_type{})) return;
      while (cuts < 2);
      if constexpr (!DELTA) {
        do
          if (!step(std::true_type{})) return;
        while (cuts > 0);
      }
    }
  }
  const bool fresh = a.start[sg] == 0;
#pragma unroll
  for (int b = 0; b < KB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 16 * b + 4 * lg + e;
      S[b][e] = (!fresh && on && i < D) ? st[(long long)i * D] : 0.f;
    }
  fetch_v(0);
  __syncthreads();
  for (int tb = 0, tc = 0, nc = 0, par = 0, cuts = 0;; par ^= 1) {
    const bool build = tb < len;
    const Buf& A = s_buf[par ^ 1];
    if (nc > 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) V[e] = tok_of(e) < nc ? to_f32(pv[e]) : 0.f;
    }
    if (build && tb > 0) fetch_v(tb);
    if (nc > 0) old_state(A);
    if (build) {                         // a value that no other row may meet: its chunk is one token long
      unsigned lim = 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) lim = max(lim, mag(to_f32(pv[e])));
      if (lim >= kInf) atomicMin(&s_n[par], 1);
    }
    // (nothing of this waits for the producers: cut so that the matrix units are not wanted by all at once)
    if (nc > 0) read_out(A, tc, nc);
    __syncthreads();
    if (build && cuts > 1) __syncthreads();
    if (nc > 0) new_state(A, 0, KB / 2);
    __syncthreads();
    if (!DELTA && build && cuts < 2 && (s_n[par] < kC || s_low[par])) {
      __syncthreads();
      __syncthreads();
    }
    const int n = build ? count(par, tb) : 0;
    cuts = !DELTA && n < min(kC, len - tb) ? cuts + 1 : 0;
    if (nc > 0) new_state(A, KB / 2, KB);
    __syncthreads();
    if (!build) break;
    tc = tb;
    nc = n;
    tb += n;
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
  const dim3 grid(n_seg, a.H, (a.D + 16 * kCol - 1) / (16 * kCol));
#define GO(KB, NP) scan_chunk_kernel<T, KB, DELTA, NP><<<grid, 64 * (kCol + NP), 0, st>>>(a)
  // Eight producer waves keep up with the column waves; four, where two such workgroups fit a CU and there are so many
  // (wkv, 32 portions of 128 x 32 heads of 64: 126 -> 99 us, delta, 8 of 512 x 64 of 32: 257 -> 171; heads of 128 not: 246 -> 261)
  const bool few = (long long)grid.x * grid.y * grid.z <= 256;
  if (a.D <= 32) { if (few) GO(2, 8); else GO(2, 4); }
  else if (a.D <= 64) { if (few) GO(4, 8); else GO(4, 4); }
  else if (a.D <= 128) GO(8, 8);
  else GO(16, 8);
#undef GO
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
