// The steps of the chunked matrix-state recurrences on the bf16 matrix instructions, shared by the kernel whose own producer
// waves build a chunk's matrices (head_scan_chunk16.hip, which explains the method) and by the one that finds them built
// (head_scan_ahead.hip).
#pragma once
#include "head_scan.h"
#include "mma.h"

namespace lumen {
namespace hc16 {

constexpr int kC = 32;             // tokens per chunk
constexpr int LT = kC + 8;         // row stride of token-inner LDS images
constexpr int LA = kC + 4;         // row stride of the fp32 scratch of the inverse

__device__ __forceinline__ f32x16 mma(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma16f(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float lo_half(unsigned v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float hi_half(unsigned v) { return __uint_as_float(v & 0xffff0000u); }

// 8 fp32 values (registers 8s .. 8s+7 of x) -> bf16 head and remainder
__device__ __forceinline__ void split8(const f32x16& x, int s, uint4& h, uint4& l) {
  unsigned hh[4], ll[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = x[8 * s + 2 * e], b = x[8 * s + 2 * e + 1];
    hh[e] = pk2<bf16>(a, b);
    ll[e] = pk2<bf16>(a - lo_half(hh[e]), b - hi_half(hh[e]));
  }
  h = make_uint4(hh[0], hh[1], hh[2], hh[3]);
  l = make_uint4(ll[0], ll[1], ll[2], ll[3]);
}

// hardware exponential and reciprocal: for values that are rounded to bf16 next
__device__ __forceinline__ float silu_fast(float x) {
  return x * __builtin_amdgcn_rcpf(1.f + __expf(-x));
}
__device__ __forceinline__ unsigned silu_pair(unsigned v) {
  return pk2<bf16>(silu_fast(lo_half(v)), silu_fast(hi_half(v)));
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// place of inner index j in its LDS row
__device__ __forceinline__ int place(int j) {
  return (j & ~15) + 8 * ((j >> 2) & 1) + 4 * ((j >> 3) & 1) + (j & 3);
}

// four rows of 8 channels each of q or k
struct Item { uint4 r[4]; };

// four fp32 values -> bf16 head and remainder, 8 bytes each
__device__ __forceinline__ void put4(bf16* h, bf16* l, float a, float b, float c, float d) {
  const unsigned h0 = pk2<bf16>(a, b), h1 = pk2<bf16>(c, d);
  *reinterpret_cast<uint2*>(h) = make_uint2(h0, h1);
  *reinterpret_cast<uint2*>(l) = make_uint2(pk2<bf16>(a - lo_half(h0), b - hi_half(h0)),
                                            pk2<bf16>(c - lo_half(h1), d - hi_half(h1)));
}

// the diagonal entry of a 32x32 accumulator: lane c's column c, in either half
__device__ __forceinline__ float diagonal(const f32x16& x, int c, int hi) {
  float d = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) d = 8 * (r >> 2) + 4 * hi + (r & 3) == c ? x[r] : d;
  return d + __shfl_xor(d, 32, 64);
}


// Rows past the segment's end are read as its last row: their step size (or beta) is zero, so they add nothing to the
// state, and their read-outs are not stored.  Item `item` of a matrix: four rows from 4 (item / NV) on, 8 channels.
template <int DKP>
__device__ __forceinline__ void fetch_item(Item& it, const bf16* base, long long ldr, int qcol, int r0, int t0, int len,
                                           int Dk, int vec, int item) {
  constexpr int NV = DKP / 8;
  const int kq = (item / NV) & 7, d = 8 * (item % NV);
#pragma unroll
  for (int y = 0; y < 4; ++y) {
    const int i = min(t0 + 4 * kq + y, len - 1);
    const bf16* p = base + (long long)(r0 + i) * ldr + qcol + d;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (d < Dk) {
      if (vec) {
        v = *reinterpret_cast<const uint4*>(p);
      } else {
        unsigned e[8];
#pragma unroll
        for (int z = 0; z < 8; ++z)
          e[z] = d + z < Dk ? (unsigned)__builtin_bit_cast(unsigned short, p[z]) : 0u;
        v = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
      }
    }
    it.r[y] = v;
  }
}

// ... into its LDS image dst [token][channel], and (keys) the transposed one kt [channel][token]
template <int DKP>
__device__ __forceinline__ void put_item(Item& it, bool is_k, int silu_in, int item, bf16* dst, bf16* kt) {
  constexpr int LK = DKP + 8, NV = DKP / 8;
  const int kq = item / NV, part = item % NV;
  if (silu_in) {
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      uint4& v = it.r[y];
      v = make_uint4(silu_pair(v.x), silu_pair(v.y), silu_pair(v.z), silu_pair(v.w));
    }
  }
  if (item >= DKP) return;
  const int s16 = 16 * (part >> 1) + 4 * (part & 1);
#pragma unroll
  for (int y = 0; y < 4; ++y) {
    bf16* row = dst + (4 * kq + y) * LK + s16;
    *reinterpret_cast<uint2*>(row) = make_uint2(it.r[y].x, it.r[y].y);
    *reinterpret_cast<uint2*>(row + 8) = make_uint2(it.r[y].z, it.r[y].w);
  }
  if (!is_k) return;
  // transposed: 4 tokens of each of the 8 channels
  const unsigned e0[4] = {it.r[0].x, it.r[0].y, it.r[0].z, it.r[0].w};
  const unsigned e1[4] = {it.r[1].x, it.r[1].y, it.r[1].z, it.r[1].w};
  const unsigned e2[4] = {it.r[2].x, it.r[2].y, it.r[2].z, it.r[2].w};
  const unsigned e3[4] = {it.r[3].x, it.r[3].y, it.r[3].z, it.r[3].w};
  // 16-byte unit of the row (swapped by the channel group: lanes spread over banks)
  const int unit = (2 * (kq >> 2) + (kq & 1)) ^ (part & 3);
  bf16* t = kt + 8 * part * LT + 8 * unit + 4 * ((kq >> 1) & 1);
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    *reinterpret_cast<uint2*>(t + 2 * z * LT) =
        make_uint2((e0[z] & 0xffffu) | (e1[z] << 16), (e2[z] & 0xffffu) | (e3[z] << 16));
    *reinterpret_cast<uint2*>(t + (2 * z + 1) * LT) =
        make_uint2((e0[z] >> 16) | (e1[z] & 0xffff0000u), (e2[z] >> 16) | (e3[z] & 0xffff0000u));
  }
}

// A head's constants of the decay
struct HeadRates {
  float dtb, eA, ldc;
  bool logits;
  __device__ __forceinline__ HeadRates(const HeadScanArgs<bf16>& a, int hd)
      : dtb(a.a != nullptr ? a.dt_bias[hd] : 0.f), eA(a.a != nullptr ? expf(a.A_log[hd]) : 0.f),
        ldc(a.a != nullptr ? 0.f : a.log_decay[hd]), logits(a.a != nullptr) {}
};

// Lane c (both halves alike) is token c with logits ra, rb (tokens past the end, not live, add nothing): the log-decay sums up
// to it (s_L [32] too) and over the chunk, and its step size or beta (be [32])
template <bool DELTA>
__device__ __forceinline__ void token_decays(const HeadRates& f, bool live, float ra, float rb, int c, int hi, double& L,
                                             double& Lc, double* s_L, float* be) {
  float ld = f.ldc, dt = 1.f;
  if (f.logits) {
    dt = softplus_f(ra + f.dtb);
    ld = -f.eA * dt;
  }
  const float wt = DELTA ? sigmoid_f(rb) : dt;
  L = live ? (double)fmaxf(ld, -1e4f) : 0.0;
#pragma unroll
  for (int m = 1; m < 32; m <<= 1) {
    const double o = __shfl_up(L, m, 32);
    if (c >= m) L += o;
  }
  Lc = __shfl(L, 31, 32);
  if (hi == 0) {
    s_L[c] = L;
    be[c] = live ? wt : 0.f;
  }
}

// A chunk's matrices and factors in LDS
struct Chunk {
  bf16 *q, *k, *kt;             // rows [token][channel], keys [channel][token]
  bf16 *p0, *p1, *t0, *t1;      // G . Q K^T and the inverse, head and remainder
  float *gq, *gk, *w, *ek, *gc; // e^L |q|, e^L |k|, dt or beta, e^{L_C - L} |k|, e^{L_C}
};

// P^T = K Q^T (lane: query, registers: keys) times G, and the chunk's factors.  s_fk [32]: scratch
template <int KT, bool DELTA>
__device__ __forceinline__ void chunk_weights(const Chunk& B, const double* s_L, float* s_fk, double L, double Lc, int c,
                                              int hi, float q_scale, float key_eps) {
  constexpr int LK = 32 * KT + 8;
  f32x16 P, A, Q;
#pragma unroll
  for (int r = 0; r < 16; ++r) { P[r] = 0.f; A[r] = 0.f; Q[r] = 0.f; }
#pragma unroll 4
  for (int s = 0; s < 2 * KT; ++s) {
    const uint4 kv = *reinterpret_cast<const uint4*>(B.k + c * LK + 16 * s + 8 * hi);
    const uint4 qv = *reinterpret_cast<const uint4*>(B.q + c * LK + 16 * s + 8 * hi);
    P = mma(kv, qv, P);
    if (DELTA) {                           // unit lengths: the diagonals of K K^T and Q Q^T
      A = mma(kv, kv, A);
      Q = mma(qv, qv, Q);
    }
  }
  float fqc = 1.f, fkc = 1.f;
  if (DELTA) {
    fqc = q_scale / sqrtf(diagonal(Q, c, hi) + key_eps);
    fkc = 1.f / sqrtf(diagonal(A, c, hi) + key_eps);
    if (hi == 0) s_fk[c] = fkc;
    wave_lds_fence();
  }
  if (hi == 0) {
    const float g = expf((float)L);
    B.gq[c] = g * fqc;
    B.gk[c] = g * fkc;
    B.ek[c] = expf((float)(Lc - L)) * fkc;
    if (c == 0) *B.gc = expf((float)Lc);
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int j0 = 8 * g + 4 * hi;         // registers 4g + e: token j0 + e
    const double2 La = *reinterpret_cast<const double2*>(&s_L[j0]);
    const double2 Lb = *reinterpret_cast<const double2*>(&s_L[j0 + 2]);
    const float d[4] = {(float)(L - La.x), (float)(L - La.y), (float)(L - Lb.x), (float)(L - Lb.y)};
    float fk[4] = {1.f, 1.f, 1.f, 1.f}, z[4];
    if (DELTA) load4<float>(&s_fk[j0], fk);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float v = P[4 * g + e] * (fqc * fk[e]) * __expf(fminf(d[e], 0.f));
      z[e] = j0 + e <= c ? v : 0.f;
    }
    const int at = c * LT + place(j0);
    put4(&B.p0[at], &B.p1[at], z[0], z[1], z[2], z[3]);
  }
}

// Delta rule: T = (I + A)^-1 into t0, t1, which lie one behind the other.  s_fk [32]: scratch
template <int KT>
__device__ __forceinline__ void chunk_inverse(const Chunk& B, const double* s_L, float* s_fk, int lane, float key_eps) {
  constexpr int LK = 32 * KT + 8;
  const int c = lane & 31, hi = lane >> 5;
  f32x16 A;
#pragma unroll
  for (int r = 0; r < 16; ++r) A[r] = 0.f;
#pragma unroll
  for (int s = 0; s < 2 * KT; ++s) {
    const uint4 kv = *reinterpret_cast<const uint4*>(B.k + c * LK + 16 * s + 8 * hi);
    A = mma(kv, kv, A);
  }
  const float fkc = 1.f / sqrtf(diagonal(A, c, hi) + key_eps);
  if (hi == 0) s_fk[c] = fkc;
  wave_lds_fence();
  // scratch, transposed: row c, entry j = A[j][c] (j > c); it lies where T is written later
  float* sA = reinterpret_cast<float*>(B.t0);
  static_assert(sizeof(float) * kC * LA <= 2 * sizeof(bf16) * kC * LT, "scratch fits");
  const double Lo = s_L[c];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int j0 = 8 * g + 4 * hi;
    const double2 La = *reinterpret_cast<const double2*>(&s_L[j0]);
    const double2 Lb = *reinterpret_cast<const double2*>(&s_L[j0 + 2]);
    const float d[4] = {(float)(La.x - Lo), (float)(La.y - Lo), (float)(Lb.x - Lo),
                        (float)(Lb.y - Lo)};
    float fk[4], be[4], x[4];
    load4<float>(&s_fk[j0], fk);
    load4<float>(&B.w[j0], be);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      x[e] = j0 + e > c ? A[4 * g + e] * (fk[e] * fkc) * (be[e] * __expf(fminf(d[e], 0.f))) : 0.f;
    store4<float>(&sA[c * LA + j0], x);
  }
  wave_lds_fence();
  // the diagonal 16x16 blocks by back substitution along a row,
  // T[i][j] = [i = j] - sum_{k > j} T[i][k] A[k][j], a lane per row i ...
  const int b0 = lane & 16, ii = lane & 15, lr = lane & 15, lg = lane >> 4;
  float t[16];
#pragma unroll
  for (int j = 15; j >= 0; --j) {
    float acc = 0.f;
#pragma unroll
    for (int k4 = 0; k4 < 16; k4 += 4) {
      if (k4 + 3 > j) {
        const float4 x = *reinterpret_cast<const float4*>(&sA[(b0 + j) * LA + b0 + k4]);
        if (k4 > j) acc += x.x * t[k4];
        if (k4 + 1 > j) acc += x.y * t[k4 + 1];
        if (k4 + 2 > j) acc += x.z * t[k4 + 2];
        acc += x.w * t[k4 + 3];
      }
    }
    t[j] = j == ii ? 1.f : (j < ii ? -acc : 0.f);
  }
  wave_lds_fence();
  if (lane < 32) {
#pragma unroll
    for (int j = 0; j < 16; j += 4)
      *reinterpret_cast<float4*>(&sA[(b0 + ii) * LA + b0 + j]) =
          make_float4(t[j], t[j + 1], t[j + 2], t[j + 3]);
  }
  wave_lds_fence();
  // ... and the block below as -T11 (A10 T00); A10[r][k] lies at scratch [k][16 + r]
  f32x4 x = {0.f, 0.f, 0.f, 0.f}, y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < 4; ++m)
    x = mma16f(sA[(4 * m + lg) * LA + 16 + lr], sA[(4 * m + lg) * LA + lr], x);
#pragma unroll
  for (int e = 0; e < 4; ++e) y = mma16f(sA[(16 + lr) * LA + 16 + 4 * lg + e], x[e], y);
  wave_lds_fence();                        // scratch read: T may be written over it
  bf16 *th = B.t0, *tl = B.t1;
  if (lane < 32) {
#pragma unroll
    for (int j = 0; j < 16; j += 4) {
      const int at = (b0 + ii) * LT + place(b0 + j);
      put4(th + at, tl + at, t[j], t[j + 1], t[j + 2], t[j + 3]);
    }
  } else if (lane < 48) {                  // the block above the diagonal
#pragma unroll
    for (int j = 16; j < 32; j += 4) {
      const int at = ii * LT + place(j);
      put4(th + at, tl + at, 0.f, 0.f, 0.f, 0.f);
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int at = (16 + 4 * lg + e) * LT + place(lr);
    const bf16 h = __float2bfloat16(-y[e]);
    th[at] = h;
    tl[at] = __float2bfloat16(-y[e] - __bfloat162float(h));
  }
}

// ---- a wave of 32 columns of the state ----
// a chunk's values, silu'd if they pass through it
__device__ __forceinline__ void take_values(const bf16 (&vn)[16], int silu_in, float (&V)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    V[r] = to_f32(vn[r]);
    if (silu_in) V[r] = silu_fast(V[r]);
  }
}

template <int KT> struct State { f32x16 r[KT]; };

template <int KT>
__device__ __forceinline__ void state_load(State<KT>& S, const float* sp, bool fresh, bool on, int Dk, int Dv, int hi) {
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * kt + 8 * (r >> 2) + 4 * hi + (r & 3);
      S.r[kt][r] = (!fresh && on && row < Dk) ? sp[(long long)row * Dv] : 0.f;
    }
}
template <int KT>
__device__ __forceinline__ void state_store(const State<KT>& S, float* sp, int Dk, int Dv, int hi) {
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 32 * kt + 8 * (r >> 2) + 4 * hi + (r & 3);
      if (row < Dk) sp[(long long)row * Dv] = S.r[kt][r];
    }
}

// a chunk matrix times a split right operand: its half s
__device__ __forceinline__ f32x16 apply_half(const bf16* mh, const bf16* ml, int s, uint4 h, uint4 l, f32x16 acc, int c, int hi) {
  const int at = c * LT + 16 * s + 8 * hi;
  const uint4 ah = *reinterpret_cast<const uint4*>(mh + at);
  const uint4 al = *reinterpret_cast<const uint4*>(ml + at);
  acc = mma(ah, h, acc);
  acc = mma(ah, l, acc);
  return mma(al, h, acc);
}
__device__ __forceinline__ f32x16 chunk_apply(const bf16* mh, const bf16* ml, const f32x16& x, f32x16 acc, int c, int hi) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    uint4 h, l;
    split8(x, s, h, l);
    acc = apply_half(mh, ml, s, h, l, acc, c, hi);
  }
  return acc;
}

// n read-outs of a chunk, 32 columns of a head
__device__ __forceinline__ void store_rows(const f32x16& O, int n, float* orow, long long ldo, int hi) {
  if (n == kC) {
#pragma unroll
    for (int r = 0; r < 16; ++r) orow[(8 * (r >> 2) + (r & 3)) * ldo] = O[r];
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (8 * (r >> 2) + 4 * hi + (r & 3) < n) orow[(8 * (r >> 2) + (r & 3)) * ldo] = O[r];
  }
}

// a chunk's transposed keys as left operands
template <int KT> struct Keys {
  uint4 k[KT][2];
  __device__ __forceinline__ Keys(const Chunk& B, int c, int hi) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        k[kt][s] = *reinterpret_cast<const uint4*>(B.kt + (32 * kt + c) * LT + 8 * ((2 * s + hi) ^ ((c >> 3) & 3)));
  }
};

// S = e^{L_C} S + K^T (e^{L_C - L} U)
template <int KT>
__device__ __forceinline__ void state_move(State<KT>& S, const Chunk& B, const Keys<KT>& K, f32x16 U, int hi) {
  const float gc = *B.gc;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float ek[4];
    load4<float>(&B.ek[8 * g + 4 * hi], ek);
#pragma unroll
    for (int e = 0; e < 4; ++e) U[4 * g + e] *= ek[e];
  }
  uint4 uh[2], ul[2];
  split8(U, 0, uh[0], ul[0]);
  split8(U, 1, uh[1], ul[1]);
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
    for (int r = 0; r < 16; ++r) S.r[kt][r] *= gc;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      S.r[kt] = mma(K.k[kt][s], uh[s], S.r[kt]);
      S.r[kt] = mma(K.k[kt][s], ul[s], S.r[kt]);
    }
  }
}

// what a chunk writes: w V, or (delta, U = K S_0) w (V - e^L |k| U) through the inverse
template <bool DELTA>
__device__ __forceinline__ f32x16 chunk_writes(const Chunk& B, f32x16 U, const float (&V)[16], int c, int hi) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float ww[4], gk[4];
    load4<float>(&B.w[8 * g + 4 * hi], ww);
    if (DELTA) load4<float>(&B.gk[8 * g + 4 * hi], gk);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 4 * g + e;
      U[r] = DELTA ? ww[e] * (V[r] - gk[e] * U[r]) : ww[e] * V[r];
    }
  }
  if (!DELTA) return U;
  f32x16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.f;
  return chunk_apply(B.t0, B.t1, U, z, c, hi);
}

// O = e^L |q| (Q S_0) + skip V
__device__ __forceinline__ f32x16 old_state_read(const Chunk& B, f32x16 O, const float (&V)[16], float skip, int hi) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    float gq[4];
    load4<float>(&B.gq[8 * g + 4 * hi], gq);
#pragma unroll
    for (int e = 0; e < 4; ++e) O[4 * g + e] = gq[e] * O[4 * g + e] + skip * V[4 * g + e];
  }
  return O;
}

}  // namespace hc16
}  // namespace lumen
