// The chunked matrix-state recurrences of head_scan_chunk.hip for bf16 models, on the bf16 matrix
// instructions (sixteen times the fp32 ones' rate) at fp32-level accuracy, with the chunk matrices
// built ahead of their use.
//
//   U   = dt * V                                                   (linear)
//   U   = (I + strict_lower(beta_i G_ij k_i.k_j))^-1 (beta (V - e^L K S_0))       (delta)
//   O   = e^L (Q S_0) + (G . Q K^T) U (+ skip V)
//   S_C = e^{L_C} S_0 + K^T (e^{L_C - L} U)
//
// Operands: the rows of q and k ARE bf16 (convolution outputs, or silu of a projection rounded
// once), so they enter exactly; the delta rule's unit lengths are fp32 factors of rows and columns
// (of Q S_0, K S_0, Q K^T, K K^T and U) instead of a rescaled copy.  Every fp32 operand -- the
// state, U, the two chunk matrices -- is split into a bf16 head and a bf16 remainder: two products
// (three where both sides are split) keep ~16 mantissa bits; sums are fp32.  The state itself
// stays fp32 in accumulator registers, a wave holding [Dk x 32 value columns].
//
// A workgroup is NW column waves and TWO producer waves, and two LDS buffers: while the column waves
// run chunk n, the producers build chunk n + 1 in two phases with a barrier after each.  First one
// stores q and the decays, the other k and k transposed, from registers they loaded one chunk
// earlier, and both start loading chunk n + 2 (meanwhile the column waves take Q S_0 and K S_0);
// then one forms G . Q K^T and the other the triangular inverse (meanwhile: U, O and the state).
//
// 32x32x16 products: accumulator register r of lane half hi is row 8 (r >> 2) + 4 hi + (r & 3); the
// registers 8s .. 8s+7 therefore hold inner indices {16s + 4hi + 0..3, 16s + 8 + 4hi + 0..3} and are
// a right operand as they are when the left operand is stored in that order: in every 16 entries of
// an LDS row the 4-entry groups 1 and 2 are swapped, and a lane reads its 8 entries as 16 bytes.
#include "head_chunk16.h"

using namespace lumen;
using namespace lumen::hc16;

namespace {

template <int DKP, bool DELTA>
struct __align__(16) ChunkBuf {
  bf16 q[kC * (DKP + 8)], k[kC * (DKP + 8)];   // [token][channel]
  bf16 kt[DKP * LT];                           // [channel][token]
  bf16 p[2][kC * LT];                          // G . Q K^T, head and remainder
  bf16 t[DELTA ? 2 : 1][DELTA ? kC * LT : 8];  // the inverse
  float gq[kC], gk[kC], w[kC], ek[kC];         // e^L |q|, e^L |k|, dt or beta, e^{L_C - L} |k|
  float gc, pad[3];                            // e^{L_C}
  __device__ __forceinline__ Chunk view() {
    return Chunk{q, k, kt, p[0], p[1], t[0], t[DELTA ? 1 : 0], gq, gk, w, ek, &gc};
  }
};

// what the old state gives: Q S_0 and (delta) K S_0
template <int KT, bool DELTA>
__device__ __forceinline__ void state_read(const State<KT>& S, const Chunk& B, f32x16& O, f32x16& U, int c, int hi) {
  constexpr int LK = 32 * KT + 8;
#pragma unroll
  for (int r = 0; r < 16; ++r) { O[r] = 0.f; U[r] = 0.f; }
#pragma unroll
  for (int kt = 0; kt < KT; ++kt)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      uint4 h, l;
      split8(S.r[kt], s, h, l);
      const int at = c * LK + 32 * kt + 16 * s + 8 * hi;
      const uint4 qv = *reinterpret_cast<const uint4*>(B.q + at);
      O = mma(qv, h, O);
      O = mma(qv, l, O);
      if (DELTA) {
        const uint4 kv = *reinterpret_cast<const uint4*>(B.k + at);
        U = mma(kv, h, U);
        U = mma(kv, l, U);
      }
    }
}

template <int KT, int NW, bool DELTA>
__global__ void __launch_bounds__(64 * (NW + 2))
head_scan_chunk16_kernel(const HeadScanArgs<bf16> a) {
  constexpr int DKP = 32 * KT;
  constexpr int NI = (DKP + 63) / 64;          // items per producer lane and matrix
  using Buf = ChunkBuf<DKP, DELTA>;
  __shared__ Buf s_buf[2];
  __shared__ __align__(16) double s_L[kC];     // the producers': log-decay sums, unit factors
  __shared__ __align__(16) float s_fk[2][kC];
  const int sg = blockIdx.x, hd = blockIdx.y;
  const int r0 = a.cu[sg], len = a.cu[sg + 1] - r0;
  if (len <= 0) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 31, hi = lane >> 5;
  const int Dk = a.Dk, Dv = a.Dv;
  const int chunks = (len + kC - 1) / kC;
  const int qcol = (hd / a.rep) * Dk;

  if (w >= NW) {
    // ---------------- the producer waves ----------------
    const bool is_k = w > NW;
    const bf16* base = is_k ? a.k : a.q;
    const long long ldr = is_k ? a.ldk : a.ldq;
    Item it[NI];
    float ra = 0.f, rb = 0.f;                  // the token's decay and write-strength logits
    auto fetch = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < NI; ++x) fetch_item<DKP>(it[x], base, ldr, qcol, r0, t0, len, Dk, a.vec, lane + 64 * x);
      if (!is_k) {
        const long long i = r0 + min(t0 + c, len - 1);
        if (a.a != nullptr) ra = to_f32(a.a[i * a.lda + hd]);
        if (DELTA) rb = to_f32(a.b[i * a.ldb + hd]);
      }
    };
    const HeadRates rates(a, hd);
    double L = 0.0, Lc = 0.0;                  // (the q wave) the lane's log-decay sum, the chunk's
    fetch(0);
    for (int n = 0; n <= chunks; ++n) {        // chunk n is built while the others run chunk n - 1
      const Chunk B = s_buf[n & 1].view();
      if (n < chunks) {                        // phase 1: rows into LDS, decays
        const int t0 = n * kC;
#pragma unroll
        for (int x = 0; x < NI; ++x) put_item<DKP>(it[x], is_k, a.silu_in, lane + 64 * x, is_k ? B.k : B.q, B.kt);
        if (!is_k) token_decays<DELTA>(rates, t0 + c < len, ra, rb, c, hi, L, Lc, s_L, B.w);
        if (t0 + kC < len) fetch(t0 + kC);     // the next chunk's rows travel meanwhile
      }
      __syncthreads();
      if (n < chunks) {
        if (!is_k) chunk_weights<KT, DELTA>(B, s_L, s_fk[0], L, Lc, c, hi, a.q_scale, a.key_eps);
        else if (DELTA) chunk_inverse<KT>(B, s_L, s_fk[1], lane, a.key_eps);
      }
      __syncthreads();
    }
    return;
  }

  // ---------------- the column waves ----------------
  const int col = (blockIdx.z * NW + w) * 32 + c;
  const bool on = col < Dv;
  const bf16* vp = a.v + (long long)r0 * a.ldv + (long long)hd * Dv + (on ? col : 0);
  State<KT> S;
  bf16 vn[16];                                 // the next chunk's values
  const auto fetch_v = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) vn[r] = vp[(long long)min(t0 + 8 * (r >> 2) + 4 * hi + (r & 3), len - 1) * a.ldv];
  };
  float* sp = a.state + ((long long)a.slot[sg] * a.H + hd) * Dk * Dv + col;
  state_load<KT>(S, sp, a.start[sg] == 0, on, Dk, Dv, hi);
  const float skip = a.skip != nullptr ? a.skip[hd] : 0.f;
  const long long ldo = (long long)a.H * Dv;
  float* op = a.out + (long long)r0 * ldo + (long long)hd * Dv + col;
  fetch_v(0);
  __syncthreads();
  __syncthreads();
  for (int ch = 0; ch < chunks; ++ch) {
    const Chunk B = s_buf[ch & 1].view();
    const int t0 = ch * kC;
    float V[16];
    take_values(vn, a.silu_in, V);
    if (ch + 1 < chunks) fetch_v(t0 + kC);
    f32x16 O, U;
    state_read<KT, DELTA>(S, B, O, U, c, hi);
    __syncthreads();
    U = chunk_writes<DELTA>(B, U, V, c, hi);
    O = chunk_apply(B.p0, B.p1, U, old_state_read(B, O, V, skip, hi), c, hi);
    if (on) store_rows(O, min(kC, len - t0), op + (long long)(t0 + 4 * hi) * ldo, ldo, hi);
    state_move<KT>(S, B, Keys<KT>(B, c, hi), U, hi);
    __syncthreads();
  }
  if (on) state_store<KT>(S, sp, Dk, Dv, hi);
}

template <bool DELTA>
hipError_t launch(const HeadScanArgs<bf16>& a, int n_seg, hipStream_t st) {
  // 32-column blocks; a grid that leaves half the CUs idle is cut finer (each column block's result
  // is the same whichever workgroup computes it)
  const int cb = (a.Dv + 31) / 32;
  const bool fine = cb > 2 && (long long)n_seg * a.H * ((cb + 3) / 4) <= 128;
#define GO(KT, NW)                                                             \
  head_scan_chunk16_kernel<KT, NW, DELTA>                                      \
      <<<dim3(n_seg, a.H, (cb + NW - 1) / NW), 64 * (NW + 2), 0, st>>>(a)
#define GO_K(KT)                                                               \
  if (cb == 1) GO(KT, 1);                                                      \
  else if (cb == 2 || fine) GO(KT, 2);                                         \
  else if (cb == 3) GO(KT, (KT == 8 ? 2 : 3));                                 \
  else GO(KT, (KT == 8 ? 2 : 4))   /* 256 state rows: two column waves' registers */
  if (a.Dk <= 32) { GO_K(1); }
  else if (a.Dk <= 64) { GO_K(2); }
  else if (a.Dk <= 128) { GO_K(4); }
  else { GO_K(8); }
#undef GO_K
#undef GO
  return hipGetLastError();
}

}  // namespace

namespace lumen {

hipError_t head_scan_chunk16(const HeadScanArgs<bf16>& args, bool delta, int n_seg,
                             hipStream_t st) {
  HeadScanArgs<bf16> a = args;
  a.vec = a.Dk % 8 == 0 && a.ldq % 8 == 0 && a.ldk % 8 == 0 && (uintptr_t)a.q % 16 == 0 &&
          (uintptr_t)a.k % 16 == 0;
  return delta ? launch<true>(a, n_seg, st) : launch<false>(a, n_seg, st);
}

}  // namespace lumen
