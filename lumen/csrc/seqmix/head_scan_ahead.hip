// The chunked matrix-state recurrences of head_scan_chunk16.hip with every chunk's matrices built ahead, for steps whose
// sequences and heads leave the chip idle: a prompt is a serial chain of chunks there, and a chunk costs as long as its producer
// waves take to build it (32 heads of 128: delta rule 5.5 us, most of it the triangle's inverse in one wave; 3.3 without, 2.1 with constant decays).
//
// None of that depends on the state.  chunk_prep_kernel builds all chunks at once, a workgroup per chunk and key head: rows of q
// and k (transposed once more) into LDS, then a wave forms G . Q K^T and the factors, and another the inverse, per head.  Its LDS
// images go to memory as they are.  chunk_run_kernel has four waves per 32 columns of a head's state.  Two own half of its
// rows each and move it on, which is the chain (with the delta rule they add in LDS what the halves gave); they leave its parts in
// LDS.  One forms the read-outs a chunk later.  One fetches, LDS-DMA of whole images and rows of values.  They meet once a chunk
// (twice with the delta rule).
// Cycles a chunk at width 2048, busy: state waves 4030 (delta) and 2670, read-outs 2040 and 3010, fetching 1000 - 1400.  One state wave that
// owned all rows was busy 5710 and 4000; one wave that formed the read-outs too took 2.9 and 2.05 us a chunk, now 1.85 and 1.25 (32 heads: 2.1 and 1.35).
#include "head_chunk16.h"

using namespace lumen;
using namespace lumen::hc16;

namespace {

constexpr int up1k(int n) { return (n + 1023) / 1024 * 1024; }

// A chunk's images, in multiples of 1 KB: what moves the state (rows of a key head SA: k with the delta rule, k transposed; of a
// head SB: the inverse, factors) and what the read-outs take (q: RA; G . Q K^T, its factor and step sizes once more: RB)
template <int KT, bool DELTA> struct Images {
  static constexpr int DKP = 32 * KT, ROWS = kC * (DKP + 8) * 2, KTB = DKP * LT * 2, MAT = kC * LT * 2;
  static constexpr int SA = up1k((DELTA ? ROWS : 0) + KTB), RA = up1k(ROWS);
  static constexpr int SF = DELTA ? 2 * MAT : 0, RF = 2 * MAT;             // the factors' places
  static constexpr int SB = up1k(SF + 3 * kC * 4 + 16), RB = up1k(RF + 2 * kC * 4);
  static constexpr int KEY = SA + RA, HEAD = SB + RB, ALL = KEY + HEAD;    // (in memory: SA RA of a key head, SB RB of a head)
  static __device__ __forceinline__ Chunk view(char* sa, char* ra, char* sb, char* rb) {
    float *f = reinterpret_cast<float*>(sb + SF), *g = reinterpret_cast<float*>(rb + RF);
    return Chunk{(bf16*)ra, (bf16*)sa, (bf16*)(DELTA ? sa + ROWS : sa), (bf16*)rb, (bf16*)(rb + MAT),
                 (bf16*)sb, (bf16*)(DELTA ? sb + MAT : sb), g, f, f + kC, f + 2 * kC, f + 3 * kC};
  }
  static __device__ __forceinline__ float* read_w(char* rb) { return reinterpret_cast<float*>(rb + RF) + kC; }
};

// chunks of the segments before `n` (every lane), a wave's work
__device__ __forceinline__ int chunks_before(const int* cu, int n, int lane) {
  int sum = 0;
  for (int s = lane; s < n; s += 64) sum += (cu[s + 1] - cu[s] + kC - 1) / kC;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  return __builtin_amdgcn_readfirstlane(sum);
}

// chunk number `at` of the step -> its segment and place there; false past the last one
__device__ __forceinline__ bool find_chunk(const int* cu, int n_seg, int at, int lane, int& sg, int& ch) {
  for (int s0 = 0; s0 < n_seg; s0 += 64) {
    const int s = s0 + lane, n = s < n_seg ? (cu[s + 1] - cu[s] + kC - 1) / kC : 0;
    int sum = n;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int o = __shfl_up(sum, m, 64);
      if (lane >= m) sum += o;
    }
    const unsigned long long past = __ballot(sum > at);
    if (past) {
      const int i = __builtin_ctzll(past);
      sg = __builtin_amdgcn_readfirstlane(s0 + i);
      ch = __builtin_amdgcn_readfirstlane(at - (__shfl(sum, i, 64) - __shfl(n, i, 64)));
      return true;
    }
    at -= __builtin_amdgcn_readfirstlane(__shfl(sum, 63, 64));
  }
  return false;
}

template <int KT, bool DELTA>
__global__ void __launch_bounds__(256)
chunk_prep_kernel(const HeadScanArgs<bf16> a, int n_seg, char* __restrict__ ws) {
  using Im = Images<KT, DELTA>;
  constexpr int DKP = Im::DKP, HPB = DELTA ? 2 : 4;        // heads of a workgroup
  static_assert(2 * DKP <= 256, "an item a thread");
  constexpr int ROWS = Im::ROWS;
  // without the delta rule k is no part of the images: it lies behind them
  __shared__ __attribute__((aligned(16))) char s_a[Im::KEY + (DELTA ? 0 : ROWS)];
  __shared__ __attribute__((aligned(16))) char s_b[HPB][Im::HEAD];
  __shared__ __attribute__((aligned(16))) double s_L[4][kC];
  __shared__ __attribute__((aligned(16))) float s_fk[4][kC], s_be[4][kC];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, hi = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int sg, ch;
  if (!find_chunk(a.cu, n_seg, blockIdx.x, lane, sg, ch)) return;
  const int g = blockIdx.y, G = gridDim.y, h0 = g * a.rep + blockIdx.z * HPB, nh = min(HPB, (g + 1) * a.rep - h0);
  const int r0 = a.cu[sg], len = a.cu[sg + 1] - r0, t0 = ch * kC;
  const int mine = DELTA ? w >> 1 : w, hd = h0 + min(mine, nh - 1);
  const bool inverse = DELTA && (w & 1);
  float ra = 0.f, rb = 0.f;
  {
    const long long i = r0 + min(t0 + c, len - 1);
    if (a.a != nullptr) ra = to_f32(a.a[i * a.lda + hd]);
    if (DELTA) rb = to_f32(a.b[i * a.ldb + hd]);
  }
  char* head = s_b[min(mine, HPB - 1)];
  Chunk B = Im::view(s_a, s_a + Im::SA, head, head + Im::SB);
  if (!DELTA) B.k = reinterpret_cast<bf16*>(s_a + Im::KEY);
  if (tid < 2 * DKP) {
    const bool is_k = tid >= DKP;
    const int item = tid & (DKP - 1);
    Item it;
    fetch_item<DKP>(it, is_k ? a.k : a.q, is_k ? a.ldk : a.ldq, g * a.Dk, r0, t0, len, a.Dk, a.vec, item);
    put_item<DKP>(it, is_k, a.silu_in, item, is_k ? B.k : B.q, B.kt);
  }
  const HeadRates rates(a, hd);
  double L, Lc;
  if (inverse) B.w = s_be[w];
  if (mine < nh) {
    token_decays<DELTA>(rates, t0 + c < len, ra, rb, c, hi, L, Lc, s_L[w], B.w);
    if (!inverse && hi == 0) Im::read_w(head + Im::SB)[c] = B.w[c];        // (this lane's own)
  }
  __syncthreads();
  const long long at = blockIdx.x;
  if (blockIdx.z == 0) {
    uint4* dst = reinterpret_cast<uint4*>(ws + (at * G + g) * Im::KEY);
    for (int i = tid; i < Im::KEY / 16; i += 256) dst[i] = reinterpret_cast<const uint4*>(s_a)[i];
  }
  if (mine < nh) {
    if (!inverse) chunk_weights<KT, DELTA>(B, s_L[w], s_fk[w], L, Lc, c, hi, a.q_scale, a.key_eps);
    else if constexpr (DELTA) chunk_inverse<KT>(B, s_L[w], s_fk[w], lane, a.key_eps);
  }
  __syncthreads();
  uint4* dst = reinterpret_cast<uint4*>(ws + (long long)gridDim.x * G * Im::KEY + (at * a.H + h0) * Im::HEAD);
  for (int i = tid; i < nh * (Im::HEAD / 16); i += 256) dst[i] = reinterpret_cast<const uint4*>(s_b)[i];
}

// all: chunk_prep_kernel's grid
template <int KT, bool DELTA>
__global__ void __launch_bounds__(64 * ((KT > 1 ? 2 : 1) + 2))
chunk_run_kernel(const HeadScanArgs<bf16> a, const char* __restrict__ ws, int all) {
  using Im = Images<KT, DELTA>;
  constexpr int NS = KT > 1 ? 2 : 1, KS = KT / NS;          // state waves, 32-row blocks of each
  constexpr int VB = kC * 64, SS = Im::SA + Im::SB + VB, RS = Im::RA + Im::RB + (DELTA ? 0 : VB);     // slots of the two rings
  constexpr int LK = 32 * KT + 8, XS = KT * 2 * 2 * 64, XU = DELTA ? 2 * 2 * 64 : 0, XP = DELTA && NS > 1 ? 4 * 64 : 0;
  __shared__ __attribute__((aligned(1024))) char lds[2 * SS + 3 * RS + 16 * (2 * (XS + XU) + NS * XP)];
  static_assert(sizeof(lds) <= 163840, "LDS");
  const int sg = blockIdx.x, hd = blockIdx.y;
  const int r0 = a.cu[sg], len = a.cu[sg + 1] - r0;
  if (len <= 0) return;
  const int lane = threadIdx.x & 63, c = lane & 31, hi = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunks = (len + kC - 1) / kC;
  // In step ch the state waves take chunk ch (two slots), the read-out wave chunk ch - 1 (three), and chunk ch + 1 lands.  All
  // waves meet at a step's end, and once within it where the state waves add what they read (delta rule).
  const auto meet = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  char* const ring_r = lds + 2 * SS;

  if (w == NS + 1) {
    // ---------------- the fetching wave ----------------
    const int G = a.H / a.rep, g = hd / a.rep;
    const long long at = chunks_before(a.cu, sg, lane);
    const char* pa = ws + (at * G + g) * Im::KEY;
    const char* pb = ws + (long long)all * G * Im::KEY + (at * a.H + hd) * Im::HEAD;
    const char* pv = reinterpret_cast<const char*>(a.v + (long long)r0 * a.ldv + (long long)hd * a.Dv);
    const unsigned voff = 2 * min((int)blockIdx.z * 32 + 8 * (lane & 3), a.Dv - 8);
    const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds);
    const auto issue = [&](int ch) __attribute__((always_inline)) {
      const char *sa = pa + (long long)ch * G * Im::KEY, *sb = pb + (long long)ch * a.H * Im::HEAD;
      const unsigned ds = __builtin_amdgcn_readfirstlane(lds0 + (ch & 1) * SS);
      const unsigned dr = __builtin_amdgcn_readfirstlane(lds0 + 2 * SS + (ch % 3) * RS);
#pragma unroll
      for (int p = 0; p < Im::KEY / 1024; ++p) dma16(sa, 1024 * p + 16 * lane, p < Im::SA / 1024 ? ds + 1024 * p : dr + 1024 * p - Im::SA);
#pragma unroll
      for (int p = 0; p < Im::HEAD / 1024; ++p)
        dma16(sb, 1024 * p + 16 * lane, p < Im::SB / 1024 ? ds + Im::SA + 1024 * p : dr + Im::RA + 1024 * p - Im::SB);
      // the values' rows [token][32 columns], four lanes a row (columns past the head's repeat its last ones)
      const int t0 = ch * kC;
      const char* sv = pv + (long long)t0 * a.ldv * 2;
#pragma unroll
      for (int p = 0; p < VB / 1024; ++p) {
        const unsigned off = (unsigned)(min(t0 + 16 * p + (lane >> 2), len - 1) - t0) * (unsigned)(2 * a.ldv) + voff;
        dma16(sv, off, ds + Im::SA + Im::SB + 1024 * p);
        if (!DELTA) dma16(sv, off, dr + Im::RA + Im::RB + 1024 * p);
      }
    };
    issue(0);
    wait_vm<0>();
    meet();
    for (int ch = 0; ch < chunks; ++ch) {
      if (ch + 1 < chunks) issue(ch + 1);
      if (XP) meet();
      wait_vm<0>();
      meet();
    }
    return;
  }

  const int Dk = a.Dk, Dv = a.Dv, col = blockIdx.z * 32 + c;
  const bool on = col < Dv;
  // from the state waves to the read-out wave: the state's and (delta) the writes' parts as right operands, two chunks' room;
  // from one state wave to the other: what it read of the state
  uint4* xs = reinterpret_cast<uint4*>(ring_r + 3 * RS);
  uint4* xu = xs + 2 * XS;
  f32x4* xp = reinterpret_cast<f32x4*>(xu + 2 * XU);
  float V[16];
  const auto values = [&](const char* at) __attribute__((always_inline)) {
    const bf16* v = reinterpret_cast<const bf16*>(at) + c;
    bf16 x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) x[r] = v[(8 * (r >> 2) + 4 * hi + (r & 3)) * 32];
    take_values(x, a.silu_in, V);
  };

  if (w < NS) {
    // ---------------- the state waves: rows 32 KS w .. ----------------
    const int kt0 = KS * w;
    State<KS> S;
    float* sp = a.state + (((long long)a.slot[sg] * a.H + hd) * Dk + 32 * kt0) * Dv + col;
    state_load<KS>(S, sp, a.start[sg] == 0, on, Dk - 32 * kt0, Dv, hi);
    meet();
    for (int ch = 0; ch < chunks; ++ch) {
      char* st = lds + (ch & 1) * SS;
      const Chunk B = Im::view(st, nullptr, st + Im::SA, nullptr);
      uint4 *ps = xs + (ch & 1) * XS + 256 * kt0 + lane, *pu = xu + (ch & 1) * XU + lane;
      const Keys<KS> kt(B, 32 * kt0 + c, hi);
      values(st + Im::SA + Im::SB);
      f32x16 U;
#pragma unroll
      for (int r = 0; r < 16; ++r) U[r] = 0.f;
#pragma unroll
      for (int x = 0; x < KS; ++x)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          uint4 h, l;
          split8(S.r[x], s, h, l);
          ps[128 * (2 * x + s)] = h;
          ps[128 * (2 * x + s) + 64] = l;
          if (DELTA) {
            const uint4 kv = *reinterpret_cast<const uint4*>(B.k + c * LK + 32 * (kt0 + x) + 16 * s + 8 * hi);
            U = mma(kv, h, U);
            U = mma(kv, l, U);
          }
        }
      if (XP) {
        f32x4 *mine = xp + XP * w + lane, *other = xp + XP * (w ^ 1) + lane;
#pragma unroll
        for (int q = 0; q < 4; ++q) mine[64 * q] = f32x4{U[4 * q], U[4 * q + 1], U[4 * q + 2], U[4 * q + 3]};
        meet();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 o = other[64 * q];
#pragma unroll
          for (int e = 0; e < 4; ++e) U[4 * q + e] += o[e];
        }
      }
      U = chunk_writes<DELTA>(B, U, V, c, hi);
      if (DELTA) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          if (NS > 1 && s != w) continue;
          uint4 h, l;
          split8(U, s, h, l);
          pu[128 * s] = h;
          pu[128 * s + 64] = l;
        }
      }
      state_move<KS>(S, B, kt, U, hi);
      meet();
    }
    if (on) state_store<KS>(S, sp, Dk - 32 * kt0, Dv, hi);
    return;
  }

  // ---------------- the read-out wave ----------------
  const float skip = a.skip != nullptr ? a.skip[hd] : 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) V[r] = 0.f;
  const long long ldo = (long long)a.H * Dv;
  float* op = a.out + (long long)r0 * ldo + (long long)hd * Dv + col;
  meet();
  if (XP) meet();
  meet();
  int slot = 0;
  for (int ch = 0; ch < chunks; ++ch) {
    char* st = ring_r + slot * RS;
    Chunk B = Im::view(nullptr, st, nullptr, st + Im::RA);
    B.w = Im::read_w(st + Im::RA);
    const uint4 *ps = xs + (ch & 1) * XS + lane, *pu = xu + (ch & 1) * XU + lane;
    if (!DELTA) values(st + Im::RA + Im::RB);
    f32x16 O;
#pragma unroll
    for (int r = 0; r < 16; ++r) O[r] = 0.f;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const uint4 qv = *reinterpret_cast<const uint4*>(B.q + c * LK + 32 * kt + 16 * s + 8 * hi);
        O = mma(qv, ps[128 * (2 * kt + s)], O);
        O = mma(qv, ps[128 * (2 * kt + s) + 64], O);
      }
    if (XP && ch + 1 < chunks) meet();
    O = old_state_read(B, O, V, skip, hi);
    if (DELTA) {
#pragma unroll
      for (int s = 0; s < 2; ++s) O = apply_half(B.p0, B.p1, s, pu[128 * s], pu[128 * s + 64], O, c, hi);
    } else {
      O = chunk_apply(B.p0, B.p1, chunk_writes<DELTA>(B, O, V, c, hi), O, c, hi);
    }
    if (on) store_rows(O, min(kC, len - ch * kC), op + (long long)(ch * kC + 4 * hi) * ldo, ldo, hi);
    slot = slot + 1 == 3 ? 0 : slot + 1;
    if (ch + 1 < chunks) meet();
  }
}

template <int KT, bool DELTA>
hipError_t launch(const HeadScanArgs<bf16>& a, int n_seg, char* ws, int chunks, hipStream_t st) {
  constexpr int HPB = DELTA ? 2 : 4;
  chunk_prep_kernel<KT, DELTA><<<dim3(chunks, a.H / a.rep, (a.rep + HPB - 1) / HPB), 256, 0, st>>>(a, n_seg, ws);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  chunk_run_kernel<KT, DELTA><<<dim3(n_seg, a.H, (a.Dv + 31) / 32), 64 * ((KT > 1 ? 2 : 1) + 2), 0, st>>>(a, ws, chunks);
  return hipGetLastError();
}

template <bool DELTA> long long bytes(int Dk, int H, int rep, int chunks) {
  const long long g = H / rep;
#define SIZE(KT) chunks * (g * Images<KT, DELTA>::KEY + (long long)H * Images<KT, DELTA>::HEAD)
  return Dk <= 32 ? SIZE(1) : Dk <= 64 ? SIZE(2) : SIZE(4);
#undef SIZE
}

}  // namespace

extern "C" {

// Bytes of the workspace for a step of at most `chunks` chunks, 0 for sizes without such a kernel
long long sm_head_scan_ahead_bytes(int delta, int Dk, int H, int rep, int chunks) {
  if (Dk < 1 || Dk > 128 || rep < 1 || H < 1 || H % rep || H > 65535 || chunks < 1) return 0;
  return delta ? bytes<true>(Dk, H, rep, chunks) : bytes<false>(Dk, H, rep, chunks);
}

// As sm_head_scan_chunk for bf16, Dk <= 128 and rows of v in multiples of 16 bytes, with a workspace (16-byte base) of sm_head_scan_ahead_bytes(chunks); chunks: at least
// the sum of ceil(rows / 32) over the segments
hipError_t sm_head_scan_ahead(int dt, int delta, const void* q, long long ldq, const void* k, long long ldk, const void* v,
                              long long ldv, const void* al, long long lda, const void* bl, long long ldb, const float* A_log,
                              const float* dt_bias, const float* log_decay, const float* skip, float* state, float* out,
                              const int* cu, const int* slot, const int* start, int n_seg, int H, int rep, int Dk, int Dv,
                              int silu_in, float key_eps, float q_scale, void* ws, int chunks, hipStream_t st) {
  if (n_seg == 0) return hipSuccess;
  if (dt != kBF16 || Dv < 1 || n_seg < 0 || !ws || (uintptr_t)ws % 16 || !sm_head_scan_ahead_bytes(delta, Dk, H, rep, chunks) ||
      (al == nullptr) == (log_decay == nullptr) || (al && (!A_log || !dt_bias)) || (delta && (!bl || !al)) || Dv % 8 ||
      ldv % 8 || (uintptr_t)v % 16 || ldv >= 1LL << 25)
    return hipErrorInvalidValue;
  const int vec = Dk % 8 == 0 && ldq % 8 == 0 && ldk % 8 == 0 && (uintptr_t)q % 16 == 0 && (uintptr_t)k % 16 == 0;
  const HeadScanArgs<bf16> a{(const bf16*)q, ldq, (const bf16*)k, ldk, (const bf16*)v, ldv, (const bf16*)al, lda,
                             (const bf16*)bl, ldb, A_log, dt_bias, log_decay, skip, state, out, cu, slot, start,
                             H, rep, Dk, Dv, silu_in, vec, key_eps, q_scale};
  char* w = (char*)ws;
  if (Dk <= 32) return delta ? launch<1, true>(a, n_seg, w, chunks, st) : launch<1, false>(a, n_seg, w, chunks, st);
  if (Dk <= 64) return delta ? launch<2, true>(a, n_seg, w, chunks, st) : launch<2, false>(a, n_seg, w, chunks, st);
  return delta ? launch<4, true>(a, n_seg, w, chunks, st) : launch<4, false>(a, n_seg, w, chunks, st);
}

}  // extern "C"
