// Latent attention over a step's prompt portions: one key/value head whose value is the first Dv columns
// of the key row, a 16-bit cache and its per-block transposed copy `vt` (see row_attention.hip, whose
// latent_attn_kernel does the same for single rows and holds the scoring rules).
//
// What bounded the row kernel on prompts: a workgroup was one row (its 16 heads are the product's columns),
// so every row pulled the whole key range through L2 for itself, 2.85 GB a call at 8 x 512 tokens, with
// dependent table, address and load chains per tile.  Here a workgroup is eight consecutive rows of a
// segment and 16 heads, a wave two of the rows:
//  * the tile of 32 keys arrives by LDS-DMA one tile ahead -- the key rows (16-byte chunks XOR-swizzled
//    through the source address) and, from `vt`, their values per channel -- and is shared by the
//    eight rows: an operand read from LDS feeds both rows of a wave;
//  * scores S^T = K Q^T (v_mfma_f32_16x16x32, the queries in registers for the whole walk) leave lane
//    (head, group g) the keys 4 g + i of both 16-key halves; the value product contracts over the same
//    keys in the same places (a contraction may order its keys freely), so the weights feed it from the
//    registers they are formed in, as a 16-bit head plus a 16-bit remainder, and the accumulator's
//    column stays the head: no exchange between lanes but the maximum over the four groups;
//  * accumulators [512 x 16 heads] of two rows are 256 registers, one wave per SIMD.  They are never
//    rescaled: a first walk over the key rows finds every (row, head)'s maximum, the second forms the
//    weights against it.  (The walk costs a third of the products again; with a running maximum the
//    compiler moved the accumulators out of the matrix registers, ~270 of them through scratch.)
// Measured (16 heads, 512 + 64 / 512, bf16) against the row kernel: 14 prompts of 63 - 509 tokens 234 -> 159
// us, 8 x 512 251 -> 195 us, one prompt of 4096 2771 -> 1339 us; one of 512 tokens (64 workgroups) 53 -> 94 us,
// hence the rule in ops/attention.py.  A tile costs a wave ~5.9 us, twice its matrix instructions' time: one
// wave per SIMD, whose softmax and masks do not overlap its products.  Eight waves of one row each were
// slower (231 us): operand reads double and the accumulators spill.
#include "mma.h"

using namespace lumen;

namespace {

constexpr int kRows = 8;          // rows of a workgroup (two per wave)
constexpr int kKeys = 32;         // keys per tile
constexpr int kTable = 4096;      // cache blocks of a segment (held in LDS)

template <typename T> struct LatentTileArgs {
  const T* q1; long long q1r, q1h; int D1;
  const T* q2; long long q2r, q2h;
  const T* kc; long long krow;
  const T* vt;
  T* out; long long our, ouh;
  const int* tables; int maxb;
  const int *q_tiles, *cu, *start;     // [n][2] (segment, first row); tiles of tile_rows rows
  int n_wg, subs, tile_rows;
  int H, bsh;                          // cache blocks of 1 << bsh tokens
  float scale, softcap, tcoef; int tevery;
  const float *r1, *r2, *sink;
  const T* gate; long long gater;
};

// 16-byte chunk c of key row r lies at chunk c ^ swz(r) of rows of 1024 bytes (tail(r): of 128 bytes), so
// that a fragment read (16 rows at one chunk) touches 16 different bank slots
__device__ __forceinline__ int swz(int r) { return r & 15; }
__device__ __forceinline__ int tail(int r) { return (r >> 1) & 7; }

// LDS-DMA of 16 bytes per lane (wave-uniform base + 32-bit lane offset); ordered by the kernel's waits
__device__ __forceinline__ void dma16(const void* base, unsigned off, const char* lds_wave_base) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(lds_wave_base))));
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(m0) : "memory", "m0");
}

// the first n (clamped to 0 .. 4) of four 16-bit elements
__device__ __forceinline__ uint2 keep4(int n) {
  const unsigned long long m = n >= 4 ? ~0ull : n <= 0 ? 0ull : (1ull << (16 * n)) - 1;
  return make_uint2((unsigned)m, (unsigned)(m >> 32));
}

// Dv = 512; DK = 512, or 576 with a second query part.  LDS of a tile: rows of 64 chunks (16 bytes), the
// last 8 chunks of DK = 576 in rows of their own, then the values
// (SHAPED: a soft cap or a distance bias between product and softmax)
template <typename T, int DK, bool SHAPED>
__global__ void __launch_bounds__(256, 1) latent_tile_kernel(const LatentTileArgs<T> a) {
  constexpr int Dv = 512, KS = DK / 32, NT = Dv / 16;
  constexpr bool TAIL = DK == 576;
  static_assert(DK == 512 || DK == 576, "key size");
  constexpr int KB = kKeys * DK * 2, VB = kKeys * Dv * 2;
  __shared__ __attribute__((aligned(16))) char lds[2 * (KB + VB)];
  __shared__ int s_tbl[kTable];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  // every tile's last rows first, its first ones (fewest keys) last: consecutive workgroups belong to
  // different tiles, so long and short walks mix on every XCD
  const int n_tiles = a.n_wg / a.subs;
  const int sub = a.subs - 1 - blockIdx.x / n_tiles, tile = blockIdx.x % n_tiles;
  const int seg = a.q_tiles[2 * tile], first = a.q_tiles[2 * tile + 1] + kRows * sub;
  const int end = min(a.cu[seg + 1], a.q_tiles[2 * tile + 1] + a.tile_rows);
  if (first >= end) return;
  const int p0 = a.start[seg] - a.cu[seg];                    // position = row + p0
  const int kmax = min(first + kRows, end) - 1 + p0;          // the workgroup's last key
  const int h0 = blockIdx.y * 16, nh = min(16, a.H - h0);
  const bool head_on = lr < nh;
  const int h = h0 + (head_on ? lr : 0);

  {
    const int* tbl = a.tables + (long long)seg * a.maxb;
    for (int i = threadIdx.x; i <= kmax >> a.bsh; i += 256) s_tbl[i] = tbl[i];
  }
  // the wave's two rows (past the end: the last row again, not stored) and their queries
  int row[2], pos[2];
  uint4 qf[2][KS];
  float qs[2], m[2], l[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    row[q] = min(first + 2 * w + q, end - 1);
    pos[q] = row[q] + p0;
    const T* b1 = a.q1 + row[q] * a.q1r + h * a.q1h;
    const T* b2 = a.q2 + row[q] * a.q2r + h * a.q2h - a.D1;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int d = 32 * k + 8 * lg;
      qf[q][k] = make_uint4(0u, 0u, 0u, 0u);
      if (head_on) qf[q][k] = *reinterpret_cast<const uint4*>((d < a.D1 ? b1 : b2) + d);
    }
    float temp = 1.f;
    if (a.tevery > 0 && a.tcoef != 0.f)
      temp = 1.f + a.tcoef * logf((float)((pos[q] + 1) / a.tevery) + 1.f);
    qs[q] = a.scale * temp;
    m[q] = a.sink != nullptr ? a.sink[h] : -INFINITY;         // the sink: a key without a value
    l[q] = 0.f;
  }
  const float r1 = a.r1 != nullptr ? a.r1[h] : 0.f, r2 = a.r1 != nullptr ? a.r2[h] : 0.f;
  f32x4 O[2][NT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int n = 0; n < NT; ++n) O[q][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();

  // wave w stages key rows 8 w .. 8 w + 7 and 256 channels of one 16-key half's values: each lies in
  // one cache block (of at least 16 tokens).  Keys past the last one repeat it.
  const unsigned voff = ((unsigned)((w & 1) * 256 + (lane >> 1)) << (a.bsh + 1)) + 16 * (lane & 1);
  const auto issue = [&](int j0, char* buf, bool values) __attribute__((always_inline)) {
    const int bm = (1 << a.bsh) - 1;
    const int k8 = min(j0 + 8 * w, kmax);
    const long long blk = __builtin_amdgcn_readfirstlane(s_tbl[k8 >> a.bsh]);
    const T* kbase = a.kc + (blk << a.bsh) * a.krow;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int key = min(j0 + 8 * w + r, kmax) & bm;
      dma16(kbase + key * a.krow, 16u * (lane ^ swz(8 * w + r)), buf + (8 * w + r) * 1024);
    }
    if constexpr (TAIL) {
      const int r = lane >> 3, key = min(j0 + 8 * w + r, kmax) & bm;
      dma16(kbase + 512, (unsigned)(key * (int)a.krow * 2) + 16u * ((lane & 7) ^ tail(8 * w + r)),
            buf + kKeys * 1024 + w * 1024);
    }
    if (!values) return;
    const int v16 = min(j0 + 16 * (w >> 1), kmax & ~15);
    const long long vblk = __builtin_amdgcn_readfirstlane(s_tbl[v16 >> a.bsh]);
    const T* vbase = a.vt + ((vblk * Dv) << a.bsh) + (v16 & bm);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      dma16(vbase + ((32 * i) << a.bsh), voff, buf + KB + (8 * w + i) * 1024);
  };
  // scores of the tile in `kb`: sv[q][i] is key j0 + 16 (i >> 2) + 4 lg + (i & 3) (-inf: not seen)
  float sv[2][8];
  const auto score = [&](int j0, const char* kb) __attribute__((always_inline)) {
    f32x4 s[2][2];
#pragma unroll
    for (int q = 0; q < 2; ++q) s[q][0] = s[q][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    // key fragments run two groups (of two k steps and both 16-key halves) ahead of their products
    constexpr int NGRP = KS / 2;
    uint4 f[3][4];
    const auto load = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = 2 * g + (u >> 1), r = 16 * (u & 1) + lr;
        f[g % 3][u] = *reinterpret_cast<const uint4*>(
            k < 16 ? kb + r * 1024 + (((4 * k + lg) ^ swz(r)) << 4)
                   : kb + kKeys * 1024 + r * 128 + (((4 * (k - 16) + lg) ^ tail(r)) << 4));
      }
    };
    load(0);
    load(1);
#pragma unroll
    for (int g = 0; g < NGRP; ++g) {
      if (g + 2 < NGRP) load(g + 2);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s[0][u & 1] = Mfma<T>::run(f[g % 3][u], qf[0][2 * g + (u >> 1)], s[0][u & 1]);
        s[1][u & 1] = Mfma<T>::run(f[g % 3][u], qf[1][2 * g + (u >> 1)], s[1][u & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int j = j0 + 16 * (i >> 2) + 4 * lg + (i & 3);
        float v = s[q][i >> 2][i & 3] * qs[q];
        if constexpr (SHAPED) {
          if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
          if (a.r1 != nullptr) v -= r1 * logf(1.f + r2 * (float)(pos[q] - j));
        }
        sv[q][i] = j <= pos[q] ? v : -INFINITY;
      }
  };
  // the tile in the current buffer has landed for every wave, and every wave is done with the other one
  const auto turn = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // ---- first walk: the maxima ----
  issue(0, lds, false);
  for (int j0 = 0, cur = 0; j0 <= kmax; j0 += kKeys, cur ^= 1) {
    turn();
    if (j0 + kKeys <= kmax) issue(j0 + kKeys, lds + (cur ^ 1) * (KB + VB), false);
    score(j0, lds + cur * (KB + VB));
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int i = 0; i < 8; ++i) m[q] = fmaxf(m[q], sv[q][i]);
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    m[q] = fmaxf(m[q], __shfl_xor(m[q], 16, 64));
    m[q] = fmaxf(m[q], __shfl_xor(m[q], 32, 64));
    if (a.sink != nullptr && lg == 0) l[q] = expf(a.sink[h] - m[q]);   // (a lane's share of the sum)
  }
  turn();

  // ---- second walk: weights and values ----
  issue(0, lds, true);
  for (int j0 = 0, cur = 0; j0 <= kmax; j0 += kKeys, cur ^= 1) {
    turn();
    const char* kb = lds + cur * (KB + VB);
    if (j0 + kKeys <= kmax) issue(j0 + kKeys, lds + (cur ^ 1) * (KB + VB), true);
    score(j0, kb);
    uint4 ph[2], pl[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      float p[8], hi[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = sv[q][i] == -INFINITY ? 0.f : expf(sv[q][i] - m[q]);
        l[q] += p[i];
        hi[i] = to_f32(from_f32<T>(p[i]));
      }
      ph[q] = make_uint4(pk2<T>(hi[0], hi[1]), pk2<T>(hi[2], hi[3]), pk2<T>(hi[4], hi[5]),
                         pk2<T>(hi[6], hi[7]));
      pl[q] = make_uint4(pk2<T>(p[0] - hi[0], p[1] - hi[1]), pk2<T>(p[2] - hi[2], p[3] - hi[3]),
                         pk2<T>(p[4] - hi[4], p[5] - hi[5]), pk2<T>(p[6] - hi[6], p[7] - hi[7]));
    }
    const char* va = kb + KB + lr * 32 + lg * 8;
    uint2 lo[4], up[4];
    const auto load = [&](int n) __attribute__((always_inline)) {
      lo[n % 4] = *reinterpret_cast<const uint2*>(va + n * 512);
      up[n % 4] = *reinterpret_cast<const uint2*>(va + Dv * 32 + n * 512);
    };
    load(0);
    load(1);
    load(2);
    // keys past a row's position carry weight 0 but may hold anything: blanked row by row (in every
    // tile: a second copy of these products without it made the compiler keep the accumulators twice)
    uint2 ml[2], mu[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      ml[q] = keep4(pos[q] - (j0 + 4 * lg) + 1);
      mu[q] = keep4(pos[q] - (j0 + 16 + 4 * lg) + 1);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      if (n + 3 < NT) load(n + 3);
      const uint2 x = lo[n % 4], y = up[n % 4];
      uint4 v[2];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        v[q] = make_uint4(x.x & ml[q].x, x.y & ml[q].y, y.x & mu[q].x, y.y & mu[q].y);
      O[0][n] = Mfma<T>::run(v[0], ph[0], O[0][n]);
      O[1][n] = Mfma<T>::run(v[1], ph[1], O[1][n]);
      O[0][n] = Mfma<T>::run(v[0], pl[0], O[0][n]);
      O[1][n] = Mfma<T>::run(v[1], pl[1], O[1][n]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // O[q][n][i]: channel 16 n + 4 lg + i of head lr
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float sum = l[q];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (!head_on || first + 2 * w + q >= end) continue;
    float inv = 1.f / sum;
    if (a.gate != nullptr) inv /= 1.f + expf(-to_f32(a.gate[row[q] * a.gater + h]));
    T* op = a.out + row[q] * a.our + h * a.ouh + 4 * lg;
#pragma unroll
    for (int n = 0; n < NT; ++n)
      *reinterpret_cast<uint2*>(op + 16 * n) =
          make_uint2(pk2<T>(O[q][n][0] * inv, O[q][n][1] * inv),
                     pk2<T>(O[q][n][2] * inv, O[q][n][3] * inv));
  }
}

template <typename T>
hipError_t launch(const LatentTileArgs<T>& a, int Dk, hipStream_t st) {
  const dim3 grid(a.n_wg, (a.H + 15) / 16);
  const bool shaped = a.softcap > 0.f || a.r1 != nullptr;
  if (Dk == 512) {
    if (shaped) latent_tile_kernel<T, 512, true><<<grid, 256, 0, st>>>(a);
    else latent_tile_kernel<T, 512, false><<<grid, 256, 0, st>>>(a);
  } else {
    if (shaped) latent_tile_kernel<T, 576, true><<<grid, 256, 0, st>>>(a);
    else latent_tile_kernel<T, 576, false><<<grid, 256, 0, st>>>(a);
  }
  return hipGetLastError();
}

}  // namespace

extern "C" {

// Does sm_latent_tiles have a kernel: a latent of 512, alone or with 64 more key columns; cache blocks of a
// power of two from 16 to 4096 tokens, at most kTable of them per sequence; rows of at most 16384.
int sm_latent_tiles_ok(int dt, int Dv, int Dk, int D1, int bs, int maxb) {
  return (dt == kBF16 || dt == kF16) && Dv == 512 && (Dk == 512 || Dk == 576) && D1 % 8 == 0 &&
         bs >= 16 && bs <= 4096 && (bs & (bs - 1)) == 0 && maxb <= kTable;
}

// The first rows of a step, cut into n_tiles tiles of tile_rows rows (q_tiles [n][2]: segment, first row);
// the other arguments as sm_latent_attn.
hipError_t sm_latent_tiles(int dt, const void* q1, long long q1r, long long q1h, int D1, const void* q2,
                           long long q2r, long long q2h, int D2, const void* kc, long long krow,
                           const void* vt, int Dv, void* out, long long our, long long ouh,
                           const int* tables, int maxb, const int* q_tiles, int n_tiles, int tile_rows,
                           const int* cu, const int* start, int H, int bs, float scale, float softcap,
                           float tcoef, int tevery, const float* r1, const float* r2,
                           const float* sink, const void* gate, long long gater, hipStream_t st) {
  if (n_tiles == 0 || H == 0) return hipSuccess;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (!sm_latent_tiles_ok(dt, Dv, D1 + D2, D1, bs, maxb) || n_tiles < 0 || H < 0 || tile_rows < 1 ||
      krow % 8 || krow < D1 + D2 || krow > 16384 || !al(kc) || !al(vt) || !al(q1) || q1r % 8 || q1h % 8 ||
      (D2 > 0 && (!q2 || !al(q2) || q2r % 8 || q2h % 8)) || our % 4 || ouh % 4 ||
      (uintptr_t)out % 8)
    return hipErrorInvalidValue;
  const int subs = (tile_rows + kRows - 1) / kRows;
  int bsh = 0;
  while ((1 << bsh) < bs) ++bsh;
#define GO(T)                                                                                    \
  {                                                                                              \
    const LatentTileArgs<T> a{(const T*)q1, q1r, q1h, D1, (const T*)(D2 > 0 ? q2 : q1),          \
                              D2 > 0 ? q2r : q1r, D2 > 0 ? q2h : q1h, (const T*)kc, krow,        \
                              (const T*)vt, (T*)out, our, ouh, tables, maxb, q_tiles, cu, start, \
                              n_tiles * subs, subs, tile_rows, H, bsh, scale, softcap, tcoef,    \
                              tevery, r1, r2, sink, (const T*)gate, gater};                      \
    return launch<T>(a, D1 + D2, st);                                                        \
  }
  if (dt == kBF16) GO(bf16)
  if (dt == kF16) GO(fp16)
  return hipErrorInvalidValue;
#undef GO
}

}  // extern "C"
