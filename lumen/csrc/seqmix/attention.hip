// Attention of the hybrid stack over a paged cache of un-normalised keys that double as values:
//   score(i, j) = scale * (q_i / rms(q_i)) . (k_j / rms(k_j)),   j <= i, same chunk as i
//   p_j = exp(s_j) / (sink + sum_j' exp(s_j')),   o_i = sum_j p_j k_j
// `chunk` > 0 restricts row i to keys with j / chunk == i / chunk (positions in the sequence);
// `sink` adds a key of score 0 that carries no value, i.e. the running softmax starts from
// (max 0, denominator 1) instead of (-inf, 0).
//
// Eight waves per (row, query head), for prefill chunks and decode rows alike (a row is a row: its
// position and its segment's block table say which keys it sees, so the result cannot depend on
// how the step was cut).  The waves take the 64-key tiles in turn; within a tile lane l scores key j0 + l -- the dot
// product and the key's sum of squares come from the same 16-byte loads -- then the wave takes
// the tile's max and sum (online softmax), and for the value pass lane l owns channels l, l + 64,
// ... of the output and walks the tile's keys (coalesced rows).  Scores, norms and the softmax
// are fp32.  The mask bounds a row's keys by `chunk`, so decode reads at most chunk keys and a
// split over the keys is not needed.
#include "mma.h"

using namespace lumen;

namespace {

constexpr int kMaxD = 256;

// waves per (row, head), each takes every kRowWaves-th 64-key tile: eight walk a context of 512 keys in one
// step each (8 rows x 16 heads: 20.2 us with four and un-unrolled loads, 17.7 with eight)
constexpr int kRowWaves = 8;

// 16-bit rows of LPT = D / 8 lanes, LPT a power of two: a key is loaded once, 16 bytes a lane, for its score, its
// square and its value.  (The form below reads a key row per lane for the scores -- 64 rows apart -- and all of them once
// more for the values: 8 rows x 16 heads, 512 keys, 17.9 us in a decode step, bound by those reads' latency; here 12.1.)
// kStep keys per lane group and step, the next step's in flight; every group keeps its own (max, sum, accumulator),
// which meet in the wave and then in LDS.  Rows past the last key repeat it and count for nothing.  (rsqrtf: 0.9 ulp at
// most where 1 / sqrtf has 1.5.  Results that are not float64's rounded: bf16 0.07 -> 0.02 %, fp16 0.57 -> 0.28.)
constexpr int kStep = 8;

template <int CTRL> __device__ __forceinline__ float row_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

template <typename T, int LPT>
__device__ __forceinline__ float key_dot(const uint4& a, const uint4& b) {
  float s = 0.f;
  if constexpr (__is_same(T, bf16)) {
    const unsigned x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
    typedef __bf16 two __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int j = 0; j < 4; ++j)
      s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(two, x[j]), __builtin_bit_cast(two, y[j]), s, false);
  } else {                                   // (mixed fmas: the dot instruction need not keep subnormals)
    const T *x = reinterpret_cast<const T*>(&a), *y = reinterpret_cast<const T*>(&b);
#pragma unroll
    for (int j = 0; j < 8; ++j) s = fmaf(to_f32(x[j]), to_f32(y[j]), s);
  }
  s += row_dpp<0xB1>(s);
  s += row_dpp<0x4E>(s);
  if (LPT > 4) s += row_dpp<0x141>(s);
  if (LPT > 8) s += row_dpp<0x140>(s);
  if (LPT > 16) s += __shfl_xor(s, 16, 64);
  return s;
}

template <typename T, int LPT>
__global__ void __launch_bounds__(64 * kRowWaves)
chunk_row_kernel(const T* __restrict__ q, long long ldq, const T* __restrict__ cache, T* __restrict__ out,
                 const int* __restrict__ tables, int maxb, const int* __restrict__ row_seg,
                 const int* __restrict__ positions, int H, int G, int bs, float scale, float eps, int chunk, int sink) {
  constexpr int D = 8 * LPT, KPW = 64 / LPT, KS = KPW * kRowWaves;      // keys a step of the workgroup per load
  const int t = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = hd / (H / G), grp = lane / LPT, part = lane % LPT;
  const int pos = positions[t], lo = chunk > 0 ? (pos / chunk) * chunk : 0;
  const int* tbl = tables + (long long)row_seg[t] * maxb;
  __shared__ float s_acc[kRowWaves][D], s_m[kRowWaves], s_l[kRowWaves];
  const int first = lo + w * KPW + grp;
  uint4 nxt[kStep];
  const auto load = [&](int j0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const unsigned j = (unsigned)min(j0 + u * KS, pos), b = j / (unsigned)bs;
      nxt[u] = *reinterpret_cast<const uint4*>(cache + (((long long)tbl[b] * bs + (j - b * bs)) * G + g) * D + 8 * part);
    }
  };
  load(first);
  const uint4 qv = *reinterpret_cast<const uint4*>(q + (long long)t * ldq + hd * D + 8 * part);
  const float qn = scale / sqrtf(key_dot<T, LPT>(qv, qv) / D + eps);
  const bool sinks = sink && w == 0 && grp == 0;          // the sink: a key of score 0 without a value
  float m = sinks ? 0.f : -INFINITY, l = sinks ? 1.f : 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int j0 = first; __any(j0 <= pos); j0 += kStep * KS) {
    uint4 k[kStep];
    float p[kStep], mx = m;
#pragma unroll
    for (int u = 0; u < kStep; ++u) k[u] = nxt[u];
    if (__any(j0 + kStep * KS <= pos)) load(j0 + kStep * KS);
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const float s = key_dot<T, LPT>(k[u], qv) * qn * rsqrtf(key_dot<T, LPT>(k[u], k[u]) * (1.f / D) + eps);
      p[u] = j0 + u * KS <= pos ? s : -INFINITY;
      mx = fmaxf(mx, p[u]);
    }
    const float mb = mx == -INFINITY ? 0.f : mx, al = expf(m - mb);
    m = mx;
    l *= al;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= al;
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      p[u] = expf(p[u] - mb);
      l += p[u];
      const T* v = reinterpret_cast<const T*>(&k[u]);
      if (j0 + u * KS <= pos) {
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(p[u], to_f32(v[e]), acc[e]);
      }
    }
  }
#pragma unroll
  for (int o = LPT; o < 64; o <<= 1) {
    const float m2 = __shfl_xor(m, o, 64), l2 = __shfl_xor(l, o, 64), M = fmaxf(m, m2);
    const float a1 = m == -INFINITY ? 0.f : expf(m - M), a2 = m2 == -INFINITY ? 0.f : expf(m2 - M);
    l = l * a1 + l2 * a2;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = acc[e] * a1 + __shfl_xor(acc[e], o, 64) * a2;
    m = M;
  }
  if (lane < LPT) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s_acc[w][8 * part + e] = acc[e];
    if (lane == 0) { s_m[w] = m; s_l[w] = l; }
  }
  __syncthreads();
  if ((int)threadIdx.x < D) {
    float mt = -INFINITY, lt = 0.f, o = 0.f;
#pragma unroll
    for (int x = 0; x < kRowWaves; ++x) mt = fmaxf(mt, s_m[x]);
#pragma unroll
    for (int x = 0; x < kRowWaves; ++x) {
      const float f = s_m[x] == -INFINITY ? 0.f : expf(s_m[x] - mt);
      lt += s_l[x] * f;
      o += s_acc[x][threadIdx.x] * f;
    }
    out[((long long)t * H + hd) * D + threadIdx.x] = from_f32<T>(o / lt);
  }
}

template <typename T>
__global__ void __launch_bounds__(64 * kRowWaves)
chunk_attn_kernel(const T* __restrict__ q, long long ldq, const T* __restrict__ cache,
                  T* __restrict__ out, const int* __restrict__ tables, int maxb,
                  const int* __restrict__ row_seg, const int* __restrict__ positions, int H, int G,
                  int D, int bs, float scale, float eps, int chunk, int sink) {
  const int t = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = hd / (H / G);
  const int pos = positions[t];
  const int* tbl = tables + (long long)row_seg[t] * maxb;
  const int lo = chunk > 0 ? (pos / chunk) * chunk : 0;
  __shared__ float s_q[kMaxD];
  __shared__ float s_p[kRowWaves][64];
  __shared__ long long s_row[kRowWaves][64];
  __shared__ float s_acc[kRowWaves][kMaxD];
  __shared__ float s_m[kRowWaves], s_l[kRowWaves];

  float ss = 0.f;
  for (int d = lane; d < D; d += 64) {
    const float v = to_f32(q[(long long)t * ldq + hd * D + d]);
    if (w == 0) s_q[d] = v;
    ss += v * v;
  }
  ss = wave_sum(ss);
  const float qn = scale / sqrtf(ss / D + eps);
  __syncthreads();

  // every wave keeps its own running (max, sum, accumulator) over its tiles; wave 0 starts from
  // the sink, the others from nothing, and the partial results are merged at the end
  float m = (sink && w == 0) ? 0.f : -INFINITY, l = (sink && w == 0) ? 1.f : 0.f;
  float acc[kMaxD / 64] = {0.f, 0.f, 0.f, 0.f};
  float acc8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const bool vec = (D % 8) == 0;
  const int lpk = vec ? D / 8 : 64, kpi = 64 / lpk;   // lanes per key row, keys per step
  const int grp = lane / lpk, part = lane % lpk;
  for (int j0 = lo + 64 * w; j0 <= pos; j0 += 64 * kRowWaves) {
    const int j = j0 + lane;
    const bool valid = j <= pos;
    float s = -INFINITY;
    long long rowoff = 0;
    if (valid) {
      rowoff = (((long long)tbl[j / bs] * bs + j % bs) * G + g) * D;
      const T* kp = cache + rowoff;
      float dot = 0.f, k2 = 0.f;
      if (vec) {
#pragma unroll 8
        for (int d = 0; d < D; d += 8) {
          float kv[8];
          load8<T>(kp + d, kv);
#pragma unroll
          for (int e = 0; e < 8; ++e) { dot += s_q[d + e] * kv[e]; k2 += kv[e] * kv[e]; }
        }
      } else {
        for (int d = 0; d < D; ++d) {
          const float kv = to_f32(kp[d]);
          dot += s_q[d] * kv;
          k2 += kv * kv;
        }
      }
      s = dot * qn / sqrtf(k2 / D + eps);
    }
    const float mn = fmaxf(m, wave_max(s));       // finite: the tile's first key is valid
    const float p = valid ? expf(s - mn) : 0.f;
    const float corr = expf(m - mn);
    l = l * corr + wave_sum(p);
    m = mn;
    s_p[w][lane] = p;
    s_row[w][lane] = rowoff;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    const int nk = min(64, pos - j0 + 1);
    if (vec) {
      // value pass, 16 bytes per lane: lpk = D / 8 lanes cover one key row, 64 / lpk keys per
      // step; a lane accumulates its 8 channels over the keys of its group, the groups are
      // summed once at the end
#pragma unroll
      for (int e = 0; e < 8; ++e) acc8[e] *= corr;
      if (grp < kpi) {
#pragma unroll 4
        for (int jj = grp; jj < nk; jj += kpi) {
          const float pj = s_p[w][jj];
          float kv[8];
          load8<T>(cache + s_row[w][jj] + 8 * part, kv);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc8[e] += pj * kv[e];
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < kMaxD / 64; ++c) acc[c] *= corr;
      for (int jj = 0; jj < nk; ++jj) {
        const float pj = s_p[w][jj];
        const T* kp = cache + s_row[w][jj];
#pragma unroll
        for (int c = 0; c < kMaxD / 64; ++c) {
          const int d = lane + 64 * c;
          if (d < D) acc[c] += pj * to_f32(kp[d]);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  if (vec) {
    // sum the key groups of this wave: every group adds its channels into s_acc[w] in turn
    for (int d = lane; d < D; d += 64) s_acc[w][d] = 0.f;
    for (int gq = 0; gq < kpi; ++gq) {
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      if (grp == gq) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s_acc[w][8 * part + e] += acc8[e];
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < kMaxD / 64; ++c) {
      const int d = lane + 64 * c;
      if (d < D) s_acc[w][d] = acc[c];
    }
  }
  if (lane == 0) { s_m[w] = m; s_l[w] = l; }
  __syncthreads();
  if ((int)threadIdx.x < D) {          // (D <= 256 < the workgroup's threads)
    float mt = -INFINITY;
#pragma unroll
    for (int x = 0; x < kRowWaves; ++x) mt = fmaxf(mt, s_m[x]);
    float lt = 0.f, f[kRowWaves];
#pragma unroll
    for (int x = 0; x < kRowWaves; ++x) {
      f[x] = s_m[x] == -INFINITY ? 0.f : expf(s_m[x] - mt);
      lt += s_l[x] * f[x];
    }
    const float inv = 1.f / lt;
    const int d = threadIdx.x;
    float o = 0.f;
#pragma unroll
    for (int x = 0; x < kRowWaves; ++x) o += s_acc[x][d] * f[x];
    out[((long long)t * H + hd) * D + d] = from_f32<T>(o * inv);
  }
}

// ---- prefill tiles on the matrix cores (16-bit dtypes, D a multiple of 32) ---------------------
// A workgroup of NW waves takes 32 * NW consecutive rows of ONE segment and one query head; the
// keys the tile can see (from the first row's chunk start to the last row's position) are visited KT = 64
// at a time (32 for heads over 128), staged in LDS twice (row-major for the scores, transposed for the value
// pass) and shared by the waves.  Bound by the chain of tiles at two waves per SIMD; the loads of a tile leave
// together one tile ahead and two buffers leave one barrier per tile, as in window_attention.hip.  Heads over 128 have
// no registers left: one buffer, value addresses formed where they are used and queries read again by the look at the
// end keep the spills out of the loop (us, two buffers -> one, 8 heads of 256 / 192: 8 x 512 rows 93 -> 84 / 54 -> 49, chunks of
// 128 39 -> 36 / 24 -> 21, 1 x 200 42 -> 41 / 27 -> 24).  us, tiles of 32 keys, one buffer -> now (bf16, heads of 128): 8 x 512
// rows x 16 heads 82 -> 43, 1 x 200 29 -> 21, 32 x 50 16 -> 12, 1 x 1024 x 32 109 -> 64; heads of 64 47 -> 31, 96 50 -> 38, 192 54
// -> 49, 256 93 -> 84.  A portion of few keys pays for a whole tile of 64 (1 x 2 8.0 -> 8.9; 64 x 5 rows x 32 heads 22 -> 29;
// a second form of the tile for 32 keys 29, and 8 x 512 46).
// Per wave (32 queries) and 32 keys, with v_mfma_f32_32x32x16:
//   S^T = K Q^T      keys on the accumulator rows, queries on the columns (lane & 31): a lane
//                    owns ONE query, so its running max / sum / correction are plain scalars;
//                    q and k enter un-normalised (exactly as projected) and the two RMS factors
//                    multiply the fp32 score (k's sum of squares comes from the operand the lane
//                    loads anyway);
//   O^T += V^T P^T   the accumulator registers 8s .. 8s+7 of S^T are keys {16s + 4hi + 0..3,
//                    16s + 8 + 4hi + 0..3}: exactly one k = 16 operand when the transposed key
//                    image is read in that order, so P goes from registers to the next product
//                    without touching LDS.  P is split into a 16-bit head and a 16-bit remainder
//                    (two products), which keeps ~16 mantissa bits of the fp32 weights.
// Accumulator layout of the 32x32 products: lane l, register 4j + i = row 8j + 4(l >> 5) + i,
// column l & 31; operand lanes hold k = 8(l >> 5) + 0..7.
template <typename T>
__device__ __forceinline__ float sumsq8(uint4 v) {
  const unsigned w[4] = {v.x, v.y, v.z, v.w};
  float s = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    float a, b;
    unpack2<T>(w[x], a, b);
    s += a * a + b * b;
  }
  return s;
}

// KS 2 (few workgroups, see kSplit): 64 rows, a row's keys shared by two waves, each one half of every tile; the upper half's maximum, sum and
// accumulators meet the lower one's in LDS at the end.
// (register budget: left to itself the compiler takes > 300 registers and runs one wave per SIMD.  Two waves
// for heads of 96 and 128, where three spill; of 256 two with spills are ahead of one without)
template <typename T, int D, int NW, int KT, int KS = 1>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(D <= 64 ? 3 : 2)))
tile_attn_kernel(const T* __restrict__ q, long long ldq, const T* __restrict__ cache,
                 T* __restrict__ out, const int* __restrict__ tables, int maxb,
                 const int* __restrict__ tiles, const int* __restrict__ cu,
                 const int* __restrict__ start, int H, int G, int bs, float scale, float eps,
                 int chunk, int sink) {
  constexpr int QT = 32 * NW / KS, LK = D + 8, LT = KT + 8, NV = D / 8, SB = KT / 32, WB = SB / KS;
  static_assert(SB % KS == 0 && NW % KS == 0, "a wave's keys of a tile");
  // two buffers: a tile is stored while the one before it is read, one barrier per tile
  constexpr int NB = D <= 128 ? 2 : 1;
  __shared__ __align__(16) T s_all[NB * (KT * LK + D * LT)];
  T (*const s_kb)[KT * LK] = reinterpret_cast<T (*)[KT * LK]>(s_all);                    // key tile, row-major
  T (*const s_tb)[D * LT] = reinterpret_cast<T (*)[D * LT]>(s_all + NB * KT * LK);       // key tile, transposed [d][key]
  static_assert(KS == 1 || NW / 2 * (D / 2 + 2) * 64 * 4 <= (int)sizeof(s_all), "the other halves' results");
  __shared__ float s_nb[NB][KT];                  // 1 / rms of the tile's keys (power-of-two D / 8)
  constexpr int kTbl = 512;                   // block-table entries of the visible keys, in LDS
  __shared__ int s_tbl[kTbl];
  constexpr bool kStagedNorm = (NV & (NV - 1)) == 0 && NV <= 64;
  const int tid = threadIdx.x, lane = tid & 63, w = (tid >> 6) % (NW / KS), c = lane & 31, hi = lane >> 5;
  const int kb = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((tid >> 6) / (NW / KS)) * WB;    // first block of 32 keys of a tile that the wave takes
  int tix, hd;
  heavy_first(blockIdx.x, gridDim.x, H, tix, hd);
  const int g = hd / (H / G);
  const int sg = tiles[2 * (tix / KS)], row0 = tiles[2 * (tix / KS) + 1] + tix % KS * QT;
  if (KS > 1 && row0 >= cu[sg + 1]) return;              // (the whole workgroup: a tile of the list with few rows)
  const int seg_r0 = cu[sg], p0 = start[sg];
  const int nrows = min(QT, cu[sg + 1] - row0);
  const int* tbl = tables + (long long)sg * maxb;

  const bool qv = 32 * w + c < nrows;
  const int qrow = row0 + 32 * w + c;
  const int pos = qv ? p0 + (qrow - seg_r0) : -1;
  const int lo = (chunk > 0 && qv) ? (pos / chunk) * chunk : 0;
  uint4 qreg[D / 16];
  float q2 = 0.f;
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk) {
    qreg[kk] = qv ? *reinterpret_cast<const uint4*>(q + (long long)qrow * ldq + hd * D + 16 * kk + 8 * hi)
                  : make_uint4(0, 0, 0, 0);
    q2 += sumsq8<T>(qreg[kk]);
  }
  q2 += __shfl_xor(q2, 32, 64);
  const float qn = scale / sqrtf(q2 / D + eps);

  const int pos_first = p0 + (row0 - seg_r0), kend = pos_first + nrows - 1;
  const int kbeg = chunk > 0 ? (pos_first / chunk) * chunk : 0;
  const bool wave_on = 32 * w < nrows;
  const int wpos_min = pos_first + 32 * w, wpos_max = min(kend, wpos_min + 31);
  const int wlo_min = chunk > 0 ? (wpos_min / chunk) * chunk : 0;

  // the block ids of the keys this tile can see, so that a key's address never waits for a table load
  // (a range of more than kTbl blocks, i.e. a very long chunk, is read from the table)
  const int b_first = kbeg / bs, b_count = kend / bs - b_first + 1;
  const bool in_lds = b_count <= kTbl;
  if (in_lds)
    for (int i = tid; i < b_count; i += 64 * NW) s_tbl[i] = tbl[b_first + i];
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  __syncthreads();

  float m = sink && kb == 0 ? 0.f : -INFINITY, l = sink && kb == 0 && hi == 0 ? 1.f : 0.f;   // (l: the lane's half)
  f32x16 O[D / 32];
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) O[db][r] = 0.f;

  // staging: one item = 4 consecutive keys x 8 channels (four 16-byte loads); the row-major
  // image takes them as they are, the transposed image takes eight 8-byte stores of 4 keys each
  // (transposed in registers).  The next tile's loads are issued before this tile's products, so
  // their latency hides behind the matrix work.
  constexpr int NT = 64 * NW, NTOT = D * SB, ITEMS = (NTOT + NT - 1) / NT;
  uint4 pre[ITEMS][4];
  auto prefetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int item = tid + it * NT;
      if (NTOT % NT == 0 || item < NTOT) {
        const int kq = item / NV, part = item % NV, j = k0 + 4 * kq;
        // the four cache rows first and without a branch per key (past the last key: that one again;
        // `commit` blanks it): then the four loads leave together
        int jb[4], blk[4];
        if (bshift >= 0) {
#pragma unroll
          for (int x = 0; x < 4; ++x) jb[x] = min(j + x, kend) >> bshift;
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x) jb[x] = min(j + x, kend) / bs;
        }
        if (in_lds) {
#pragma unroll
          for (int x = 0; x < 4; ++x) blk[x] = s_tbl[jb[x] - b_first];
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x) blk[x] = tbl[jb[x]];
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const long long row = (long long)blk[x] * bs + (min(j + x, kend) - jb[x] * bs);
          pre[it][x] = *reinterpret_cast<const uint4*>(cache + (row * G + g) * D + 8 * part);
        }
      }
    }
  };
  auto commit = [&](int k0, T* s_k, T* s_t, float* s_kn) __attribute__((always_inline)) {
    const bool tail = k0 + KT - 1 > kend;            // keys past the last one: zeros
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int item = tid + it * NT;
      if (NTOT % NT == 0 || item < NTOT) {
        const int kq = item / NV, part = item % NV;
        if (tail) {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            if (k0 + 4 * kq + x > kend) pre[it][x] = make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int x = 0; x < 4; ++x)
          *reinterpret_cast<uint4*>(&s_k[(4 * kq + x) * LK + 8 * part]) = pre[it][x];
        if (kStagedNorm) {   // the NV lanes of a key quad are adjacent: sum their partial squares
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            float k2 = sumsq8<T>(pre[it][x]);
#pragma unroll
            for (int o = 1; o < NV; o <<= 1) k2 += __shfl_xor(k2, o, 64);
            if (part == 0) s_kn[4 * kq + x] = 1.f / sqrtf(k2 / D + eps);
          }
        }
        const unsigned w0[4] = {pre[it][0].x, pre[it][0].y, pre[it][0].z, pre[it][0].w};
        const unsigned w1[4] = {pre[it][1].x, pre[it][1].y, pre[it][1].z, pre[it][1].w};
        const unsigned w2[4] = {pre[it][2].x, pre[it][2].y, pre[it][2].z, pre[it][2].w};
        const unsigned w3[4] = {pre[it][3].x, pre[it][3].y, pre[it][3].z, pre[it][3].w};
#pragma unroll
        for (int mm = 0; mm < 4; ++mm) {     // word mm holds channels 2mm (low half), 2mm + 1
          // the key quads of a row are permuted by the row's group of 8 (all rows a lane
          // writes share it): lanes that differ in `part` land in different banks
          T* t0 = &s_t[(8 * part + 2 * mm) * LT + 4 * (kq ^ (part & 7))];
          *reinterpret_cast<uint2*>(t0) = make_uint2((w0[mm] & 0xffffu) | (w1[mm] << 16),
                                                     (w2[mm] & 0xffffu) | (w3[mm] << 16));
          *reinterpret_cast<uint2*>(t0 + LT) = make_uint2(
              (w0[mm] >> 16) | (w1[mm] & 0xffff0000u), (w2[mm] >> 16) | (w3[mm] & 0xffff0000u));
        }
      }
    }
  };

  const int t0 = c * LT + 4 * (hi ^ (c >> 3)) + 32 * kb, t1 = c * LT + 4 * ((2 + hi) ^ (c >> 3)) + 32 * kb;
  // the wave's share of tile k0
  auto tile = [&](int kt, const T* s_k, const T* s_t, const float* s_kn) __attribute__((always_inline)) {
    const int k0 = kt + 32 * kb;             // first of the wave's keys
    if (!wave_on || k0 > wpos_max || k0 + 32 * WB - 1 < wlo_min) return;   // nothing this wave may see

    f32x16 sc[WB];
    float k2[WB], kn[WB];
#pragma unroll
    for (int b = 0; b < WB; ++b) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[b][r] = 0.f;
      k2[b] = kn[b] = 0.f;
    }
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int b = 0; b < WB; ++b) {
        const uint4 a = *reinterpret_cast<const uint4*>(&s_k[(32 * (kb + b) + c) * LK + 16 * kk + 8 * hi]);
        if (!kStagedNorm) k2[b] += sumsq8<T>(a);
        sc[b] = Mma32<T>::run(a, qreg[kk], sc[b]);
      }
    if (!kStagedNorm) {                                  // of key k0 + 32 b + c (other head sizes)
#pragma unroll
      for (int b = 0; b < WB; ++b) {
        k2[b] += __shfl_xor(k2[b], 32, 64);
        kn[b] = 1.f / sqrtf(k2[b] / D + eps);
      }
    }
    // register r of sc[b] is key k0 + key_of(b, r)
    const auto key_of = [&](int b, int r) { return 32 * b + 8 * (r >> 2) + 4 * hi + (r & 3); };
    // a tile every query of the wave sees whole needs no mask
    const bool whole = k0 >= (chunk > 0 ? (wpos_max / chunk) * chunk : 0) && k0 + 32 * WB - 1 <= wpos_min &&
                       32 * w + 31 < nrows;
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float knr = kStagedNorm ? s_kn[32 * kb + key_of(b, r)] : __shfl(kn[b], key_of(0, r), 64);
        sc[b][r] *= qn * knr;
      }
    if (!whole) {
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = k0 + key_of(b, r);
          sc[b][r] = (j >= lo && j <= pos) ? sc[b][r] : -INFINITY;
        }
    }
    float mloc = -INFINITY;
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) mloc = fmaxf(mloc, sc[b][r]);
    mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));
    // the reference of the weights follows the running maximum only when that passes it by kRise: weights
    // stay under e^kRise, and the accumulators are rescaled on a few tiles of a row, not on most
    if (__any(mloc > m + kRise)) {
      const float mn = mloc > m + kRise ? mloc : m;
      const float corr = mn == m ? 1.f : __expf(m - mn);
      l *= corr;
      m = mn;
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) O[db][r] *= corr;
    }
    const float ms = m == -INFINITY ? 0.f : m;
    // (v_exp_f32: this kernel serves 16-bit dtypes only, the weights are rounded to ~16 bits)
    float psum = 0.f;
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) { sc[b][r] = __expf(sc[b][r] - ms); psum += sc[b][r]; }
    l += psum;                                 // (the lane's half: the other lane's is added at the end)
#pragma unroll
    for (int s2 = 0; s2 < 2 * WB; ++s2) {
      unsigned ph[4], pl[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float a0 = sc[s2 / 2][8 * (s2 & 1) + 2 * x], a1 = sc[s2 / 2][8 * (s2 & 1) + 2 * x + 1];
        ph[x] = pk2<T>(a0, a1);                      // one packed conversion
        float h0, h1;
        unpack2<T>(ph[x], h0, h1);
        pl[x] = pk2<T>(a0 - h0, a1 - h1);
      }
      const uint4 bh = make_uint4(ph[0], ph[1], ph[2], ph[3]);
      const uint4 bl = make_uint4(pl[0], pl[1], pl[2], pl[3]);
#pragma unroll
      for (int db = 0; db < D / 32; ++db) {
        // quads 4 s2 + hi and 4 s2 + 2 + hi of row 32 db + c, under the store's permutation: both low bits lie in t0 /
        // t1, the others in the instruction's offset (heads over 128: formed here, those take no registers)
        const int sw = ((32 * db + c) >> 3) & 7, at = 32 * db * LT + 32 * (s2 >> 1) + 16 * ((s2 & 1) ^ (db & 1));
        const T* row = s_t + (32 * db + c) * LT;
        const uint2 a0 = *reinterpret_cast<const uint2*>(D <= 128 ? s_t + t0 + at : row + 4 * ((4 * s2 + hi) ^ sw));
        const uint2 a1 = *reinterpret_cast<const uint2*>(D <= 128 ? s_t + t1 + at : row + 4 * ((4 * s2 + 2 + hi) ^ sw));
        const uint4 a = make_uint4(a0.x, a0.y, a1.x, a1.y);
        O[db] = Mma32<T>::run(a, bh, O[db]);
        O[db] = Mma32<T>::run(a, bl, O[db]);
      }
    }
  };

  prefetch(kbeg);
  if constexpr (NB == 1) {
    for (int k0 = kbeg; k0 <= kend; k0 += KT) {
      __syncthreads();                       // the tile before has been read
      commit(k0, s_kb[0], s_tb[0], s_nb[0]);
      __syncthreads();
      if (k0 + KT <= kend) prefetch(k0 + KT);
      tile(k0, s_kb[0], s_tb[0], s_nb[0]);
    }
  } else {
    commit(kbeg, s_kb[0], s_tb[0], s_nb[0]);
    __builtin_amdgcn_s_waitcnt(0xF70);     // vmcnt(0): or the loop's first product would wait, every time, for
    __syncthreads();                       // the queries, and with them for the tile just asked for
    for (int k0 = kbeg, cur = 0; k0 <= kend; k0 += KT, cur ^= 1) {
      const bool more = k0 + KT <= kend;
      if (more) prefetch(k0 + KT);
      tile(k0, s_kb[cur], s_tb[cur], s_nb[cur]);
      if (more) commit(k0 + KT, s_kb[cur ^ 1], s_tb[cur ^ 1], s_nb[cur ^ 1]);
      __syncthreads();
    }
  }
  if constexpr (KS == 2) {                   // the upper keys' waves hand their sums to the lower ones'
    float* box = reinterpret_cast<float*>(s_all) + w * (D / 2 + 2) * 64 + lane;
    if (kb > 0) {
#pragma unroll
      for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) box[(16 * db + r) * 64] = O[db][r];
      box[D / 2 * 64] = m;
      box[(D / 2 + 1) * 64] = l;
    }
    __syncthreads();
    if (kb > 0) return;
    const float m2 = box[D / 2 * 64], mn = fmaxf(m, m2);
    const float c1 = m == mn ? 1.f : __expf(m - mn), c2 = m2 == mn ? 1.f : __expf(m2 - mn);
    l = l * c1 + box[(D / 2 + 1) * 64] * c2;
    m = mn;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[db][r] = O[db][r] * c1 + box[(16 * db + r) * 64] * c2;
  }
  l += __shfl_xor(l, 32, 64);
  // A hidden key has weight 0, but 0 times an infinite or NaN value is NaN: channels that are not finite are formed
  // again, key by key over what the row sees (m and l stand).
  float odd[4] = {0.f, 0.f, 0.f, 0.f};             // (0 times a finite number stays 0)
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) odd[r & 3] = fmaf(O[db][r], 0.f, odd[r & 3]);
  const long long qat = (long long)(qv ? qrow : row0) * ldq + hd * D;      // (heads over 128: q is read again)
  if (__builtin_expect(__any(odd[0] + odd[1] + odd[2] + odd[3] != 0.f && qv), 0)) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      f32x16 o;
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = 0.f;
      for (int j = wlo_min; j <= wpos_max; ++j) {
        const int jb = j / bs;
        const T* kp = cache + (((long long)tbl[jb] * bs + (j - jb * bs)) * G + g) * D;
        float s = 0.f, k2 = 0.f;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
          __builtin_amdgcn_sched_barrier(0);       // (one load at a time: registers)
          float x[8];
          load8<T>(kp + 16 * kk + 8 * hi, x);
          uint4 qk = D <= 128 ? qreg[kk] : *reinterpret_cast<const uint4*>(q + qat + 16 * kk + 8 * hi);
          asm volatile("" : "+v"(qk.x), "+v"(qk.y), "+v"(qk.z), "+v"(qk.w));   // (converted here, not ahead of the loop)
          const T* y = reinterpret_cast<const T*>(&qk);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            s = fmaf(x[e], to_f32(y[e]), s);
            k2 = fmaf(x[e], x[e], k2);
          }
        }
        s += __shfl_xor(s, 32, 64);
        k2 += __shfl_xor(k2, 32, 64);
        const float p = __expf(s * qn / sqrtf(k2 / D + eps) - m);
        if (j > pos || j < lo) continue;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          float v[4];
          load4<T>(kp + 32 * db + 8 * q4 + 4 * hi, v);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[4 * q4 + e] = fmaf(p, v[e], o[4 * q4 + e]);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) O[db][r] = fabsf(O[db][r]) < INFINITY ? O[db][r] : o[r];
    }
  }
  if (qv) {
    const float inv = 1.f / l;
    T* op = out + ((long long)qrow * H + hd) * D;
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 32 * db + 8 * j + 4 * hi;
        const unsigned x0 = pk2<T>(O[db][4 * j] * inv, O[db][4 * j + 1] * inv);
        const unsigned x1 = pk2<T>(O[db][4 * j + 2] * inv, O[db][4 * j + 3] * inv);
        *reinterpret_cast<uint2*>(op + d) = make_uint2(x0, x1);
      }
  }
}

// Tiles of 128 rows by heads up to which tiles of 64 rows with the keys in halves are faster: the exponentials and conversions of a wave's
// scores bound the chain of key tiles, and few workgroups leave half of the vector units idle.  us, whole -> in halves, 16 heads of 128:
// 1 x 512 tokens 33.8 -> 27.4 (chunks of 256 20.7 -> 17.1), 1 x 1024 59.8 -> 48.0, 4 x 512 34.3 -> 29.9; 5 x 512 37.0 -> 40.0; heads of 64, 1 x
// 512 26.0 -> 21.9.
constexpr int kSplit = 256;

template <typename T>
hipError_t launch_tiles(const void* q, long long ldq, const void* cache, void* out,
                        const int* tables, int maxb, const int* tiles, int ntiles, const int* cu,
                        const int* start, int H, int G, int D, int bs, float scale, float eps,
                        int chunk, int sink, int tile_rows, hipStream_t st) {
  const dim3 grid((unsigned)((long long)ntiles * H));
#define GO(DD)                                                                                   \
  {                                                                                              \
    constexpr int KT = DD <= 128 ? 64 : 32;                                                      \
    if constexpr (KT == 64) {                                                                    \
      if (tile_rows == 128 && (long long)ntiles * H <= kSplit) {                                   \
        tile_attn_kernel<T, DD, 4, KT, 2><<<2 * grid.x, 256, 0, st>>>((const T*)q, ldq, (const T*)cache, (T*)out, \
                                                       tables, maxb, tiles, cu, start, H, G, bs, \
                                                       scale, eps, chunk, sink);                 \
        return hipGetLastError();                                                                \
      }                                                                                          \
    }                                                                                            \
    if (tile_rows == 128)                                                                        \
      tile_attn_kernel<T, DD, 4, KT><<<grid, 256, 0, st>>>((const T*)q, ldq, (const T*)cache, (T*)out, \
                                                       tables, maxb, tiles, cu, start, H, G, bs, \
                                                       scale, eps, chunk, sink);                 \
    else                                                                                         \
      tile_attn_kernel<T, DD, 2, KT><<<grid, 128, 0, st>>>((const T*)q, ldq, (const T*)cache, (T*)out, \
                                                       tables, maxb, tiles, cu, start, H, G, bs, \
                                                       scale, eps, chunk, sink);                 \
  }
  switch (D) {
    case 32: GO(32); break;
    case 64: GO(64); break;
    case 96: GO(96); break;
    case 128: GO(128); break;
    case 192: GO(192); break;
    case 256: GO(256); break;
    default: return hipErrorInvalidValue;
  }
#undef GO
  return hipGetLastError();
}

}  // namespace

extern "C" {

// 1 when sm_chunk_attn_tiles has a kernel for this dtype / head size
int sm_chunk_attn_tiles_ok(int dt, int D) {
  return (dt == kBF16 || dt == kF16) &&
         (D == 32 || D == 64 || D == 96 || D == 128 || D == 192 || D == 256);
}

// tiles: [ntiles, 2] int32 (segment, first row); every tile covers up to tile_rows (64 or 128)
// rows of its segment
hipError_t sm_chunk_attn_tiles(int dt, const void* q, long long ldq, const void* cache, void* out,
                               const int* tables, int maxb, const int* tiles, int ntiles,
                               const int* cu, const int* start, int H, int G, int D, int bs,
                               float scale, float eps, int chunk, int sink, int tile_rows,
                               hipStream_t st) {
  if (ntiles == 0) return hipSuccess;
  if (G < 1 || H % G || bs < 1 || chunk < 0 || (ldq % 8) != 0) return hipErrorInvalidValue;
  if (tile_rows != 64 && tile_rows != 128) return hipErrorInvalidValue;
  if (dt == kBF16)
    return launch_tiles<bf16>(q, ldq, cache, out, tables, maxb, tiles, ntiles, cu, start, H, G, D,
                              bs, scale, eps, chunk, sink, tile_rows, st);
  if (dt == kF16)
    return launch_tiles<fp16>(q, ldq, cache, out, tables, maxb, tiles, ntiles, cu, start, H, G, D,
                              bs, scale, eps, chunk, sink, tile_rows, st);
  return hipErrorInvalidValue;
}

hipError_t sm_chunk_attn(int dt, const void* q, long long ldq, const void* cache, void* out,
                         const int* tables, int maxb, const int* row_seg, const int* positions,
                         int T, int H, int G, int D, int bs, float scale, float eps, int chunk,
                         int sink, hipStream_t st) {
  if (T == 0) return hipSuccess;
  if (D < 1 || D > kMaxD || G < 1 || H % G || bs < 1 || chunk < 0) return hipErrorInvalidValue;
  const dim3 grid(T, H);
  if ((dt == kBF16 || dt == kF16) && (D == 32 || D == 64 || D == 128 || D == 256) && ldq % 8 == 0 &&
      ((uintptr_t)q | (uintptr_t)cache) % 16 == 0) {
#define ROW(TT, LPT)                                                                                                \
  chunk_row_kernel<TT, LPT><<<grid, 64 * kRowWaves, 0, st>>>((const TT*)q, ldq, (const TT*)cache, (TT*)out, tables, \
                                                             maxb, row_seg, positions, H, G, bs, scale, eps, chunk, sink)
#define ROWS(TT)                 \
  if (D == 32) ROW(TT, 4);       \
  else if (D == 64) ROW(TT, 8);  \
  else if (D == 128) ROW(TT, 16); \
  else ROW(TT, 32)
    if (dt == kBF16) { ROWS(bf16); } else { ROWS(fp16); }
#undef ROWS
#undef ROW
    return hipGetLastError();
  }
#define CALL(TT) chunk_attn_kernel<TT><<<grid, 64 * kRowWaves, 0, st>>>((const TT*)q, ldq, (const TT*)cache, (TT*)out, tables, maxb, row_seg, positions, H, G, D, bs, scale, eps, chunk, sink)
  SM_DISPATCH(dt, CALL)
#undef CALL
  return hipGetLastError();
}

}  // extern "C"
