// Prefill attention over paged key and value caches on the matrix cores, with a soft cap, a
// linear distance bias, a sliding window that also keeps the sequence's first keys, and a
// per-head output gate -- every one optional:
//   s(i, j) = cap * tanh(q_i . k_j * scale / cap) - slope_h * (i - j)
//   row i sees key j when j <= i and (window == 0 or i - j < window or j < keep)
//   o_i = sigmoid(gate[i, h]) * sum_j softmax_j(s(i, j)) v_j
// or, with a per-head bias `sigb`, weights that are sigmoids and are not normalised:
//   o_i = sum_j sigmoid(s(i, j) + sigb_h) v_j
// q arrives as the projection left it (already normed where the design norms it), the key cache
// [blocks][bs][G][D] holds what the scores read and the value cache [blocks][bs][G / vdiv][DV]
// what is summed: the value size may differ from the key size, and `vdiv` consecutive key heads
// may share one value head (several score maps over the same values).
//
// A workgroup of NW waves takes 32 * NW consecutive rows of ONE segment and one query head.  The
// keys the tile can see are visited KT = 64 at a time (32 for values over 128 wide): first the tiles of the
// kept keys that lie below the window of the tile's first row, then the tiles from that window's start to the
// last row's position; what lies between is never loaded, so a long prompt's portion costs rows x (window +
// keep) and not rows x position.  A key tile is staged in LDS from the key cache (row-major, the
// score operand) and from the value cache (transposed, the value operand) and shared by the waves.
//
// What bounds it: the chain of one tile after the other at one or two waves per SIMD, ~9000 cycles per 64 keys
// where the products take 1500.  So the loads of a tile leave together one tile ahead (block ids from LDS, no
// branch between two loads: a table lookup that could also go to memory made each wait for the one
// before), two LDS buffers leave one barrier per tile, 64 keys share its exchanges, and the accumulators follow
// the maximum only when it rises by kRise.  Measured (us, tiles of 32 keys, one buffer -> now; bf16, heads of
// 128, soft cap): 1 x 512 rows x 32 heads 55 -> 33, 8 x 512 x 16 91 -> 43, 14 of 63 - 509 x 16 110 -> 58, 1 x 4096 x 32
// (window 1024) 380 -> 168; heads of 64 44 -> 23, of 256 191 -> 113, values of 256 169 -> 101; the look for infinite
// results at the end, which later came to it, 0.1 - 1.3 us (8 x 512 x 16 39.0 -> 39.7, 1 x 64 9.2 -> 9.5; with a comparison
// per result 0.3 - 1.9).  A portion of few keys pays for a whole tile of 64 (1 x 16 7.4 -> 9.0, 64 x 5 x 32 heads 22 -> 31).
//
// The exponentials and conversions of a wave's scores bound that chain, so few workgroups (kSplit below) leave half of the chip's vector
// units idle: there a workgroup takes 64 rows and KS = 2 waves share a row's keys, each one half of every tile; the upper half's
// maximum, sum and accumulators meet the lower one's in LDS at the end.
//
// Per wave (32 queries) and 32 keys, with v_mfma_f32_32x32x16:
//   S^T = K Q^T      keys on the accumulator rows, queries on the columns (lane & 31): a lane
//                    owns ONE query, so its running max / sum / correction are plain scalars;
//   O^T += V^T P^T   the accumulator registers 8s .. 8s+7 of S^T are keys {16s + 4hi + 0..3,
//                    16s + 8 + 4hi + 0..3}: exactly one k = 16 operand when the transposed value
//                    image is read in that order, so P goes from registers to the next product
//                    without touching LDS.  P is split into a 16-bit head and a 16-bit remainder
//                    (two products), which keeps ~16 mantissa bits of the fp32 weights.
// Accumulator layout of the 32x32 products: lane l, register 4j + i = row 8j + 4(l >> 5) + i,
// column l & 31; operand lanes hold k = 8(l >> 5) + 0..7.  Scores, cap, bias, softmax and the
// gate's sigmoid are fp32; the kernel serves 16-bit dtypes (fp32 models take the row kernel).
#include "mma.h"

using namespace lumen;

namespace {

// s + the products of 8 16-bit values at k with those of q
template <typename T> __device__ __forceinline__ float dot8(const T* k, const uint4& q, float s) {
  float x[8];
  load8<T>(k, x);
  const T* y = reinterpret_cast<const T*>(&q);
#pragma unroll
  for (int e = 0; e < 8; ++e) s = fmaf(x[e], to_f32(y[e]), s);
  return s;
}

// tanh through one exponential: 1 - 2 / (1 + e^(2x)); exact limits at both ends
__device__ __forceinline__ float tanh_exp(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __expf(2.f * x));
}

template <typename T>
struct WinTileArgs {
  const T* q; long long ldq;                 // rows [T][>= H * D]
  const T* kc; const T* vc;                  // [blocks][bs][G][D], [blocks][bs][G / vdiv][DV]
  // FRESH: the step's own rows, head after head (row strides ldk, ldv), and the kDr last columns of a key,
  // which the heads share
  const T* kr; long long ldk, ldv, ldr;
  T* out;                                    // [T][H][DV]
  const T* gate; long long gater;            // gate logits [T][H], row stride (nullable)
  const int* tables; int maxb;
  const int* tiles; const int* cu; const int* start;
  int H, G, bs;
  float scale, softcap;
  const float* slopes;                       // [H] (nullable)
  int window, keep;
  const float* sigb; int vdiv;               // sigmoid weights' bias [H] (nullable); key heads per value head
};

constexpr int kDr = 64;

// FRESH: prompts whose every key is a row of this step (positions from 0): keys and values are read where the
// projection left them and the block tables are not used.  A key is the head's own D - kDr columns, then kDr
// columns that all heads share.  Latent attention of fresh prompts (keys and values expanded from the latents): 192
// + 128 columns a score and value instead of 576 + 512, so ~0.3 of the products of latent_tile.hip.  us, projections
// around it included, absorbed -> expanded (bf16): 14 prompts of 63 - 509 tokens x 16 heads 197 -> 81 (this kernel
// 58), 8 x 512 224 -> 65, 1 x 512 72 -> 42, 1 x 30 60 -> 29, 1 x 2048 x 32 714 -> 141: at every size.  Error against
// float64, absorbed -> expanded: bf16 2.53e-3 -> 2.51e-3 and 2.57e-3 -> 2.53e-3, fp16 3.16e-4 -> 3.15e-4 (the weights through
// __expf; with an exponential near to the last bit the same, and 34 -> 40 us for 1 x 512).
template <typename T, int D, int DV, int NW, int KT, bool FRESH = false, int KS = 1>
__global__ void __launch_bounds__(64 * NW)
    __attribute__((amdgpu_waves_per_eu((D <= 128 || FRESH) && DV <= 128 ? 2 : 1)))
win_tile_attn_kernel(const WinTileArgs<T> a) {
  constexpr int QT = 32 * NW / KS, LK = D + 8, LT = KT + 8, NV = D / 8, NVV = DV / 8, SB = KT / 32, WB = SB / KS;
  static_assert(SB % KS == 0 && NW % KS == 0, "a wave's keys of a tile");
  // two buffers: a tile is stored while the one before it is read, one barrier per tile
  __shared__ __align__(16) T s_all[2 * KT * LK + 2 * DV * LT];
  T (*const s_kb)[KT * LK] = reinterpret_cast<T (*)[KT * LK]>(s_all);                    // key tile, row-major
  T (*const s_tb)[DV * LT] = reinterpret_cast<T (*)[DV * LT]>(s_all + 2 * KT * LK);      // value tile, transposed [d][key]
  static_assert(KS == 1 || NW / 2 * (DV / 2 + 2) * 64 * 4 <= (int)sizeof(s_all), "the other halves' results");
  constexpr int kTbl = 512;                   // block-table entries of the window's keys, in LDS
  __shared__ int s_tbl[kTbl];
  const int tid = threadIdx.x, lane = tid & 63, w = (tid >> 6) % (NW / KS), c = lane & 31, hi = lane >> 5;
  const int kb = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane((tid >> 6) / (NW / KS)) * WB;    // first block of 32 keys of a tile that the wave takes
  int tix, hd;
  heavy_first(blockIdx.x, gridDim.x, a.H, tix, hd);
  const int g = hd / (a.H / a.G);
  const int Gv = a.G / a.vdiv, gv = g / a.vdiv;
  const float sbias = a.sigb != nullptr ? a.sigb[hd] : 0.f;
  const int sg = a.tiles[2 * (tix / KS)], row0 = a.tiles[2 * (tix / KS) + 1] + tix % KS * QT;
  if (KS > 1 && row0 >= a.cu[sg + 1]) return;            // (the whole workgroup: a tile of the list with few rows)
  const int seg_r0 = a.cu[sg], p0 = a.start[sg];
  const int nrows = min(QT, a.cu[sg + 1] - row0);
  const int* tbl = a.tables + (long long)sg * a.maxb;
  const int window = a.window, keep = window > 0 ? a.keep : 0, bs = a.bs;

  const bool qv = 32 * w + c < nrows;
  const int qrow = row0 + 32 * w + c;
  const int pos = qv ? p0 + (qrow - seg_r0) : -1;
  uint4 qreg[D / 16];
#pragma unroll
  for (int kk = 0; kk < D / 16; ++kk)
    qreg[kk] = qv ? *reinterpret_cast<const uint4*>(a.q + (long long)qrow * a.ldq + hd * D + 16 * kk + 8 * hi)
                  : make_uint4(0, 0, 0, 0);
  const float slope = a.slopes != nullptr ? a.slopes[hd] : 0.f;
  const float cap = a.softcap, rcap = cap > 0.f ? 1.f / cap : 0.f;

  // key tiles: [0, khead) in steps of KT (kept keys below the window), then from kwin on
  const int pos_first = p0 + (row0 - seg_r0), kend = pos_first + nrows - 1;
  const int wlo = window > 0 ? max(0, pos_first - window + 1) : 0;
  const int kwin = wlo / 32 * 32;
  const int khead = min((min(keep, wlo) + KT - 1) / KT * KT, kwin);
  const int kfirst = khead > 0 ? 0 : kwin;
  auto next_tile = [&](int k0) {
    const int n = k0 + KT;
    return (n >= khead && n < kwin) ? kwin : n;
  };
  const bool wave_on = 32 * w < nrows;
  const int wpos_min = pos_first + 32 * w, wpos_max = min(kend, wpos_min + 31);

  // block ids of the keys the tile visits (the kept keys' blocks, then the window's), so that a key's
  // address never waits for a table load; a range of more than kTbl blocks is read from the table
  const int b_first = FRESH ? 0 : kwin / bs, b_head = khead > 0 ? min((khead + bs - 1) / bs, b_first) : 0;
  const int b_count = FRESH ? 0 : b_head + kend / bs - b_first + 1;
  const bool in_lds = b_count <= kTbl;
  if (!FRESH && in_lds)
    for (int i = tid; i < b_count; i += 64 * NW) s_tbl[i] = tbl[i < b_head ? i : i - b_head + b_first];
  const int bshift = (bs & (bs - 1)) == 0 ? __ffs(bs) - 1 : -1;
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  f32x16 O[DV / 32];
#pragma unroll
  for (int db = 0; db < DV / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) O[db][r] = 0.f;

  // staging: one item = 4 consecutive keys x 8 channels of the key cache or of the value cache (four
  // 16-byte loads); the row-major image takes the keys as they are, the transposed image takes eight
  // 8-byte stores of 4 values each (transposed in registers)
  constexpr int NT = 64 * NW, NK = D * SB, NTOT = (D + DV) * SB, ITEMS = (NTOT + NT - 1) / NT;
  uint4 pre[ITEMS][4];
  // cache rows of the four keys from j on (past the last key: that one again; `commit` blanks it).  The
  // rows come first and without a branch per key: then an item's four loads leave together
  auto cache_rows = [&](int j, long long (&row)[4]) __attribute__((always_inline)) {
    int jb[4], jo[4], blk[4];
    if (bshift >= 0) {
#pragma unroll
      for (int x = 0; x < 4; ++x) jb[x] = min(j + x, kend) >> bshift;
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) jb[x] = min(j + x, kend) / bs;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) jo[x] = min(j + x, kend) - jb[x] * bs;
    if (in_lds) {
#pragma unroll
      for (int x = 0; x < 4; ++x) blk[x] = s_tbl[jb[x] >= b_first ? jb[x] - b_first + b_head : jb[x]];
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) blk[x] = tbl[jb[x]];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) row[x] = (long long)blk[x] * bs + jo[x];
  };
  auto prefetch = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int item = tid + it * NT;
      const bool val = item >= NK;
      const int i = val ? item - NK : item;
      if (NTOT % NT != 0 && item >= NTOT) continue;
      const int kq = val ? i / NVV : i / NV, part = val ? i % NVV : i % NV;
      long long row[4];
      if constexpr (FRESH) {
        constexpr int P1 = (D - kDr) / 8;
        const T* base = val ? a.vc + gv * DV + 8 * part
                            : part < P1 ? a.kc + g * (D - kDr) + 8 * part : a.kr + 8 * (part - P1);
        const long long ld = val ? a.ldv : part < P1 ? a.ldk : a.ldr;
#pragma unroll
        for (int x = 0; x < 4; ++x)
          pre[it][x] = *reinterpret_cast<const uint4*>(base + (seg_r0 + min(k0 + 4 * kq + x, kend)) * ld);
        continue;
      }
      cache_rows(k0 + 4 * kq, row);
      const T* base = val ? a.vc + (long long)gv * DV + 8 * part : a.kc + (long long)g * D + 8 * part;
      const long long ld = val ? (long long)Gv * DV : (long long)a.G * D;
#pragma unroll
      for (int x = 0; x < 4; ++x) pre[it][x] = *reinterpret_cast<const uint4*>(base + row[x] * ld);
    }
  };
  auto commit = [&](int k0, T* s_k, T* s_t) __attribute__((always_inline)) {
    const bool tail = k0 + KT - 1 > kend;            // keys past the last one: zeros
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int item = tid + it * NT;
      const bool val = item >= NK;
      const int i = val ? item - NK : item;
      if (NTOT % NT != 0 && item >= NTOT) continue;
      const int kq = val ? i / NVV : i / NV, part = val ? i % NVV : i % NV;
      if (tail) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
          if (k0 + 4 * kq + x > kend) pre[it][x] = make_uint4(0, 0, 0, 0);
      }
      if (!val) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
          *reinterpret_cast<uint4*>(&s_k[(4 * kq + x) * LK + 8 * part]) = pre[it][x];
      } else {
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
  auto tile = [&](int kt, const T* s_k, const T* s_t) __attribute__((always_inline)) {
    const int k0 = kt + 32 * kb;             // first of the wave's keys
    // nothing this wave may see: past its last row, or before its first row's window and not kept
    if (!wave_on || k0 > wpos_max ||
        (window > 0 && k0 + 32 * WB - 1 < wpos_min - window + 1 && k0 >= keep))
      return;

    f32x16 sc[WB];
#pragma unroll
    for (int b = 0; b < WB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[b][r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk)
#pragma unroll
      for (int b = 0; b < WB; ++b)
        sc[b] = Mma32<T>::run(*reinterpret_cast<const uint4*>(&s_k[(32 * (kb + b) + c) * LK + 16 * kk + 8 * hi]),
                              qreg[kk], sc[b]);
    // register r of sc[b] is key k0 + key_of(b, r)
    const auto key_of = [&](int b, int r) { return 32 * b + 8 * (r >> 2) + 4 * hi + (r & 3); };
    // a tile every query of the wave sees whole needs no mask
    const bool whole = k0 + 32 * WB - 1 <= wpos_min && 32 * w + 31 < nrows &&
                       (window <= 0 || k0 >= wpos_max - window + 1 || k0 + 32 * WB - 1 < keep);
#pragma unroll
    for (int b = 0; b < WB; ++b) sc[b] *= a.scale;
    if (cap > 0.f) {
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[b][r] = cap * tanh_exp(sc[b][r] * rcap);
    }
    if (a.slopes != nullptr) {
      const float d0 = (float)(pos - k0);
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[b][r] -= slope * (d0 - (float)key_of(b, r));
    }
    if (!whole) {
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int j = k0 + key_of(b, r);
          const bool seen = j <= pos && (window <= 0 || pos - j < window || j < keep);
          sc[b][r] = seen ? sc[b][r] : -INFINITY;
        }
    }
    if (a.sigb != nullptr) {
      // weights as they are: a hidden key's -inf gives 1 / (1 + e^inf) = 0
#pragma unroll
      for (int b = 0; b < WB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[b][r] = 1.f / (1.f + __expf(-(sc[b][r] + sbias)));
    } else {
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
        for (int db = 0; db < DV / 32; ++db)
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
      l += psum;                               // (the lane's half: the other lane's is added at the end)
    }
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
      for (int db = 0; db < DV / 32; ++db) {
        // quads 4 s2 + hi and 4 s2 + 2 + hi of row 32 db + c, under the store's permutation: both low
        // bits lie in t0 / t1, the others in the instruction's offset
        const int at = 32 * db * LT + 32 * (s2 >> 1) + 16 * ((s2 & 1) ^ (db & 1));
        const uint2 a0 = *reinterpret_cast<const uint2*>(s_t + t0 + at);
        const uint2 a1 = *reinterpret_cast<const uint2*>(s_t + t1 + at);
        const uint4 av = make_uint4(a0.x, a0.y, a1.x, a1.y);
        O[db] = Mma32<T>::run(av, bh, O[db]);
        O[db] = Mma32<T>::run(av, bl, O[db]);
      }
    }
  };

  // tile n is stored after tile n - 1 was read: the loads of a tile have the products of the one before
  // it to arrive in
  prefetch(kfirst);
  commit(kfirst, s_kb[0], s_tb[0]);
  __builtin_amdgcn_s_waitcnt(0xF70);       // vmcnt(0): or the loop's first product would wait, every time, for
  __syncthreads();                         // the queries, and with them for the tile just asked for
  for (int k0 = kfirst, cur = 0; k0 <= kend; cur ^= 1) {
    const int kn = next_tile(k0);
    if (kn <= kend) prefetch(kn);
    tile(k0, s_kb[cur], s_tb[cur]);
    if (kn <= kend) commit(kn, s_kb[cur ^ 1], s_tb[cur ^ 1]);
    __syncthreads();
    k0 = kn;
  }
  if constexpr (KS == 2) {                   // the upper keys' waves hand their sums to the lower ones'
    float* box = reinterpret_cast<float*>(s_all) + w * (DV / 2 + 2) * 64 + lane;
    if (kb > 0) {
#pragma unroll
      for (int db = 0; db < DV / 32; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) box[(16 * db + r) * 64] = O[db][r];
      box[DV / 2 * 64] = m;
      box[(DV / 2 + 1) * 64] = l;
    }
    __syncthreads();
    if (kb > 0) return;
    const float m2 = box[DV / 2 * 64], mn = fmaxf(m, m2);
    const float c1 = m == mn ? 1.f : __expf(m - mn), c2 = m2 == mn ? 1.f : __expf(m2 - mn);
    l = l * c1 + box[(DV / 2 + 1) * 64] * c2;
    m = mn;
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) O[db][r] = O[db][r] * c1 + box[(16 * db + r) * 64] * c2;
  }
  l += __shfl_xor(l, 32, 64);
  // A hidden key has weight 0, but 0 times an infinite or NaN value is NaN: channels that are not finite are formed
  // again, key by key over what the row sees (m and l stand).
  float odd[4] = {0.f, 0.f, 0.f, 0.f};             // (0 times a finite number stays 0)
#pragma unroll
  for (int db = 0; db < DV / 32; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) odd[r & 3] = fmaf(O[db][r], 0.f, odd[r & 3]);
  if (__builtin_expect(__any(odd[0] + odd[1] + odd[2] + odd[3] != 0.f && qv), 0)) {
#pragma unroll
    for (int db = 0; db < DV / 32; ++db) {
      f32x16 o;
#pragma unroll
      for (int r = 0; r < 16; ++r) o[r] = 0.f;
      for (int j = kfirst; j <= wpos_max; ++j) {
        if (window > 0 && j >= keep) j = max(j, wpos_min - window + 1);
        const T *kp, *kr, *vp;
        if constexpr (FRESH) {
          kp = a.kc + (seg_r0 + j) * a.ldk + g * (D - kDr);
          kr = a.kr + (seg_r0 + j) * a.ldr - (D - kDr);
          vp = a.vc + (seg_r0 + j) * a.ldv + gv * DV;
        } else {
          const int jb = j / bs;
          const long long row = (long long)tbl[jb] * bs + (j - jb * bs);
          kp = kr = a.kc + (row * a.G + g) * D;
          vp = a.vc + (row * Gv + gv) * DV;
        }
        float s = 0.f;
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
          __builtin_amdgcn_sched_barrier(0);     // (one load at a time: registers)
          s = dot8<T>((FRESH && 16 * kk >= D - kDr ? kr : kp) + 16 * kk + 8 * hi, qreg[kk], s);
        }
        s = (s + __shfl_xor(s, 32, 64)) * a.scale;
        if (cap > 0.f) s = cap * tanh_exp(s * rcap);
        s -= slope * (float)(pos - j);
        const float p = a.sigb != nullptr ? 1.f / (1.f + __expf(-(s + sbias))) : __expf(s - m);
        if (j > pos || (window > 0 && pos - j >= window && j >= keep)) continue;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          float v[4];
          load4<T>(vp + 32 * db + 8 * q4 + 4 * hi, v);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[4 * q4 + e] = fmaf(p, v[e], o[4 * q4 + e]);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) O[db][r] = fabsf(O[db][r]) < INFINITY ? O[db][r] : o[r];
    }
  }
  if (qv) {
    float inv = a.sigb != nullptr ? 1.f : 1.f / l;   // l > 0: a row always sees its own key
    if (a.gate != nullptr) inv *= sigmoid_f(to_f32(a.gate[(long long)qrow * a.gater + hd]));
    T* op = a.out + ((long long)qrow * a.H + hd) * DV;
#pragma unroll
    for (int db = 0; db < DV / 32; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 32 * db + 8 * j + 4 * hi;
        const unsigned x0 = pk2<T>(O[db][4 * j] * inv, O[db][4 * j + 1] * inv);
        const unsigned x1 = pk2<T>(O[db][4 * j + 2] * inv, O[db][4 * j + 3] * inv);
        *reinterpret_cast<uint2*>(op + d) = make_uint2(x0, x1);
      }
  }
}

// Tiles of 128 rows by heads up to which tiles of 64 rows with the keys in halves are faster.  us, whole -> in halves: heads of 128
// 64 workgroups (1 x 512 x 16) 28.5 -> 21.4, 128 (x 32, soft cap) 33.0 -> 23.8, 256 (1 x 1024 x 32) 58.1 -> 44.9, (4 x 512 x 16) 30.2 -> 25.4, 100
// rows behind 3000 keys 182 -> 126; 320 35.7 -> 34.8, 512 (8 x 512 x 16) 37.4 -> 47.1; heads of 64, 128 21.0 -> 15.7.  Two such workgroups share
// a CU; of the fresh form one does: 64 workgroups (1 x 512 x 16) 33.3 -> 24.9, 128 (1 x 2048 x 8) 106.8 -> 76.6, 192 34.0 -> 40.1; its
// key tiles are longer then, for nothing with portions of up to 64 rows (30 rows 6.8 -> 8.7).
constexpr int kSplit = 256, kSplitFresh = 128;

template <typename T>
hipError_t launch_win_tiles(const WinTileArgs<T>& a, int ntiles, int D, int Dv, int tile_rows,
                            hipStream_t st) {
  const dim3 grid((unsigned)((long long)ntiles * a.H));
#define GO(DD, DVV)                                                                          \
  {                                                                                          \
    constexpr int KT = DVV <= 128 ? 64 : 32;                                                 \
    if constexpr (KT == 64) {                                                                \
      if (tile_rows == 128 && (long long)ntiles * a.H <= kSplit) {                           \
        win_tile_attn_kernel<T, DD, DVV, 4, KT, false, 2><<<2 * grid.x, 256, 0, st>>>(a);    \
        return hipGetLastError();                                                            \
      }                                                                                      \
    }                                                                                        \
    if (tile_rows == 128) win_tile_attn_kernel<T, DD, DVV, 4, KT><<<grid, 256, 0, st>>>(a);  \
    else win_tile_attn_kernel<T, DD, DVV, 2, KT><<<grid, 128, 0, st>>>(a);                   \
  }
  switch (D * 1024 + Dv) {
    case 32 * 1024 + 32: GO(32, 32); break;
    case 64 * 1024 + 64: GO(64, 64); break;
    case 96 * 1024 + 96: GO(96, 96); break;
    case 128 * 1024 + 128: GO(128, 128); break;
    case 192 * 1024 + 192: GO(192, 192); break;
    case 256 * 1024 + 256: GO(256, 256); break;
    // values twice the key size (two score maps per head, or wide values)
    case 32 * 1024 + 64: GO(32, 64); break;
    case 48 * 1024 + 96: GO(48, 96); break;
    case 64 * 1024 + 128: GO(64, 128); break;
    case 96 * 1024 + 192: GO(96, 192); break;
    case 128 * 1024 + 256: GO(128, 256); break;
    default: return hipErrorInvalidValue;
  }
#undef GO
  return hipGetLastError();
}

template <typename T>
hipError_t launch_fresh_tiles(const WinTileArgs<T>& a, int rows, int ntiles, int tile_rows, hipStream_t st) {
  const dim3 grid((unsigned)((long long)ntiles * a.H));
  if (tile_rows == 128 && (long long)ntiles * a.H <= kSplitFresh && rows > 64LL * ntiles)
    win_tile_attn_kernel<T, 192, 128, 4, 64, true, 2><<<2 * grid.x, 256, 0, st>>>(a);
  else if (tile_rows == 128) win_tile_attn_kernel<T, 192, 128, 4, 32, true><<<grid, 256, 0, st>>>(a);
  else win_tile_attn_kernel<T, 192, 128, 2, 32, true><<<grid, 128, 0, st>>>(a);
  return hipGetLastError();
}

}  // namespace

extern "C" {

// Prompts from position 0 whose keys and values are rows of the step: q rows [T][>= H * (D1 + Dr)], k rows
// [T][>= H * D1] and v rows [T][>= H * Dv] head after head, kr rows [T][>= Dr] the key part all heads share;
// D1 = Dv = 128, Dr = 64; row strides % 8, 16-byte aligned bases; out [T][H][Dv] contiguous; tiles, cu and start
// as below (every start is 0); rows: of all tiles.
int sm_fresh_tiles_ok(int dt, int D1, int Dr, int Dv) {
  return (dt == kBF16 || dt == kF16) && D1 == 128 && Dr == kDr && Dv == 128;
}

hipError_t sm_fresh_tiles(int dt, const void* q, long long ldq, const void* k, long long ldk, const void* kr,
                          long long ldr, const void* v, long long ldv, void* out, const int* tiles, int rows, int ntiles,
                          int tile_rows, const int* cu, const int* start, int H, int D1, int Dr, int Dv,
                          float scale, hipStream_t st) {
  if (ntiles == 0) return hipSuccess;
  if (!sm_fresh_tiles_ok(dt, D1, Dr, Dv) || ntiles < 0 || rows < 0 || H < 1 || (tile_rows != 64 && tile_rows != 128) ||
      ldq % 8 || ldk % 8 || ldr % 8 || ldv % 8 || ldq < (long long)H * (D1 + Dr) || ldk < (long long)H * D1 ||
      ldr < Dr || ldv < (long long)H * Dv ||
      ((uintptr_t)q | (uintptr_t)k | (uintptr_t)kr | (uintptr_t)v) % 16 || (uintptr_t)out % 8)
    return hipErrorInvalidValue;
#define CALL(TT)                                                                                          \
  {                                                                                                       \
    WinTileArgs<TT> a{(const TT*)q, ldq, (const TT*)k, (const TT*)v, (const TT*)kr, ldk, ldv, ldr, (TT*)out, \
                      nullptr, 0, nullptr, 0, tiles, cu, start, H, H, 1, scale, 0.f, nullptr, 0, 0, nullptr, 1}; \
    return launch_fresh_tiles<TT>(a, rows, ntiles, tile_rows, st);                                        \
  }
  if (dt == kBF16) CALL(bf16)
  CALL(fp16)
#undef CALL
}

// 1 when sm_win_attn_tiles has a kernel for this dtype / key size / value size
int sm_win_attn_tiles_ok(int dt, int D, int Dv) {
  if (dt != kBF16 && dt != kF16) return 0;
  if (Dv == D) return D == 32 || D == 64 || D == 96 || D == 128 || D == 192 || D == 256;
  return Dv == 2 * D && (D == 32 || D == 48 || D == 64 || D == 96 || D == 128);
}

// tiles: [ntiles, 2] int32 (segment, first row); every tile covers up to tile_rows (64 or 128)
// rows of its segment.  q rows [T][>= H * D] with row stride ldq (a multiple of 8, 16-byte
// aligned base); kc [blocks][bs][G][D], vc [blocks][bs][G / vdiv][Dv]; out [T][H][Dv] contiguous;
// gate (nullable) [T][H] with row stride gater; slopes (nullable) fp32 [H]; window 0: plain causal
// attention; sigb (nullable) fp32 [H]: sigmoid weights, not normalised.
hipError_t sm_win_attn_tiles(int dt, const void* q, long long ldq, const void* kc, const void* vc,
                             void* out, const void* gate, long long gater, const int* tables,
                             int maxb, const int* tiles, int ntiles, const int* cu,
                             const int* start, int H, int G, int D, int bs, float scale,
                             float softcap, const float* slopes, int window, int keep,
                             int tile_rows, int Dv, const float* sigb, int vdiv, hipStream_t st) {
  if (ntiles == 0) return hipSuccess;
  if (vdiv < 1 || G % vdiv || !sm_win_attn_tiles_ok(dt, D, Dv)) return hipErrorInvalidValue;
  if (G < 1 || H % G || bs < 1 || window < 0 || keep < 0 || (ldq % 8) != 0 ||
      (uintptr_t)q % 16 || (uintptr_t)kc % 16 || (uintptr_t)vc % 16 || (uintptr_t)out % 8)
    return hipErrorInvalidValue;
  if (tile_rows != 64 && tile_rows != 128) return hipErrorInvalidValue;
#define CALL(TT)                                                                               \
  {                                                                                            \
    WinTileArgs<TT> a{(const TT*)q, ldq, (const TT*)kc, (const TT*)vc, nullptr, 0, 0, 0, (TT*)out, \
                      (const TT*)gate, gater, tables, maxb, tiles, cu, start, H, G, bs, scale, \
                      softcap, slopes, window, keep, sigb, vdiv};                              \
    return launch_win_tiles<TT>(a, ntiles, D, Dv, tile_rows, st);                              \
  }
  if (dt == kBF16) CALL(bf16)
  if (dt == kF16) CALL(fp16)
#undef CALL
  return hipErrorInvalidValue;
}

}  // extern "C"
