// Routed experts over the rows that chose them (prompt steps): for every row t with weights r[t, e] (dense, zero off
// the chosen experts), out[t] = sum_e W_down,e act(W_gate,e h_t, W_up,e h_t; r[t, e]) (+ the shared expert's).
//   sm_expert_sort    the (row, expert) pairs in expert order, rows ascending: one workgroup per expert
//   sm_expert_act     first projection and activation of all pairs and of the shared expert
//   sm_expert_down    second projection, fp32 results per pair
//   sm_expert_sum     out[t] = the sum of the row's pairs in expert order and of its shared result, rounded once
//
// The dense form (two library products over ALL experts, ops/moe.py) does E / top times the work; the library's
// grouped product runs at 300 TFLOP/s.  Here a workgroup takes 64, 128 or 256 pairs of one expert and 256 rows of its weights,
// both products on the loop of kernels/tile_loop.h:
//  * the rows of a tile are gathered by the DMA's source addresses; no sorted copy of h exists;
//  * a wave's weight rows of the first product are alternating fragments of 16 gate rows and their 16 up rows, so the activation
//    with the routing weight is formed from the fp32 sums and the [pairs, 2 ff] intermediate is never stored;
//  * counts stay on the device: the grid is sized for the most tiles the step can have and the surplus leaves at once.
//    Nothing synchronises, nothing depends on host-visible counts (a capture may hold it);
//  * XCDs take consecutive tiles, an expert's row tiles within a weight panel first: a panel comes from HBM once;
//  * a tile occupies its CU, so the time goes by whole rounds of 256 tiles: tiles of 256 pairs run whole rounds, and what is
//    left over, known on the device, is cut into two or four smaller tiles each where those make one round.
// Bound by the rounds: a tile of 256 x 256 takes 1.25 us a stage of 64 k, as in the dense products, and 11 us around them (first
// stages, activation, stores); under ~200 rows by reading the weights once.  Measured (us, a whole layer of experts, weights from
// HBM, bf16; tiles of 128 pairs alone, on a loop of their own -> here): width 2048, 8 experts of 1408, top 2, and a
// shared one: 4096 rows 294 -> 247, 2048 172 -> 141, 512 77 -> 74, 160 70 -> 66; 16, top 3, shared: 4096 373 -> 336, 1024 148 ->
// 127, 256 91 -> 87, 64 84 -> 82; 16 ungated, top 4: 4096 298 -> 251; width 4096, 16 of 2816, top 4: 8192 rows 2370 -> 2026, 300
// 257 -> 258; dense form: 4096 rows of the first 534, of the second 1130.  Error against float64 2.3e-3 where the dense form has
// 3.5e-3: nothing is rounded between the products and the activation, nor before the sum.
#include "mma.h"
#include "../kernels/tile_loop.h"

using namespace lumen;

namespace {

constexpr int BN = 256, BK = tile::BK;                   // weight rows of a tile
constexpr int kMaxE = 64;

struct ExpertArgs {
  const void *x, *xs;          // rows of the experts' (gathered) and of the shared expert's product
  long long ldx, ldxs;
  const void* w;               // stacked weights, row stride ldw
  long long ldw;
  void *y, *ys;                // results of the pairs and of the shared expert
  const int* off;              // [E + 1]: an expert's first pair
  const int* idx;              // [pairs] row of a pair (null: pairs follow each other in x)
  const float* wt;             // [pairs] routing weight
  int T, W, E, ff, ffs;
  GateForm form;
};

// sigmoid on the exponential and reciprocal units (the results are rounded to 16 bits)
__device__ __forceinline__ float sigmoid_fast(float x) { return __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

// MODE 0: column (of 64) of row r of a wave's 128 weight rows, alternating fragments of 16 gate and their 16 up rows; a
// lane's fragments of two such pairs hold 8 consecutive columns
__device__ __forceinline__ int gate_col(int r) {
  return 32 * (r >> 6) + 8 * ((r >> 2) & 3) + 4 * ((r >> 5) & 1) + (r & 3);
}

// activation results of pair fragment j (MODE 0: acc[even]: gate, acc[odd]: up)
template <typename T, int MODE, int NI, int MJ, int ACT>
__device__ __forceinline__ void put_row(const GateForm& f, tile::f32x4 (&acc)[NI][MJ], int j, T* o, int c0, int ff,
                                        int wn, int lg, float w, bool shared) {
  const float wi = f.weigh_in ? w : 1.f, wo = f.weigh_in ? 1.f : w, lim = shared ? f.limit_s : f.limit;
  const auto act = [&](float g) {
    if constexpr (ACT == 0) return g * sigmoid_fast(g);
    else return gate_act(g, ACT);
  };
  constexpr int STEP = MODE == 0 ? 4 : 2;                // fragments of 8 columns
#pragma unroll
  for (int i = 0; i < NI; i += STEP) {
    const int col = c0 + (MODE == 0 ? 8 : 16) * (NI * wn + i) + 8 * lg;
    unsigned out[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float r[4];
      tile::f32x4& a0 = acc[i + STEP / 2 * h][j];
      tile::hold(a0);
      if constexpr (MODE == 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] = act(a0[q] * wi) * wo;
      } else {
        tile::f32x4& a1 = acc[i + 2 * h + 1][j];
        tile::hold(a1);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float g = a0[q] * wi, u = a1[q] * wi;
          if constexpr (ACT == 4) {
            g = fminf(g, lim);
            u = fminf(fmaxf(u, -lim), lim);
            r[q] = g * sigmoid_fast(f.slope * g) * (u + f.shift) * wo;
          } else {
            r[q] = act(g) * u * wo;
          }
        }
      }
      out[2 * h] = pk2<T>(r[0], r[1]);
      out[2 * h + 1] = pk2<T>(r[2], r[3]);
    }
    if (col < ff) *reinterpret_cast<uint4*>(o + col) = make_uint4(out[0], out[1], out[2], out[3]);
  }
}

// the tile of an expert's (or the shared one's) pairs m0 .. and result columns c0 ..: 32 MJ pairs by 32 NI weight rows.
// MODE 0: gate and up rows -> activation ACT (GateForm's), 1: up rows alone -> activation, 2: second projection -> fp32.
// (A choice of the activation at run time makes the compiler copy accumulators, which it does not know to be under way still,
// between the products; chosen inside the element it also made the epilogue 14000 instructions long.)
template <typename T, int MODE, int NI, int MJ, int ACT>
__device__ __forceinline__ void run_tile(const ExpertArgs& a, char* lds, int e, int r0, int rows, int m0, int c0) {
  constexpr int PIECES = tile::Shape<NI, MJ>::PIECES;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const bool shared = e == a.E;
  const int ff = shared ? a.ffs : a.ff;
  const int nk = MODE == 2 ? (ff + BK - 1) / BK : a.W / BK, N = MODE == 2 ? a.W : ff;
  const T* x = (const T*)(shared ? a.xs : a.x);
  const long long ldx = shared ? a.ldxs : a.ldx;
  const bool gather = MODE != 2 && !shared;
  const char* xb = (const char*)(x + (gather ? 0 : (long long)(r0 + m0) * ldx));
  // weights: MODE 0 / 1 row blocks per expert, MODE 2 column blocks
  const char* wb = (const char*)((const T*)a.w + (MODE == 2 ? (long long)c0 * a.ldw + (long long)e * a.ff
                                                            : (long long)e * (MODE == 0 ? 2 : 1) * a.ff * a.ldw));
  unsigned off[PIECES];                                  // (past the edges the last row is read: never stored)
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int r = 8 * (wid + 4 * (q < MJ ? q : q - MJ)) + (lane >> 3), c = (lane & 7) ^ tile::swz(r);
    if (q < MJ) {
      const int i = min(r, rows - m0 - 1);
      off[q] = (unsigned)(gather ? a.idx[r0 + m0 + i] : i) * (unsigned)(2 * ldx) + 16 * c;
    } else if (MODE == 0) {
      const int col = min(c0 + r / (16 * NI) * (8 * NI) + gate_col(r % (16 * NI)), ff - 1);
      off[q] = (unsigned)(col + ((r >> 4) & 1 ? ff : 0)) * (unsigned)(2 * a.ldw) + 16 * c;
    } else {
      const int col = r / (16 * NI) * (16 * NI) + tile::colperm<NI>(r % (16 * NI));
      off[q] = (unsigned)(MODE == 1 ? min(c0 + col, ff - 1) : min(col, N - c0 - 1)) * (unsigned)(2 * a.ldw) + 16 * c;
    }
  }
  tile::f32x4 acc[NI][MJ];
  tile::products<T, NI, MJ, false, MODE == 2>(lds, xb, wb, nk, 0, off, acc, MODE == 2 && ff % BK != 0);
  // lane (lr, lg) holds pair 16 j + lr, weight rows 16 i + 4 lg .. + 3 of its wave's block
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int m = m0 + 16 * MJ * wm + 16 * j + lr;
    if (m >= rows) continue;
    if constexpr (MODE == 2) {
      float* o = (float*)(shared ? a.ys : a.y) + (long long)(r0 + m) * a.W;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int col = c0 + 16 * NI * wn + 32 * (i >> 1) + 8 * lg + 4 * (i & 1);
        tile::hold(acc[i][j]);
        if (col < N) *reinterpret_cast<tile::f32x4*>(o + col) = acc[i][j];
      }
    } else {
      const float wt = shared ? 1.f : a.wt[r0 + m];
      T* o = (T*)(shared ? a.ys : a.y) + (long long)(r0 + m) * ff;
      put_row<T, MODE, NI, MJ, ACT>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared);
    }
  }
}

// Tiles of 32 MJ pairs and 256 weight rows.  MJ 8: whole rounds of the CUs; what is left over is cut into two or four where that
// makes one round of smaller tiles.
template <typename T, int MODE, int MJ, int ACT>
__global__ void __launch_bounds__(256, 1) expert_kernel(const ExpertArgs a) {
  constexpr int BM = 32 * MJ, CT = MODE == 0 ? BN / 2 : BN;            // rows and result columns of a tile
  __shared__ __attribute__((aligned(16))) char lds[MJ == 8 && tile::Shape<8, 4>::LDS > tile::Shape<8, 8>::LDS
                                                       ? tile::Shape<8, 4>::LDS : tile::Shape<8, MJ>::LDS];
  static_assert(tile::Shape<4, 4>::LDS <= 163840);
  const int lane = threadIdx.x & 63;
  // the tile: experts in order (the shared one last), weight panels in order, row tiles within a panel
  const int ce = ((MODE == 2 ? a.W : a.ff) + CT - 1) / CT, cs = a.ffs > 0 ? ((MODE == 2 ? a.W : a.ffs) + CT - 1) / CT : 0;
  const int rows_e = lane < a.E ? a.off[lane + 1] - a.off[lane] : 0;
  int pre = (rows_e + BM - 1) / BM;                      // inclusive prefix of row tiles over the lanes
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int n = __shfl_up(pre, o, 64);
    if (lane >= o) pre += n;
  }
  const int tiles_e = __builtin_amdgcn_readlane(pre, 63) * ce, ts = (a.T + BM - 1) / BM;
  const int total = tiles_e + ts * cs, b = blockIdx.x;
  int v, cut = 1, part = 0;
  if constexpr (MJ == 8) {
    const int full = total / tile::CUS * tile::CUS, left = total - full;
    if (b < full) {
      v = tile::unit_of(b, full);
    } else {
      cut = 4 * left <= tile::CUS ? 4 : 2 * left <= tile::CUS ? 2 : 1;
      if (b - full >= cut * left) return;
      const int u = tile::unit_of(b - full, cut * left);
      v = full + u / cut;
      part = u % cut;
    }
  } else {
    if (b >= total) return;
    v = tile::unit_of(b, total);
  }
  int e = a.E, r0 = 0, rows = a.T, u = v - tiles_e, nt = ts;
  if (v < tiles_e) {
    e = __popcll(__ballot(pre * ce <= v));               // (lanes past E hold the total: never counted)
    e = __builtin_amdgcn_readfirstlane(e);
    const int before = e > 0 ? __builtin_amdgcn_readlane(pre, e - 1) : 0;
    nt = __builtin_amdgcn_readlane(pre, e) - before;
    u = v - before * ce;
    r0 = a.off[e];
    rows = a.off[e + 1] - r0;
  }
  const int tn = u / nt, m0 = (u - tn * nt) * BM, c0 = tn * CT;
  if constexpr (MJ == 8) {
    if (cut > 1) {
      const int m = m0 + BM / 2 * (part & 1), c = c0 + CT / 2 * (part >> 1);
      if (m >= rows || c >= (MODE == 2 ? a.W : e == a.E ? a.ffs : a.ff)) return;
      if (cut == 2) run_tile<T, MODE, 8, 4, ACT>(a, lds, e, r0, rows, m, c0);
      else run_tile<T, MODE, 4, 4, ACT>(a, lds, e, r0, rows, m, c);
      return;
    }
  }
  run_tile<T, MODE, 8, MJ, ACT>(a, lds, e, r0, rows, m0, c0);
}

// One workgroup per expert e: pairs of experts before e are counted along the way (a row's chosen experts below e
// also give the pair's place among the row's), then e's pairs are numbered in row order.  A thread takes four rows of
// 4096 at a time, as bit masks of their experts.
__global__ void __launch_bounds__(1024)
expert_sort_kernel(const float* __restrict__ wts, int* __restrict__ off, int* __restrict__ idx,
                   float* __restrict__ wt, int* __restrict__ place, int T, int E, int top) {
  __shared__ int s_n[4][16], s_b[16];
  const int e = blockIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned long long lower = (1ull << e) - 1;
  unsigned long long mask[4];
  const auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) mask[i] = 0;
    if (E % 4 == 0 && (uintptr_t)wts % 16 == 0) {
#pragma unroll 4
      for (int c = 0; c < E; c += 4)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = t0 + 1024 * i + (int)threadIdx.x;
          const f32x4 v = t < T ? *reinterpret_cast<const f32x4*>(wts + (long long)t * E + c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < 4; ++q) mask[i] |= (unsigned long long)(v[q] != 0.f) << (c + q);
        }
    } else {
      for (int c = 0; c < E; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = t0 + 1024 * i + (int)threadIdx.x;
          mask[i] |= (unsigned long long)(t < T && wts[(long long)t * E + c] != 0.f) << c;
        }
    }
  };
  int before = 0;
  for (int t0 = 0; t0 < T; t0 += 4096) {
    load(t0);
#pragma unroll
    for (int i = 0; i < 4; ++i) before += min(__popcll(mask[i] & lower), top);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
  if (lane == 0) s_b[w] = before;
  __syncthreads();
  int at = 0;
#pragma unroll
  for (int i = 0; i < 16; ++i) at += s_b[i];
  if (threadIdx.x == 0) off[e] = at;
  for (int t0 = 0; t0 < T; t0 += 4096) {
    if (T > 4096) load(t0);
    unsigned long long rank[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {                          // (no row has more than `top` pairs, whatever it holds)
      const bool on = (mask[i] >> e & 1) && __popcll(mask[i] & lower) < top;
      rank[i] = __ballot(on);
      if (lane == 0) s_n[i][w] = __popcll(rank[i]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + 1024 * i + (int)threadIdx.x;
      int p = at;
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        if (x < w) p += s_n[i][x];
        at += s_n[i][x];
      }
      const int k = __popcll(mask[i] & lower);
      const bool on = rank[i] >> lane & 1;
      if (on) {
        p += __popcll(rank[i] & ((1ull << lane) - 1));
        idx[p] = t;
        wt[p] = wts[(long long)t * E + e];
        place[(long long)t * top + k] = p;
      }
      if (e == E - 1 && t < T)
        for (int x = min(k, top) + on; x < top; ++x) place[(long long)t * top + x] = -1;
    }
    __syncthreads();
  }
  if (e == E - 1 && threadIdx.x == 0) off[E] = at;
}

template <typename T>
__global__ void __launch_bounds__(256)
expert_sum_kernel(const float* __restrict__ y, const float* __restrict__ ys, const int* __restrict__ place,
                  T* __restrict__ out, int top, int W) {
  const long long t = blockIdx.x;
  const int c = 4 * (blockIdx.y * 256 + threadIdx.x);
  if (c >= W) return;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < top; ++k) {
    const int p = place[t * top + k];
    if (p >= 0) s += *reinterpret_cast<const f32x4*>(y + (long long)p * W + c);
  }
  if (ys != nullptr) s += *reinterpret_cast<const f32x4*>(ys + t * W + c);
  *reinterpret_cast<uint2*>(out + t * W + c) = make_uint2(pk2<T>(s[0], s[1]), pk2<T>(s[2], s[3]));
}

bool sizes_ok(int dt, int T, int W, int E, int top, int ff, int ffs) {
  return (dt == kBF16 || dt == kF16) && T >= 1 && W >= BK && W % BK == 0 && E >= 1 && E <= kMaxE && top >= 1 &&
         top <= E && ff >= 32 && ff % 32 == 0 && ffs >= 0 && ffs % 32 == 0 && (long long)T * top < (1 << 30) &&
         (long long)(2 * E * (long long)ff + 2 * ffs) * W < (1LL << 40);
}
constexpr int kMinRows = 64;                             // of a tile
// the most tiles of `bm` rows and ce (an expert's) or cs (the shared one's) column tiles
long long tiles_of(int T, int E, int top, int bm, long long ce, long long cs) {
  return ((long long)T * top / bm + E) * ce + (long long)((T + bm - 1) / bm) * cs;
}

// Rows of a tile / 32: the least time expected of all rounds of the CUs; an expert's and the shared one's weights in bytes.  The host
// knows T top / E rows an expert, more or less by their root and some for routers that prefer: the tiles are counted at eight places of that
// spread, the rounds at that many and at their own spread above and below.  us a tile by stages of 64 k, and the memory's time for the
// weights (behind which tiles of 256 rows leave the more to do), fitted to 616 sizes and routings by chance and by preference: over the best
// of the three the choice takes 1.1 % more time on average, by the mean and one spread alone it took 1.8 %, tiles of 128 always 11 % (act, us,
// rows 64 / 128 / 256: 256 rows, 4 experts of 5632, width 2048 67 / 45 / 55, 512 rows 61 / 75 / 55; 512 rows, 8 of 2816, width 4096 113 / 137 / 102;
// 4096 rows, 8 of 1408 and a shared one 240 / 165 / 139).
int pick_rows(int T, int E, int top, int nk, int ce, int cs, double expert, double shared) {
  static const double kPlaces[8] = {-1.53, -0.89, -0.49, -0.16, 0.16, 0.49, 0.89, 1.53};
  const double r = (double)T * top / E, s = 1.25 * sqrt(r);
  const double t4 = 0.86 * nk + 10., t2 = 0.56 * nk + 8., cut = 0.33 * nk + 7., t8 = 1.2 * nk + 6.;
  double chosen = 0.;                                     // the share of experts with rows
  for (const double z : kPlaces) chosen += r + z * s > 0.5 ? 0.125 : 0.;
  const double memory = (E * chosen * expert + shared) / 6.3e6;
  const auto expected = [&](int bm, double least, const auto& cost) {
    double sum = 0., sq = 0.;
    for (const double z : kPlaces) {
      const double x = r + z * s, n = x <= 0.5 ? 0. : ceil(x / bm);
      sum += n;
      sq += n * n;
    }
    const double mean = sum / 8., each = sqrt(fmax(0., sq / 8. - mean * mean) * E) * ce;
    const double n = mean * E * ce + (double)((T + bm - 1) / bm) * cs;
    return fmax(least, cost(ceil(n - each))) + fmax(least, cost(ceil(n))) + fmax(least, cost(ceil(n + each)));
  };
  const double all8 = expected(256, memory + 16., [&](double n) {
    const double full = floor(n / tile::CUS), left = n - full * tile::CUS;
    return full * t8 + (left <= 0. ? 0. : 4 * left <= tile::CUS ? cut : 2 * left <= tile::CUS ? t4 : t8);
  });
  const double all4 = expected(128, memory, [&](double n) { return ceil(n / tile::CUS) * t4; });
  const double all2 = expected(64, memory, [&](double n) { return ceil(n / tile::CUS) * t2; });
  return all8 < all4 && all8 < all2 ? 8 : all4 <= all2 ? 4 : 2;
}

template <typename T, int MODE, int ACT>
hipError_t launch(const ExpertArgs& p, int top, int ce, int cs, hipStream_t st) {
  const int nk = (MODE == 2 ? (p.ff > p.ffs ? p.ff : p.ffs) : p.W) / BK;
  const double row = (MODE == 0 ? 4. : 2.) * p.W;         // bytes of weights for an activation
  const int mj = pick_rows(p.T, p.E, top, nk, ce, cs, row * p.ff, row * p.ffs);
  // (MJ 8: what is left over may take a round of its own)
  const unsigned grid = (unsigned)(tiles_of(p.T, p.E, top, 32 * mj, ce, cs) + (mj == 8 ? tile::CUS : 0));
  switch (mj) {
    case 2: expert_kernel<T, MODE, 2, ACT><<<grid, 256, 0, st>>>(p); break;
    case 4: expert_kernel<T, MODE, 4, ACT><<<grid, 256, 0, st>>>(p); break;
    default: expert_kernel<T, MODE, 8, ACT><<<grid, 256, 0, st>>>(p);
  }
  return hipGetLastError();
}

}  // namespace

extern "C" {

// T rows, width W, E experts of ff of which a row chooses at most `top`, a shared one of ffs (or 0)
int sm_expert_ok(int dt, int T, int W, int E, int top, int ff, int ffs) {
  return sizes_ok(dt, T, W, E, top, ff, ffs) && tiles_of(T, E, top, kMinRows, (W + ff) / 64 + 2, (W + ffs) / 64 + 2) < (1 << 30);
}

// wts [T, E] fp32 -> off [E + 1], idx and wt [T top], place [T, top] (a row's pairs in expert order, -1: none)
hipError_t sm_expert_sort(const float* wts, int* off, int* idx, float* wt, int* place, int T, int E, int top,
                          hipStream_t st) {
  if (T < 1 || E < 1 || E > kMaxE || top < 1 || top > E) return hipErrorInvalidValue;
  expert_sort_kernel<<<E, 1024, 0, st>>>(wts, off, idx, wt, place, T, E, top);
  return hipGetLastError();
}

// a [T top, ff] and as [T, ffs] = activations of h [T, W] (row stride ldh) by w [(1 + gated) (E ff + ffs), W]
hipError_t sm_expert_act(int dt, const void* h, long long ldh, const void* w, const int* off, const int* idx,
                         const float* wt, void* a, void* as, int T, int W, int E, int top, int ff, int ffs, int gated,
                         int act, int weigh_in, float limit, float limit_s, float slope, float shift,
                         hipStream_t st) {
  if (!sm_expert_ok(dt, T, W, E, top, ff, ffs) || act < 0 || act > (gated ? 4 : 3) || (weigh_in && !gated) ||
      ldh % 8 || ldh < W || (long long)T * ldh >= (1LL << 31) || 2LL * (ff > ffs ? ff : ffs) * W >= (1LL << 31) ||
      ((uintptr_t)h | (uintptr_t)w | (uintptr_t)a | (uintptr_t)as) % 16)
    return hipErrorInvalidValue;
  const ExpertArgs p{h, h, ldh, ldh, w, W, a, as, off, idx, wt, T, W, E, ff, ffs,
                     GateForm{act, weigh_in, limit, limit_s, slope, shift}};
  const int ct = gated ? BN / 2 : BN;
  const int ce = (ff + ct - 1) / ct, cs = ffs > 0 ? (ffs + ct - 1) / ct : 0;
#define GO(TT)                                                                    \
  if (!gated) return act == 0   ? launch<TT, 1, 0>(p, top, ce, cs, st)            \
                     : act == 1 ? launch<TT, 1, 1>(p, top, ce, cs, st)            \
                     : act == 2 ? launch<TT, 1, 2>(p, top, ce, cs, st)            \
                                : launch<TT, 1, 3>(p, top, ce, cs, st);           \
  return act == 0   ? launch<TT, 0, 0>(p, top, ce, cs, st)                        \
         : act == 1 ? launch<TT, 0, 1>(p, top, ce, cs, st)                        \
         : act == 2 ? launch<TT, 0, 2>(p, top, ce, cs, st)                        \
         : act == 3 ? launch<TT, 0, 3>(p, top, ce, cs, st)                        \
                    : launch<TT, 0, 4>(p, top, ce, cs, st);
  if (dt == kBF16) { GO(bf16) } else { GO(fp16) }
#undef GO
}

// y [T top, W] and ys [T, W] fp32 = a and as by w [W, E ff + ffs]; then out [T, W] their sum per row
hipError_t sm_expert_down(int dt, const void* a, const void* as, const void* w, const int* off, const int* place,
                          float* y, float* ys, void* out, int T, int W, int E, int top, int ff, int ffs,
                          hipStream_t st) {
  const long long ldw = (long long)E * ff + ffs;
  if (!sm_expert_ok(dt, T, W, E, top, ff, ffs) || BN * ldw >= (1LL << 31) || 256LL * ff >= (1LL << 31) ||
      256LL * ffs >= (1LL << 31) || ((uintptr_t)a | (uintptr_t)as | (uintptr_t)w | (uintptr_t)y | (uintptr_t)ys) % 16 ||
      (uintptr_t)out % 8)
    return hipErrorInvalidValue;
  const ExpertArgs p{a, as, ff, ffs, w, ldw, y, ys, off, nullptr, nullptr, T, W, E, ff, ffs, GateForm{}};
  const int c = (W + BN - 1) / BN;
  const dim3 sum((unsigned)T, (unsigned)((W + 1023) / 1024));
#define GO(TT)                                                                                       \
  if (const hipError_t rc = launch<TT, 2, 0>(p, top, c, ffs > 0 ? c : 0, st)) return rc;         \
  expert_sum_kernel<TT><<<sum, 256, 0, st>>>(y, ffs > 0 ? ys : nullptr, place, (TT*)out, top, W);
  if (dt == kBF16) { GO(bf16) } else { GO(fp16) }
#undef GO
  return hipGetLastError();
}

}  // extern "C"
