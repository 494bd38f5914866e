// Routed experts over the rows that chose them (prompt steps): for every row t with weights r[t, e] (dense, zero off
// the chosen experts), out[t] = sum_e W_down,e act(W_gate,e h_t, W_up,e h_t; r[t, e]) (+ the shared expert's).
//   sm_expert_sort    the (row, expert) pairs in expert order, rows ascending: one workgroup per expert
//   sm_expert_act     first projection and activation of all pairs and of the shared expert
//   sm_expert_down    second projection, fp32 results per pair
//   sm_expert_sum     out[t] = the sum of the row's pairs in expert order and of its shared result, rounded once
//
// The dense form (two library products over ALL experts, ops/moe.py) does E / top times the work; the library's
// grouped product runs at 300 TFLOP/s.  Here a workgroup takes 128 pairs of one expert and 256 rows of its weights,
// both products on a loop like that of kernels/tile_loop.h (three LDS stages of 64 k by LDS-DMA under counted waits, one
// barrier a step, four waves of 64 pairs x 128 weight rows):
//  * the rows of a tile are gathered by the DMA's source addresses; no sorted copy of h exists;
//  * a wave's 128 weight rows of the first product are 64 gate rows and their 64 up rows, so the activation with the
//    routing weight is formed from the fp32 sums and the [pairs, 2 ff] intermediate is never stored;
//  * counts stay on the device: the grid is sized for the most tiles the step can have and the surplus leaves at once.
//    Nothing synchronises, nothing depends on host-visible counts (a capture may hold it);
//  * XCDs take consecutive tiles, an expert's row tiles within a weight panel first: a panel comes from HBM once.
// Bound by the loop at one wave per SIMD (1.0 us a step where kernels/tile_loop.h takes 0.7: an expert's pairs are
// fetched again for every few panels) and by each tile's own prologue and epilogue; under ~200 rows by reading the
// weights once.  Measured (us, a whole layer of experts, dense form -> here; bf16, width 2048, experts of 1408, weights that
// the last-level cache holds; ops/moe.py has few rows with weights from HBM): 8 experts, top 2, and a shared one: 4096 rows
// 534 -> 283, 512 90 -> 60, 256 62 -> 56; 16, top 3, shared: 4096 1130 -> 371, 512 166 -> 99, 64 149 -> 79; 16 ungated,
// top 4: 4096 810 -> 298, 8192 at width 4096 2721 (grouped library product) -> 1685.  Error against float64 2.3e-3 where the dense form has 3.5e-3: nothing is rounded between the
// products and the activation, nor before the sum.
#include "mma.h"

using namespace lumen;

namespace {

constexpr int BM = 128, BN = 256, BK = 64, ROWB = 128;   // pairs, weight rows; a stage row is 64 elements
constexpr int NI = 8, MJ = 4;                            // fragments of a wave: 128 weight rows x 64 pairs
constexpr int XB = BM * ROWB, STAGE = (BM + BN) * ROWB;  // [pairs | weights]
constexpr int XP = BM / 32, PIECES = (BM + BN) / 32;     // 1-KiB LDS-DMA pieces of a wave and stage (x's first)
constexpr int kMaxE = 64;

__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

__device__ __forceinline__ void done_reading() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

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

// activation results of pair fragment j: columns of a lane's accumulators (acc[i]: gate, acc[NI / 2 + i]: up)
template <typename T, int MODE, int ACT>
__device__ __forceinline__ void put_row(const GateForm& f, const f32x4 (&acc)[NI][MJ], int j, T* o, int c0, int ff,
                                        int wn, int lg, float w, bool shared) {
  constexpr int NO = MODE == 0 ? NI / 2 : NI;
  const int col0 = c0 + (MODE == 0 ? 64 : 128) * wn + 4 * lg;
  const float wi = f.weigh_in ? w : 1.f, wo = f.weigh_in ? 1.f : w, lim = shared ? f.limit_s : f.limit;
  const auto act = [&](float g) {
    if constexpr (ACT == 0) return g * sigmoid_fast(g);
    else return gate_act(g, ACT);
  };
#pragma unroll
  for (int i = 0; i < NO; ++i) {
    if (col0 + 16 * i >= ff) continue;
    float r[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float g = acc[i][j][q] * wi;
      if constexpr (MODE == 1) {
        r[q] = act(g) * wo;
      } else {
        float u = acc[(NI / 2 + i) % NI][j][q] * wi;
        if constexpr (ACT == 4) {
          g = fminf(g, lim);
          u = fminf(fmaxf(u, -lim), lim);
          r[q] = g * sigmoid_fast(f.slope * g) * (u + f.shift) * wo;
        } else {
          r[q] = act(g) * u * wo;
        }
      }
    }
    *reinterpret_cast<uint2*>(o + col0 + 16 * i) = make_uint2(pk2<T>(r[0], r[1]), pk2<T>(r[2], r[3]));
  }
}

// MODE 0: gate and up rows -> activation, 1: up rows alone -> activation, 2: second projection -> fp32
template <typename T, int MODE>
__global__ void __launch_bounds__(256, 1) expert_kernel(const ExpertArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[3 * STAGE];
  constexpr int CT = MODE == 0 ? BN / 2 : BN;            // result columns of a tile
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
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
  const int total = tiles_e + ts * cs;
  if ((int)blockIdx.x >= total) return;
  const int xcd = blockIdx.x & 7, q8 = total >> 3, r8 = total & 7;
  const int v = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + ((int)blockIdx.x >> 3);
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
  const bool shared = e == a.E;
  const int ff = shared ? a.ffs : a.ff;
  const int tn = u / nt, m0 = (u - tn * nt) * BM, c0 = tn * CT;
  const int nk = MODE == 2 ? (ff + BK - 1) / BK : a.W / BK, N = MODE == 2 ? a.W : ff;
  // a contraction of 32 more: the last stage reads its first half twice and multiplies it once
  const bool odd = MODE == 2 && ff % BK != 0;
  const T* x = (const T*)(shared ? a.xs : a.x);
  const long long ldx = shared ? a.ldxs : a.ldx;
  const bool gather = MODE != 2 && !shared;
  const char* xb = (const char*)(x + (gather ? 0 : (long long)(r0 + m0) * ldx));
  // weights: MODE 0 / 1 row blocks per expert, MODE 2 column blocks
  const char* wb = (const char*)((const T*)a.w + (MODE == 2 ? (long long)c0 * a.ldw + (long long)e * a.ff
                                                            : (long long)e * (MODE == 0 ? 2 : 1) * a.ff * a.ldw));
  unsigned off[PIECES];
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int p = wid + 4 * q, r = 8 * (q < XP ? p : p - BM / 8) + (lane >> 3);
    const int c = (lane & 7) ^ swz(r);
    if (q < XP) {
      const int i = min(r, rows - m0 - 1);
      off[q] = (unsigned)(gather ? a.idx[r0 + m0 + i] : i) * (unsigned)(2 * ldx) + 16 * c;
    } else if (MODE == 0) {                              // [64 gate | 64 up] rows of each wave column
      const int col = min(c0 + 64 * (r >> 7) + (r & 63), ff - 1);
      off[q] = (unsigned)(col + (r & 64 ? ff : 0)) * (unsigned)(2 * a.ldw) + 16 * c;
    } else if (MODE == 1) {
      off[q] = (unsigned)min(c0 + r, ff - 1) * (unsigned)(2 * a.ldw) + 16 * c;
    } else {
      off[q] = (unsigned)min(r, N - c0 - 1) * (unsigned)(2 * a.ldw) + 16 * c;
    }
  }
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds);
  const unsigned upper = ((lane >> 2) ^ wid) & 1 ? BK : 0;     // (bytes) the lane's chunk lies in the upper half
  auto issue = [&](int t, int slot, int q0, int q1) __attribute__((always_inline)) {
    const unsigned back = odd && t == nk - 1 ? upper : 0;
    const char *xs = xb + (long long)t * (BK * 2), *wsrc = wb + (long long)t * (BK * 2);
    const unsigned dst = __builtin_amdgcn_readfirstlane(lds0 + slot * STAGE + wid * 1024);
#pragma unroll
    for (int q = q0; q < q1; ++q) dma16(q < XP ? xs : wsrc, MODE == 2 ? off[q] - back : off[q], dst + q * 4096);
  };
  f32x4 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint4 fa[2][NI], fb[2][MJ];
  const int rb0 = (64 * wm + lr) * ROWB, ra0 = XB + (128 * wn + lr) * ROWB;
  // fragments u0 .. u1 - 1 of half h of a stage (x's, then w's)
  auto frags = [&](int h, int slot, int u0, int u1) __attribute__((always_inline)) {
    const char* p = lds + slot * STAGE + (((4 * h + lg) ^ swz(lr)) << 4);
#pragma unroll
    for (int i = u0; i < u1; ++i)
      if (i < MJ) fb[h][i] = *reinterpret_cast<const uint4*>(p + rb0 + i * 16 * ROWB);
      else fa[h][i - MJ] = *reinterpret_cast<const uint4*>(p + ra0 + (i - MJ) * 16 * ROWB);
  };
  // the products of half h; between them the reads of the other half's fragments (from stage slot fs) and
  // half of the pieces of stage `t` into slot `ds` (t < 0: none)
  auto half = [&](int h, int fs, int t, int ds) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (2 * i < NI + MJ) frags(1 - h, fs, 2 * i, 2 * i + 2);
      if (t >= 0 && i < PIECES / 2) issue(t, ds, (1 - h) * (PIECES / 2) + i, (1 - h) * (PIECES / 2) + i + 1);
#pragma unroll
      for (int j = 0; j < MJ; ++j) acc[i][j] = Mfma<T>::run(fa[h][i], fb[h][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  issue(0, 0, 0, PIECES);
  if (nk > 1) issue(1, 1, 0, PIECES);
  if (nk > 2) issue(2, 2, 0, PIECES / 2);
  if (nk > 2) wait_vm<PIECES + PIECES / 2>(); else if (nk > 1) wait_vm<PIECES>(); else wait_vm<0>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  frags(0, 0, 0, NI + MJ);
  int slot = 0, t = 0;
  for (; t + 3 < nk; ++t) {
    const int next = slot == 2 ? 0 : slot + 1, last = slot == 0 ? 2 : slot - 1;
    half(0, slot, t + 2, last);
    wait_vm<PIECES>();
    done_reading();
    half(1, next, t + 3, slot);
    slot = next;
  }
  for (; t < nk; ++t) {       // the last three stages
    const int next = slot == 2 ? 0 : slot + 1, last = slot == 0 ? 2 : slot - 1;
    half(0, slot, t + 2 < nk ? t + 2 : -1, last);
    if (t + 2 < nk) wait_vm<PIECES>(); else wait_vm<0>();
    done_reading();
    if (!odd || t + 1 < nk) half(1, next, -1, 0);     // (the last step reads a slot that holds an earlier stage: unused)
    slot = next;
  }
  // lane (lr, lg) holds pair 16 j + lr, weight rows 16 i + 4 lg .. + 3 of its wave's block
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int m = m0 + 64 * wm + 16 * j + lr;
    if (m >= rows) continue;
    if constexpr (MODE == 2) {
      float* o = (float*)(shared ? a.ys : a.y) + (long long)(r0 + m) * a.W + c0 + 128 * wn + 4 * lg;
#pragma unroll
      for (int i = 0; i < NI; ++i)
        if (c0 + 128 * wn + 16 * i + 4 * lg < N) *reinterpret_cast<f32x4*>(o + 16 * i) = acc[i][j];
    } else {
      const float wt = shared ? 1.f : a.wt[r0 + m];
      T* o = (T*)(shared ? a.ys : a.y) + (long long)(r0 + m) * ff;
      // (one branch per row: with the choice inside the element the epilogue was 14000 instructions long, and
      // fetching them took as long as half of the products)
      switch (a.form.act) {
        case 0: put_row<T, MODE, 0>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared); break;
        case 1: put_row<T, MODE, 1>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared); break;
        case 2: put_row<T, MODE, 2>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared); break;
        case 3: put_row<T, MODE, 3>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared); break;
        default: put_row<T, MODE, 4>(a.form, acc, j, o, c0, ff, wn, lg, wt, shared);
      }
    }
  }
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
long long tiles_of(int T, int E, int top, long long ce, long long cs) {
  return ((long long)T * top / BM + E) * ce + (long long)((T + BM - 1) / BM) * cs;
}

}  // namespace

extern "C" {

// T rows, width W, E experts of ff of which a row chooses at most `top`, a shared one of ffs (or 0)
int sm_expert_ok(int dt, int T, int W, int E, int top, int ff, int ffs) {
  return sizes_ok(dt, T, W, E, top, ff, ffs) && tiles_of(T, E, top, (W + ff) / 64 + 2, (W + ffs) / 64 + 2) < (1 << 30);
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
      ((uintptr_t)h | (uintptr_t)w) % 16 || ((uintptr_t)a | (uintptr_t)as) % 8)
    return hipErrorInvalidValue;
  const ExpertArgs p{h, h, ldh, ldh, w, W, a, as, off, idx, wt, T, W, E, ff, ffs,
                     GateForm{act, weigh_in, limit, limit_s, slope, shift}};
  const int ct = gated ? BN / 2 : BN;
  const unsigned grid = (unsigned)tiles_of(T, E, top, (ff + ct - 1) / ct, ffs > 0 ? (ffs + ct - 1) / ct : 0);
#define GO(TT)                                                          \
  if (gated) expert_kernel<TT, 0><<<grid, 256, 0, st>>>(p);             \
  else expert_kernel<TT, 1><<<grid, 256, 0, st>>>(p);
  if (dt == kBF16) { GO(bf16) } else { GO(fp16) }
#undef GO
  return hipGetLastError();
}

// y [T top, W] and ys [T, W] fp32 = a and as by w [W, E ff + ffs]; then out [T, W] their sum per row
hipError_t sm_expert_down(int dt, const void* a, const void* as, const void* w, const int* off, const int* place,
                          float* y, float* ys, void* out, int T, int W, int E, int top, int ff, int ffs,
                          hipStream_t st) {
  const long long ldw = (long long)E * ff + ffs;
  if (!sm_expert_ok(dt, T, W, E, top, ff, ffs) || BN * ldw >= (1LL << 31) || (long long)BM * ff >= (1LL << 31) ||
      (long long)BM * ffs >= (1LL << 31) || ((uintptr_t)a | (uintptr_t)as | (uintptr_t)w | (uintptr_t)y | (uintptr_t)ys) % 16 ||
      (uintptr_t)out % 8)
    return hipErrorInvalidValue;
  const ExpertArgs p{a, as, ff, ffs, w, ldw, y, ys, off, nullptr, nullptr, T, W, E, ff, ffs, GateForm{}};
  const long long c = (W + BN - 1) / BN;
  const unsigned grid = (unsigned)tiles_of(T, E, top, c, ffs > 0 ? c : 0);
  const dim3 sum((unsigned)T, (unsigned)((W + 1023) / 1024));
#define GO(TT)                                                                                       \
  expert_kernel<TT, 2><<<grid, 256, 0, st>>>(p);                                                     \
  expert_sum_kernel<TT><<<sum, 256, 0, st>>>(y, ffs > 0 ? ys : nullptr, place, (TT*)out, top, W);
  if (dt == kBF16) { GO(bf16) } else { GO(fp16) }
#undef GO
  return hipGetLastError();
}

}  // extern "C"
