// a = act(x Wg^T) * (x Wu^T) of some hundred to some thousand rows, W = [gate ff | up ff rows]: the gated activation in the
// epilogue of the products (kernels/tile_loop.h), from the fp32 sums; the [rows, 2 ff] intermediate is never stored.
//
// Before, the library wrote it (90 MB for 4010 rows x 11264) and a pass of its own read it back.  A wave's 16 NI weight rows
// are alternating fragments of 16 gate rows and their 16 up rows, so a lane holds both of a result; two such pairs give
// it 8 consecutive columns (one 16-byte store).  A launch covers a range of columns: the caller gives whole rounds of
// workgroups to 256 x 256 tiles (NI 8) and the rest to one round of narrower ones.
// Bound by the products (tile_loop.h); the epilogue is half the stores of the plain product and ~3 us of exponentials and divisions a
// tile, as exact as expf's (us, 4010 rows x 5632 x 2048 and 8000: on the bare exponential and reciprocal units 140, 268; with expf and `/`
// 154, 303; here 145, 281).
#include "mma.h"
#include "../kernels/tile_loop.h"

using namespace lumen;

namespace {

constexpr int MJ = 8, BM = 32 * MJ;                      // rows of a tile

struct ActArgs {
  const void* x; long long ldx;
  const void* w;               // [2 ff, K] contiguous
  void* y;                     // [M, ff]
  int M, ff, K, c0, c1, tiles_m, tiles_n, group;         // columns c0 .. c1 - 1 of the result
  GateForm form;
};

// column (of 8 NI) and part (0 gate, 1 up) of row r of a wave's 16 NI
template <int NI>
__device__ __forceinline__ int col_of(int r) {
  const int i = r >> 4, q = i >> 2;
  return 4 * q + 4 <= NI ? 32 * q + 8 * ((r >> 2) & 3) + 4 * ((i >> 1) & 1) + (r & 3) : 32 * q + (r & 15);
}

template <int ACT>
__device__ __forceinline__ float gated(const GateForm& f, float g, float u) {
  if constexpr (ACT == 4) {
    g = fminf(g, f.limit_s);
    u = fminf(fmaxf(u, -f.limit_s), f.limit_s);
    return logistic_gate<true>(g, f.slope * g) * (u + f.shift);
  }
  if constexpr (ACT == 0) return logistic_gate<false>(g, g) * u;
  return gate_act(g, ACT) * u;
}

template <typename T, int NI, int ACT>
__global__ void __launch_bounds__(256, 1) tile_act_kernel(const ActArgs a) {
  using tile::hold;
  using S = tile::Shape<NI, MJ>;
  constexpr int PIECES = S::PIECES, CT = 16 * NI;        // CT: result columns of a tile
  __shared__ __attribute__((aligned(16))) char lds[S::LDS];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  tile::tile_at(tile::unit_of(blockIdx.x, gridDim.x), a.tiles_m, a.tiles_n, a.group, tm, tn);
  const int m0 = tm * BM, n0 = a.c0 + tn * CT;
  unsigned off[PIECES];                                  // (rows past the edge read the last row: never stored)
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int r = 8 * (wid + 4 * (q < MJ ? q : q - MJ)) + (lane >> 3), c = (lane & 7) ^ tile::swz(r);
    const int col = min(n0 + r / (16 * NI) * (8 * NI) + col_of<NI>(r % (16 * NI)), a.c1 - 1);
    off[q] = q < MJ ? (unsigned)min(r, a.M - m0 - 1) * (unsigned)(2 * a.ldx) + 16 * c
                   : (unsigned)(col + ((r >> 4) & 1 ? a.ff : 0)) * (unsigned)(2 * a.K) + 16 * c;
  }
  tile::f32x4 acc[NI][MJ];
  tile::products<T, NI, MJ>(lds, (const char*)a.x + (long long)m0 * a.ldx * 2, (const char*)a.w, a.K / tile::BK, 0, off, acc);
  // lane (lr, lg) holds row 16 j + lr, columns col_of(16 i + 4 lg ..), of gate (i even) and up (i odd)
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int m = m0 + 16 * MJ * (wid >> 1) + 16 * j + lr;
#pragma unroll
    for (int i = 0; i < NI; i += 4) {
      constexpr int last = NI - 1;
      const bool two = i + 4 <= NI;
      const int n = n0 + 8 * NI * (wid & 1) + 8 * i + (two ? 8 : 4) * lg;
      uint2 o[2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
        if (s == 0 || two) {
          tile::f32x4 &g = acc[i + 2 * s < NI ? i + 2 * s : last][j], &u = acc[i + 2 * s + 1 < NI ? i + 2 * s + 1 : last][j];
          hold(g), hold(u);
          float r[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = gated<ACT>(a.form, g[e], u[e]);
          o[s] = make_uint2(pk2<T>(r[0], r[1]), pk2<T>(r[2], r[3]));
        }
      if (m >= a.M || n >= a.c1) continue;
      T* p = (T*)a.y + (long long)m * a.ff + n;          // (c1 and ff are multiples of 8)
      if (two) *reinterpret_cast<uint4*>(p) = make_uint4(o[0].x, o[0].y, o[1].x, o[1].y);
      else *reinterpret_cast<uint2*>(p) = o[0];
    }
  }
}

}  // namespace

extern "C" {

// columns c0 .. c1 - 1 of y [M, ff] = act(x Wg^T) * (x Wu^T), x [M, K] at ldx, w [2 ff, K], act: GateForm's, on 256 x 16 ni tiles.
// K % 64 == 0, ff, c0, c1 % 8 == 0, ni 4, 6 or 8, w under 4 GiB.
hipError_t sm_tile_act(int dt, const void* x, long long ldx, const void* w, void* y, int M, int K, int ff, int c0, int c1,
                       int ni, int act, float limit, float slope, float shift, hipStream_t st) {
  if (M < 1 || K < tile::BK || K % tile::BK || ff < 8 || ff % 8 || c0 < 0 || c0 % 8 || c1 % 8 || c1 <= c0 || c1 > ff ||
      ldx % 8 || ldx < K || ldx > (1 << 22) || 4LL * ff * K >= (1LL << 32) || (dt != kF16 && dt != kBF16) || act < 0 || act > 4 ||
      ((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) % 16 || (ni != 4 && ni != 6 && ni != 8))
    return hipErrorInvalidValue;
  const long long tm = (M + BM - 1LL) / BM, tn = (c1 - c0 + 16 * ni - 1) / (16 * ni);
  if (tm * tn >= (1 << 20)) return hipErrorInvalidValue;
  const ActArgs a{x, ldx, w, y, M, ff, K, c0, c1, (int)tm, (int)tn, (int)(tm < 4 ? tm : 4),
                  GateForm{act, 0, limit, limit, slope, shift}};
#define ACTS(TT, NI)                                                                          \
  switch (act) {                                                                              \
    case 0: tile_act_kernel<TT, NI, 0><<<(int)(tm * tn), 256, 0, st>>>(a); break;             \
    case 1: tile_act_kernel<TT, NI, 1><<<(int)(tm * tn), 256, 0, st>>>(a); break;             \
    case 2: tile_act_kernel<TT, NI, 2><<<(int)(tm * tn), 256, 0, st>>>(a); break;             \
    case 3: tile_act_kernel<TT, NI, 3><<<(int)(tm * tn), 256, 0, st>>>(a); break;             \
    default: tile_act_kernel<TT, NI, 4><<<(int)(tm * tn), 256, 0, st>>>(a);                   \
  }
#define GO(TT) if (ni == 4) { ACTS(TT, 4) } else if (ni == 6) { ACTS(TT, 6) } else { ACTS(TT, 8) }
  if (dt == kBF16) { GO(bf16) } else { GO(fp16) }
#undef GO
#undef ACTS
  return hipGetLastError();
}

}  // extern "C"
