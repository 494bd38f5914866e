// y = x w^T (+ bias) of 65 - some thousand rows on 256 x (32 NI) tiles (tile_loop.h), where the library's tiles fill the chip
// badly: the caller takes NI 3 - 6 so that one round of workgroups covers the result, and cuts long contractions into S
// slices where even that leaves CUs idle.
//  * XCDs take consecutive (slice, tile) pairs, `group` row tiles by all columns, so an L2 holds few panels;
//  * slices leave fp32 slabs in the order of the lanes' registers (whole-line stores) and a second kernel adds
//    them in slice order: 7 us for 32 MB.
// Measured (bf16, us, library -> here, weights from HBM): S = 1: 4010 x 2048 x 2048 32.4 -> 31.3, x 5632 75 -> 72, 2048 x 4096 x
// 11008 160 -> 143; 4010 x 2112 x 2048 42 -> 34 (NI 5), 4010 x 1536 x 2048 26.9 -> 26.6 (NI 3), 1000 x 11264 x 2048 49 -> 43 (NI 6).
// Sliced: 512 x 4096 x 22016 235 -> 97, x 11008 79 -> 54; 256 x 4096 x 11008 53 -> 39; 1000 x 2048 x 11264 63 -> 51.
// Bound by the power of the products and of the operands' way through LDS (tile_loop.h), and by 5 - 8 us in which all CUs
// write their results at once (4 TB/s).  A form that runs several tiles a workgroup without a gap, stores under the next
// tile's products, was faster for 2.75 and 4 rounds of 256 x 128 tiles (93 -> 80, 124 -> 118) but not for 256 x 256 ones.
#include "tile_loop.h"

namespace lumen {
namespace tile {

struct GemmArgs {
  const void* x; long long ldx;
  const void* w; long long ldw;
  void* y; long long ldy;
  const void* bias;
  float* ws;
  int M, N, K, tiles_m, tiles_n, group, S, wide;         // wide: y's rows can be written 16 bytes at a time
};

template <typename T>
__device__ __forceinline__ void add_bias(f32x4& c, const T* b) {
  const uint2 r = *reinterpret_cast<const uint2*>(b);
  const T* e = reinterpret_cast<const T*>(&r);
#pragma unroll
  for (int k = 0; k < 4; ++k) c[k] += to_f32(e[k]);
}

// the results of fragments i and i + 1 (or of i alone, the last of an odd number) of row m, columns n ..
template <typename T, int NI>
__device__ __forceinline__ void put(const GemmArgs& a, int m, int n, int i, f32x4 u, f32x4 v) {
  const bool pair = i + 1 < NI;
  T* p = (T*)a.y + (long long)m * a.ldy + n;
  if (n >= a.N) return;
  const bool more = pair && n + 4 < a.N;
  if (a.bias != nullptr) {
    add_bias(u, (const T*)a.bias + n);
    if (more) add_bias(v, (const T*)a.bias + n + 4);
  }
  const uint2 lo = make_uint2(pk2<T>(u[0], u[1]), pk2<T>(u[2], u[3])), hi = make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
  if (more && a.wide) {
    *reinterpret_cast<uint4*>(p) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    return;
  }
  *reinterpret_cast<uint2*>(p) = lo;
  if (more) *reinterpret_cast<uint2*>(p + 4) = hi;
}

template <typename T, int NI>
__global__ void __launch_bounds__(256, 1) tile_gemm_kernel(const GemmArgs a) {
  constexpr int BN = Shape<NI>::BN, PIECES = Shape<NI>::PIECES;
  __shared__ __attribute__((aligned(16))) char lds[Shape<NI>::LDS];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = a.tiles_m * a.tiles_n, v = unit_of(blockIdx.x, gridDim.x);
  const int slice = v / tiles, tile = v - slice * tiles;
  int tm, tn;
  tile_at(tile, a.tiles_m, a.tiles_n, a.group, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int steps = a.K / BK;
  const int k0 = steps * slice / a.S, nk = steps * (slice + 1) / a.S - k0;       // (steps * S < 2^31)
  const char* xb = (const char*)a.x + ((long long)m0 * a.ldx + (long long)k0 * BK) * 2;
  const char* wb = (const char*)a.w + ((long long)n0 * a.ldw + (long long)k0 * BK) * 2;
  unsigned off[PIECES];                                  // (rows past the edge read the last row: never stored)
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int r = 8 * (wid + 4 * (q < 8 ? q : q - 8)) + (lane >> 3), c = (lane & 7) ^ swz(r);
    const int col = r / (16 * NI) * (16 * NI) + colperm<NI>(r % (16 * NI));
    off[q] = q < 8 ? (unsigned)min(r, a.M - m0 - 1) * (unsigned)(2 * a.ldx) + 16 * c
                   : (unsigned)min(col, a.N - n0 - 1) * (unsigned)(2 * a.ldw) + 16 * c;
  }
  f32x4 acc[NI][MJ];
  products<T, NI>(lds, xb, wb, nk, off, acc);
  if (a.S > 1) {
    f32x4* o = (f32x4*)a.ws + (((long long)slice * tiles + tile) * 4 + wid) * (NI * MJ * 64) + lane;
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i) hold(acc[i][j]), o[(j * NI + i) * 64] = acc[i][j];
    return;
  }
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const int m = m0 + 128 * (wid >> 1) + 16 * j + lr;
#pragma unroll
    for (int i = 0; i < NI; i += 2) {
      constexpr int last = NI - 1;
      hold(acc[i][j]);
      if (i + 1 < NI) hold(acc[i + 1][j]);
      if (m < a.M)
        put<T, NI>(a, m, n0 + 16 * (NI * (wid & 1) + i) + (i + 1 < NI ? 8 : 4) * lg, i, acc[i][j], acc[i + 1 < NI ? i + 1 : last][j]);
    }
  }
}

// y = the sum of the S slabs, which lie in the order of the lanes that wrote them; a wave sums a pair of fragments
template <typename T, int NI>
__global__ void __launch_bounds__(256) tile_sum_kernel(const GemmArgs a) {
  constexpr int NP = (NI + 1) / 2;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6);     // (tile, wave, j, pair)
  const int i = 2 * (f % NP), j = f / NP % MJ, wid = f / (NP * MJ) % 4, tile = f / (NP * MJ * 4);
  int tm, tn;
  tile_at(tile, a.tiles_m, a.tiles_n, a.group, tm, tn);
  const int m = tm * BM + 128 * (wid >> 1) + 16 * j + lr;
  if (m >= a.M) return;
  const bool pair = i + 1 < NI;
  const f32x4* p = (const f32x4*)a.ws + ((long long)(tile * 4 + wid) * (NI * MJ) + j * NI + i) * 64 + lane;
  const long long plane = (long long)a.tiles_m * a.tiles_n * 4 * NI * MJ * 64;
  f32x4 s = p[0], r = pair ? p[64] : s;
  for (int k = 1; k < a.S; ++k) {
    s += p[k * plane];
    if (pair) r += p[k * plane + 64];
  }
  put<T, NI>(a, m, tn * Shape<NI>::BN + 16 * (NI * (wid & 1) + i) + (pair ? 8 : 4) * lg, i, s, r);
}

}  // namespace tile
}  // namespace lumen

extern "C" {

// y [M, N] = x [M, K] w [N, K]^T + bias [N] (or null), 16-bit, rows at ldx, ldw, ldy, on 256 x 32 ni tiles, K in S slices; ws (S
// > 1): S * tiles * 8192 ni fp32.  K % 64 == 0, N % 4 == 0, rows of x and w at 16-byte addresses, of y and bias at 8-byte ones.
hipError_t lumen_tile_gemm(int dt, const void* x, long long ldx, const void* w, long long ldw, const void* bias, void* y,
                           long long ldy, float* ws, int M, int N, int K, int S, int ni, hipStream_t st) {
  using namespace lumen;
  using namespace lumen::tile;
  if ((long long)M * N == 0) return hipSuccess;
  if (K <= 0 || K % BK || N % 4 || S < 1 || S > K / BK || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K ||
      ldw < K || ldy < N || ldx > (1 << 22) || ldw > (1 << 22) || (S > 1 && !ws) || (dt != kF16 && dt != kBF16) ||
      ((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) % 16 || ((uintptr_t)y | (uintptr_t)bias) % 8 || ni < 3 || ni > 6 ||
      (S > 1 && ni != 4) || (long long)(K / BK) * S >= (1LL << 31))
    return hipErrorInvalidValue;
  const long long tm = (M + BM - 1) / BM, tn = (N + 32 * ni - 1) / (32 * ni), tiles = tm * tn;
  if (tiles * S >= (1 << 20)) return hipErrorInvalidValue;
  const GemmArgs a{x, ldx, w, ldw, y, ldy, bias, ws, M, N, K, (int)tm, (int)tn, (int)(tm < 4 ? tm : 4), S,
                   ldy % 8 == 0 && (uintptr_t)y % 16 == 0};
#define GO(NI)                                                                                            \
  if (dt == kBF16) tile_gemm_kernel<bf16, NI><<<(int)tiles * S, 256, 0, st>>>(a);                         \
  else tile_gemm_kernel<fp16, NI><<<(int)tiles * S, 256, 0, st>>>(a);
  if (ni == 3) { GO(3) } else if (ni == 4) { GO(4) } else if (ni == 5) { GO(5) } else { GO(6) }
#undef GO
  if (S > 1) {
    const int blocks = (int)tiles * 2 * MJ;              // NI 4: two pairs, MJ rows, four waves a tile, four to a block
    if (dt == kBF16) tile_sum_kernel<bf16, 4><<<blocks, 256, 0, st>>>(a);
    else tile_sum_kernel<fp16, 4><<<blocks, 256, 0, st>>>(a);
  }
  return hipGetLastError();
}

}  // extern "C"
