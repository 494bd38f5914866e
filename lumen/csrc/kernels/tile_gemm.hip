// y = x w^T (+ bias) of 17 - some thousand rows on 32 mj x 32 ni tiles (tile_loop.h), where the library's tiles fill the chip
// badly: the caller takes mj 2, 4 or 8 by the rows and ni so that one round of workgroups covers the result, and cuts long
// contractions into S slices where even that leaves CUs idle.
//  * XCDs take consecutive (slice, tile) pairs, `group` row tiles by all columns, so an L2 holds few panels;
//  * slices leave fp32 slabs in the order of the lanes' registers (whole-line stores) and a second kernel adds
//    them in slice order: 7 us for 32 MB;
//  * `turned`: column tiles start their walk of k at different stages, for rows of w that meet in the same memory channels.
// Measured (bf16, us, library or thin kernel -> here, weights from HBM): 256-row tiles, S = 1: 4010 x 2048 x 2048 32.4 -> 31.3, x 5632
// 75 -> 72, 2048 x 4096 x 11008 160 -> 143; 4010 x 2112 x 2048 42 -> 34 (ni 5), 4010 x 1536 x 2048 26.9 -> 26.6 (ni 3), 1000 x 11264 x 2048
// 49 -> 43 (ni 6).  Sliced: 512 x 4096 x 22016 235 -> 97, x 11008 79 -> 54.  Few rows: 64 x 32000 x 4096 61 -> 48.5 (5.4 TB/s of weights),
// 100 x 22016 x 4096 49 -> 41, 256 x 8192 x 4096 42.5 -> 31.9; sliced 64 x 2048 x 11264 32.7 -> 19.5, 128 x 4096 x 11008 39 -> 29.  A decode
// step of 4 layers of width 4096 at 48 rows 651 -> 550, at 112 rows 805 -> 725.  The lines are in ops/gemm.py.
// From some hundred rows on bound by the power of the products and of the operands' way through LDS (tile_loop.h), and by 5 - 8 us in
// which all CUs write their results at once (4 TB/s); below by w's way from HBM.  A form that runs several tiles a
// workgroup without a gap, stores under the next tile's products, was faster for 2.75 and 4 rounds of 256 x 128 tiles (93 -> 80, 124
// -> 118) but not for 256 x 256 ones.
#include "tile_loop.h"

namespace lumen {
namespace tile {

struct GemmArgs {
  const void* x; long long ldx;
  const void* w; long long ldw;
  void* y; long long ldy;
  const void* bias;
  float* ws;
  int M, N, K, tiles_m, tiles_n, group, S;
  int wide, turned;          // y's rows can be written 16 bytes at a time; column tiles start at different k
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

template <typename T, int NI, int MJ, bool APART>
__global__ void __launch_bounds__(256, 1) tile_gemm_kernel(const GemmArgs a) {
  using S = Shape<NI, MJ>;
  constexpr int BM = S::BM, BN = S::BN, PIECES = S::PIECES;
  __shared__ __attribute__((aligned(16))) char lds[S::LDS];
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
    const int r = 8 * (wid + 4 * (q < MJ ? q : q - MJ)) + (lane >> 3), c = (lane & 7) ^ swz(r);
    const int col = r / (16 * NI) * (16 * NI) + colperm<NI>(r % (16 * NI));
    off[q] = q < MJ ? (unsigned)min(r, a.M - m0 - 1) * (unsigned)(2 * a.ldx) + 16 * c
                   : (unsigned)min(col, a.N - n0 - 1) * (unsigned)(2 * a.ldw) + 16 * c;
  }
  f32x4 acc[NI][MJ];
  products<T, NI, MJ, APART>(lds, xb, wb, nk, APART && a.turned ? (int)(13u * tn % nk) : 0, off, acc);
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
    const int m = m0 + 16 * MJ * (wid >> 1) + 16 * j + lr;
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
template <typename T, int NI, int MJ>
__global__ void __launch_bounds__(256) tile_sum_kernel(const GemmArgs a) {
  using S = Shape<NI, MJ>;
  constexpr int NP = (NI + 1) / 2;
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6);     // (tile, wave, j, pair)
  const int i = 2 * (f % NP), j = f / NP % MJ, wid = f / (NP * MJ) % 4, tile = f / (NP * MJ * 4);
  int tm, tn;
  tile_at(tile, a.tiles_m, a.tiles_n, a.group, tm, tn);
  const int m = tm * S::BM + 16 * MJ * (wid >> 1) + 16 * j + lr;
  if (m >= a.M) return;
  const bool pair = i + 1 < NI;
  const f32x4* p = (const f32x4*)a.ws + ((long long)(tile * 4 + wid) * (NI * MJ) + j * NI + i) * 64 + lane;
  const long long plane = (long long)a.tiles_m * a.tiles_n * 4 * NI * MJ * 64;
  f32x4 s = p[0], r = pair ? p[64] : s;
  for (int k = 1; k < a.S; ++k) {
    s += p[k * plane];
    if (pair) r += p[k * plane + 64];
  }
  put<T, NI>(a, m, tn * S::BN + 16 * (NI * (wid & 1) + i) + (pair ? 8 : 4) * lg, i, s, r);
}

}  // namespace tile
}  // namespace lumen

extern "C" {

// y [M, N] = x [M, K] w [N, K]^T + bias [N] (or null), 16-bit, rows at ldx, ldw, ldy, on 32 mj x 32 ni tiles, K in S slices; ws (S
// > 1): S * tiles * 1024 mj ni fp32; turned: column tiles start at different k.  K % 64 == 0, N % 4 == 0, rows of x and w at 16-byte addresses, of y and bias at 8-byte ones.
hipError_t lumen_tile_gemm(int dt, const void* x, long long ldx, const void* w, long long ldw, const void* bias, void* y,
                           long long ldy, float* ws, int M, int N, int K, int S, int ni, int mj, int turned, hipStream_t st) {
  using namespace lumen;
  using namespace lumen::tile;
  if ((long long)M * N == 0) return hipSuccess;
  if (K <= 0 || K % BK || N % 4 || S < 1 || S > K / BK || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K ||
      ldw < K || ldy < N || ldx > (1 << 22) || ldw > (1 << 22) || (S > 1 && !ws) || (dt != kF16 && dt != kBF16) ||
      ((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) % 16 || ((uintptr_t)y | (uintptr_t)bias) % 8 ||
      (S > 1 && (ni != 4 || (mj != 2 && mj != 4 && mj != 8))) || (long long)(K / BK) * S >= (1LL << 31))
    return hipErrorInvalidValue;
  const int BM = 32 * mj;
  const long long tm = (M + BM - 1LL) / BM, tn = (N + 32 * ni - 1) / (32 * ni), tiles = tm * tn;
  if (tiles * S >= (1 << 20)) return hipErrorInvalidValue;
  const GemmArgs a{x, ldx, w, ldw, y, ldy, bias, ws, M, N, K, (int)tm, (int)tn, (int)(tm < 4 ? tm : 4), S,
                   ldy % 8 == 0 && (uintptr_t)y % 16 == 0, turned};
  const int grid = (int)tiles * S;
  // (256 rows in step without the walk's arithmetic: 4010 x 2048 x 5632 78.3 -> 76.5 us)
  switch (10 * mj + ni + (mj == 8 && turned ? 100 : 0)) {
#define GO(MJ, NI, APART)                                                                                       \
  case 10 * MJ + NI + (MJ == 8 && APART ? 100 : 0):                                                             \
    if (dt == kBF16) tile_gemm_kernel<bf16, NI, MJ, APART><<<grid, 256, 0, st>>>(a);                            \
    else tile_gemm_kernel<fp16, NI, MJ, APART><<<grid, 256, 0, st>>>(a);                                        \
    break;
    GO(2, 1, true) GO(2, 2, true) GO(2, 3, true) GO(2, 4, true) GO(2, 5, true) GO(2, 6, true) GO(2, 8, true)
    GO(4, 2, true) GO(4, 3, true) GO(4, 4, true) GO(4, 5, true) GO(4, 6, true) GO(4, 8, true)
    GO(8, 3, false) GO(8, 4, false) GO(8, 5, false) GO(8, 6, false) GO(8, 3, true) GO(8, 4, true)
#undef GO
    default: return hipErrorInvalidValue;
  }
  if (S > 1) {
    const int blocks = (int)tiles * 2 * mj;              // NI 4: two pairs, mj rows' fragments, four waves a tile, four to a block
#define GO(MJ)                                                                    \
  case MJ:                                                                        \
    if (dt == kBF16) tile_sum_kernel<bf16, 4, MJ><<<blocks, 256, 0, st>>>(a);     \
    else tile_sum_kernel<fp16, 4, MJ><<<blocks, 256, 0, st>>>(a);                 \
    break;
    switch (mj) { GO(2) GO(4) GO(8) }
#undef GO
  }
  return hipGetLastError();
}

}  // extern "C"
