// y = x w^T for long contractions over 65 - 1500 rows (a training step of one short sequence, prompts, the input
// gradients of wide projections): few output tiles, so K is cut into S slices to fill the chip.
//
// What bounded these in the library: one workgroup per CU needs small tiles (64 x 128 at 512 x 4096), and small
// tiles read each operand from L2 often -- 15 TB/s at 0.65 PFLOP/s.  Here a workgroup is a 256 x 128 tile
// of one slice: half the L2 traffic per product.  The XCDs take consecutive (slice, tile) pairs, slice-major, so
// an L2 holds few slices of x and w and every weight comes from HBM once.
//  * four waves of 128 x 64 (acc 128 registers, fragments of both k halves 96): an operand row read from LDS
//    feeds 4 or 8 products, LDS reads take 3/4 of the matrix time;
//  * three LDS stages of 64 k (48 KiB each), filled by LDS-DMA two steps ahead under counted waits; one barrier
//    per step.  The DMA and the other half's fragment reads are dealt out between the products: issued in
//    one go they held the wave's products back (0.81 -> 0.73 us a step);
//  * slices leave fp32 slabs in the order of the lanes' registers (whole-line stores) and a second kernel adds
//    them in slice order: 7 us for 32 MB, and ~12 us of a call are its prologue and the slabs' stores.
// Measured (bf16, us, library -> here): 512 x 4096 x 22016 139 -> 91, x 32000 290 -> 123, x 11008 72 -> 50; 256 x
// 4096 x 11008 51 -> 35; 1000 x 2048 x 11264 72 -> 51.  Bound now by LDS bandwidth and latency: one wave per
// SIMD runs its matrix core at 59 %.
#include "common.h"

namespace lumen {
namespace sg {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
template <typename T> struct Mfma;
template <> struct Mfma<bf16> {
  static __device__ __forceinline__ f32x4 run(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mfma<fp16> {
  static __device__ __forceinline__ f32x4 run(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

constexpr int BM = 256, BN = 128, BK = 64, ROWB = 128;   // a row of a stage is 64 elements, 128 bytes
constexpr int NI = 4, MJ = 8;                            // fragments of a wave: 64 columns x 128 rows
constexpr int XB = BM * ROWB, STAGE = (BM + BN) * ROWB;  // [x rows | w rows]
constexpr int NSTAGE = 3, PIECES = (BM + BN) / 8 / 4;    // 1-KiB LDS-DMA pieces of a wave and stage

struct SplitArgs {
  const void* x; long long ldx;
  const void* w; long long ldw;
  void* y; long long ldy;
  float* ws;
  int M, N, K, tiles_m, tiles, S;
};

// 16-byte chunk c of stage row r lies at chunk c ^ swz(r): a fragment read (16 rows at one chunk) and an
// LDS-DMA piece (8 whole rows) are both conflict free
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

template <typename T>
__device__ __forceinline__ void store4(T* p, const float (&f)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pk2<T>(f[0], f[1]), pk2<T>(f[2], f[3]));
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// LDS-DMA of 16 bytes per lane into the wave's 1-KiB piece (M0: its LDS address).  Inline asm, so that
// the waits of this kernel's own counting order it.
__device__ __forceinline__ void dma16(const void* base, unsigned off, unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

// this wave's fragment reads have arrived, and every wave's: their stage may be overwritten
__device__ __forceinline__ void done_reading() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename T>
__global__ void __launch_bounds__(256, 1) split_gemm_kernel(const SplitArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[NSTAGE * STAGE];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  // block -> (k slice, tile): XCD x (block % 8) gets consecutive ids, slice-major, so the blocks that
  // share an L2 read few slices of x and w, and the row tiles of one w panel follow each other
  const int nb = gridDim.x, xcd = blockIdx.x & 7, q8 = nb >> 3, r8 = nb & 7;
  const int v = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (blockIdx.x >> 3);
  const int slice = v / a.tiles, tile = v - slice * a.tiles;
  const int tn = tile / a.tiles_m, tm = tile - tn * a.tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;
  const int steps = a.K / BK;
  const int k0 = steps * slice / a.S, nk = steps * (slice + 1) / a.S - k0;   // (steps * S < 2^31)
  const char* xb = (const char*)a.x + ((long long)m0 * a.ldx + (long long)k0 * BK) * 2;
  const char* wb = (const char*)a.w + ((long long)n0 * a.ldw + (long long)k0 * BK) * 2;
  // this wave's pieces of a stage: wid, wid + 4, ...; the first BM / 8 are x, the others w.  Rows past the
  // edge read the last row (never stored).
  unsigned off[PIECES];
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int p = wid + 4 * q, r = 8 * (q < BM / 32 ? p : p - BM / 8) + (lane >> 3);
    const int c = (lane & 7) ^ swz(r);
    off[q] = q < BM / 32 ? (unsigned)min(r, a.M - m0 - 1) * (unsigned)(2 * a.ldx) + 16 * c
                         : (unsigned)min(r, a.N - n0 - 1) * (unsigned)(2 * a.ldw) + 16 * c;
  }
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds);
  auto issue = [&](int t, int slot, int q0, int q1) __attribute__((always_inline)) {
    const char *xs = xb + (long long)t * (BK * 2), *wsrc = wb + (long long)t * (BK * 2);
    const unsigned dst = __builtin_amdgcn_readfirstlane(lds0 + slot * STAGE + wid * 1024);
#pragma unroll
    for (int q = q0; q < q1; ++q) dma16(q < BM / 32 ? xs : wsrc, off[q], dst + q * 4096);
  };
  f32x4 acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint4 fa[2][NI], fb[2][MJ];
  const int rb0 = (128 * wm + lr) * ROWB, ra0 = XB + (64 * wn + lr) * ROWB;
  // fragments u0 .. u1 - 1 of half h of a stage (w's, then x's)
  auto frags = [&](int h, int slot, int u0, int u1) __attribute__((always_inline)) {
    const char* p = lds + slot * STAGE + (((4 * h + lg) ^ swz(lr)) << 4);
#pragma unroll
    for (int u = u0; u < u1; ++u)
      if (u < NI) fa[h][u] = *reinterpret_cast<const uint4*>(p + ra0 + u * 16 * ROWB);
      else fb[h][u - NI] = *reinterpret_cast<const uint4*>(p + rb0 + (u - NI) * 16 * ROWB);
  };
  // the products of half h; between them the reads of the other half's fragments (from stage slot fs) and
  // half of the pieces of stage `t` into slot `ds` (t < 0: none)
  auto half = [&](int h, int fs, int t, int ds) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      if (2 * j < NI + MJ) frags(1 - h, fs, 2 * j, 2 * j + 2);
      if (t >= 0 && j < PIECES / 2) issue(t, ds, (1 - h) * (PIECES / 2) + j, (1 - h) * (PIECES / 2) + j + 1);
#pragma unroll
      for (int i = 0; i < NI; ++i) acc[i][j] = Mfma<T>::run(fa[h][i], fb[h][j], acc[i][j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Step t multiplies stage t; at its start the first half's fragments are in registers.  Behind the first
  // half's products it reads the second half's and issues the rest of stage t + 2; then stage t + 1 has to be
  // there, and every wave done with stage t, whose slot takes stage t + 3 behind the second half's products.
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
    half(1, next, -1, 0);     // (the last step reads a slot that holds an earlier stage: unused)
    slot = next;
  }
  // (lane (lr, lg) holds row 16 j + lr, columns 16 i + 4 lg .. + 3 of its wave's block)
  f32x4* o = (f32x4*)a.ws + (((long long)slice * a.tiles + tile) * 4 + wid) * (NI * MJ * 64) + lane;
#pragma unroll
  for (int j = 0; j < MJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) o[(j * NI + i) * 64] = acc[i][j];
}

// y = the sum of the S slabs, which lie in the order of the lanes that wrote them
template <typename T>
__global__ void __launch_bounds__(256) split_sum_kernel(const SplitArgs a) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6);       // (tile, wave, j, i)
  const int i = f % NI, j = f / NI % MJ, wid = f / (NI * MJ) % 4, tile = f / (NI * MJ * 4);
  const int tn = tile / a.tiles_m, tm = tile - tn * a.tiles_m;
  const int m = tm * BM + 128 * (wid >> 1) + 16 * j + lr, n = tn * BN + 64 * (wid & 1) + 16 * i + 4 * lg;
  if (m >= a.M || n >= a.N) return;
  const f32x4* p = (const f32x4*)a.ws + (long long)f * 64 + lane;
  const long long plane = (long long)a.tiles * 4 * NI * MJ * 64;
  f32x4 s = p[0];
  for (int k = 1; k < a.S; ++k) s += p[k * plane];
  float o[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = s[e];
  store4((T*)a.y + (long long)m * a.ldy + n, o);
}

}  // namespace sg
}  // namespace lumen

extern "C" {

// y [M, N] = x [M, K] w [N, K]^T (16-bit, rows at ldx, ldw, ldy), K in S >= 2 slices; ws: S * tiles * 32768
// fp32.  K % 64 == 0, N % 4 == 0, rows of x and w at 16-byte addresses, of y at 8-byte ones.
hipError_t lumen_split_gemm(int dt, const void* x, long long ldx, const void* w, long long ldw, void* y,
                         long long ldy, float* ws, int M, int N, int K, int S, hipStream_t st) {
  using namespace lumen;
  using namespace lumen::sg;
  if ((long long)M * N == 0) return hipSuccess;
  if (K <= 0 || K % BK || N % 4 || S < 2 || S > K / BK || ldx % 8 || ldw % 8 || ldy % 4 || ldx < K ||
      ldw < K || ldy < N || ldx > (1 << 22) || ldw > (1 << 22) || !ws || (dt != kF16 && dt != kBF16) ||
      ((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) % 16 || (uintptr_t)y % 8)
    return hipErrorInvalidValue;
  const long long tm = (M + BM - 1) / BM, tiles = tm * ((N + BN - 1) / BN);
  if (tiles * S >= (1 << 20)) return hipErrorInvalidValue;
  const SplitArgs a{x, ldx, w, ldw, y, ldy, ws, M, N, K, (int)tm, (int)tiles, S};
#define CALL(TT)                                                                     \
  split_gemm_kernel<TT><<<(int)tiles * S, 256, 0, st>>>(a);                          \
  split_sum_kernel<TT><<<(int)tiles * NI * MJ, 256, 0, st>>>(a);
  if (dt == kBF16) { CALL(bf16) } else { CALL(fp16) }
#undef CALL
  return hipGetLastError();
}

}  // extern "C"
