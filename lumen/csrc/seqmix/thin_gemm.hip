// Few-row projections: y[M, N] = x[M, K] @ W[N, K]^T (+ bias), 1 <= M <= 64 -- a decode step's GEMMs
// and a prompt step's output head.
//
// What bounds it: the one pass over W from HBM, and for matrices of a few MB the latency of that pass
// -- 6 TB/s x ~1.5 us means that ~9 MB have to be in flight, i.e. all of a 2048 x 2048 weight at once.
// Library tiles at these M run one k loop per 16 - 64 columns with too few loads in flight (2048 x
// 2048: 8.3 us for 8.4 MB).  Here
//  * a workgroup's NW waves split K and every wave streams its share of a tile of RT x 16 weight rows
//    through a ring of its own in LDS, D stages of 64 k deep, filled by LDS-DMA (whole 128-byte lines
//    of 8 rows per instruction; a direct fragment load reads 64-byte pieces of 16 rows and reached
//    2.3 - 3.4 TB/s).  No barrier in the k loop: a wave waits for its own stages with a counted vmcnt;
//  * the ring runs on across the tiles of a persistent workgroup, so the loads of the next tile are in
//    flight while this one is summed;
//  * the product is formed transposed (W rows: A operand, x rows: B operand of v_mfma_f32_16x16x32),
//    the waves' partial tiles meet in LDS in wave order (deterministic), a lane holds four consecutive
//    columns of a row: 8-byte stores, fp32 results 16-byte ones.
// x rows past M re-read the last one; image rows that a piece does not hold are read modulo the piece
// (those columns of the product are never stored).
//
// Measured on MI355X, weights rotated through > 600 MB, in a graph, us per call, against the library
// (F.linear) and for M = 1 the rows-per-lane GEMV of kernels/skinny_gemm.hip:
//   M = 8:  2048 x 2048 3.9 / 8.4, 11264 x 2048 10.1 / 16.3, 2048 x 5632 8.3 / 11.6, 32000 x 2048 23.8 /
//           33.2, 4096 x 4096 7.8 / 12.9, 22528 x 4096 31.5 / 51.9 (5.9 TB/s), 4096 x 11264 17.5 / 20.7
//   M = 32: 4.8 / 8.6, 12.5 / 16.3, 12.4 / 15.6, 25.5 / 27.4, 9.5 / 12.7, 37.8 / 42.9, 24.7 / 27.3
//   M = 64: 6.5 / 9.0, 15.3 / 17.6, 17.4 / 18.4, 29.4 / 27.9, 13.3 / 14.3, 52.0 / 45.1, 33.9 / 34.9
//   M = 1:  3.8 / 8.3 (GEMV 4.4), 9.8 / 16.1 (10.5), 7.3 / 11.7 (6.6), 22.4 / 32.0 (22.9), 7.5 / 12.1
//           (8.1), 30.7 / 51.6 (28.5), 17.2 / 20.6 (17.2)
// From 33 rows on every tile re-reads more x than W, so the widest matrices stay with the library
// there; at M = 1 the GEMV stays ahead on long rows (ops/gemm.py has the rule).
#include "seqmix.h"

using namespace lumen;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

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

constexpr int BK = 64, ROWB = 128;   // k per stage, bytes of an image row

// 16-byte chunk c of image row r lives at chunk c ^ swz(r): a fragment read (16 rows at one chunk)
// touches 16 different bank slots
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// LDS-DMA of 16 bytes per lane (wave-uniform base + 32-bit lane offset) as inline asm, so that the
// compiler does not drain the ring before the next fragment read; the counted waits below order it
__device__ __forceinline__ void dma16(const void* base, unsigned off, const char* lds_wave_base) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(lds_wave_base))));
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(m0) : "memory", "m0");
}

struct ThinArgs {
  const void *x, *W, *bias;
  void* y;
  int M, N, K;
  long long ldx, ldy;
  int tiles;       // ceil(N / (16 RT))
  int out32;       // fp32 result
};

// XP: pieces of 8 x rows (1, 2, 4, 8: M <= 8, 16, 32, 64)
template <typename T, int RT, int XP, int NW, int D>
__global__ void __launch_bounds__(64 * NW, 1) thin_kernel(const ThinArgs p) {
  constexpr int MT = XP < 2 ? 1 : XP / 2;
  constexpr int WB = RT * 16 * ROWB, SB = WB + XP * 8 * ROWB;
  constexpr int G = 2 * RT + XP;                   // DMA instructions of a stage
  constexpr int PB = RT * MT * 1024;               // a wave's partial tile
  static_assert(G * (D - 1) < 64, "stages in flight");
  static_assert(NW * D * SB + 2 * NW * PB <= 163840, "LDS");
  __shared__ __attribute__((aligned(16))) char lds[NW * D * SB + 2 * NW * PB];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* ring = lds + wid * D * SB;
  char* part = lds + NW * D * SB;                  // [2][NW][PB]: this tile's and the last one's
  const T* x = (const T*)p.x;
  const T* W = (const T*)p.W;
  const int kt = p.K / BK;
  const int k0 = kt * wid / NW, nk = kt * (wid + 1) / NW - k0;
  const int mine = (p.tiles - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = mine * nk;                     // stages this wave streams
  const int rr = lane >> 3, c = lane & 7;          // row within a piece, LDS chunk
  int at_t = blockIdx.x, at_k = 0, issued = 0, put = 0;
  const auto issue = [&]() {
    char* img = ring + put * SB;
    const int kk = (k0 + at_k) * BK;
    const T* Wt = W + (long long)at_t * (RT * 16) * p.K;
    const int last = min(RT * 16, p.N - at_t * RT * 16) - 1;
#pragma unroll
    for (int q = 0; q < 2 * RT; ++q) {
      const int r = 8 * q + rr;
      dma16(Wt, ((unsigned)min(r, last) * (unsigned)p.K + kk + 8 * (c ^ swz(r))) * 2u,
            img + 8 * q * ROWB);
    }
#pragma unroll
    for (int q = 0; q < XP; ++q) {
      const int r = 8 * q + rr;
      dma16(x, ((unsigned)min(r, p.M - 1) * (unsigned)p.ldx + kk + 8 * (c ^ swz(r))) * 2u,
            img + WB + 8 * q * ROWB);
    }
    put = put + 1 == D ? 0 : put + 1;
    ++issued;
    if (++at_k == nk) { at_k = 0; at_t += gridDim.x; }
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (issued < total) issue();
  const int lr = lane & 15, lg = lane >> 4;
  int get = 0, done = 0, buf = 0;
  for (int t = blockIdx.x; t < p.tiles; t += gridDim.x) {
    f32x4 acc[RT][MT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < nk; ++k) {
      // stage `done` has landed (the tile's stores may add to the count: that only waits longer);
      // the fragments of the stage before it have been read, so its slot may be filled again
      if (total - done >= D - 1) wait_vm<G * (D - 2)>(); else wait_vm<0>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (issued < total) issue();
      const char* img = ring + get * SB;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        uint4 a[RT], b[MT];
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          const int r = 16 * i + lr;
          a[i] = *reinterpret_cast<const uint4*>(img + r * ROWB + (((4 * s + lg) ^ swz(r)) << 4));
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const int r = (16 * j + lr) & (8 * XP - 1);
          b[j] = *reinterpret_cast<const uint4*>(img + WB + r * ROWB +
                                                 (((4 * s + lg) ^ swz(r)) << 4));
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[i][j] = Mfma<T>::run(a[i], b[j], acc[i][j]);
      }
      get = get + 1 == D ? 0 : get + 1;
      ++done;
    }
    char* pb = part + buf * NW * PB;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        *reinterpret_cast<f32x4*>(pb + wid * PB + (i * MT + j) * 1024 + lane * 16) = acc[i][j];
    // one barrier per tile: the partial tiles alternate between two buffers, and a wave writes a
    // buffer again only after the barrier of the tile between
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    for (int q = wid; q < RT * MT; q += NW) {
      const int i = q / MT, j = q - i * MT;
      f32x4 v = *reinterpret_cast<const f32x4*>(pb + q * 1024 + lane * 16);
#pragma unroll
      for (int w = 1; w < NW; ++w)
        v += *reinterpret_cast<const f32x4*>(pb + w * PB + q * 1024 + lane * 16);
      const int m = 16 * j + lr, n = t * RT * 16 + 16 * i + 4 * lg;
      if (m >= p.M || n >= p.N) continue;
      if (p.bias != nullptr) {
        const T* b = (const T*)p.bias + n;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += to_f32(b[e]);
      }
      if (p.out32)
        *reinterpret_cast<f32x4*>((float*)p.y + (long long)m * p.ldy + n) = v;
      else
        *reinterpret_cast<uint2*>((T*)p.y + (long long)m * p.ldy + n) =
            make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
    }
    buf ^= 1;
  }
}

template <typename T, int RT, int XP, int NW, int D>
hipError_t run(ThinArgs p, int per_cu, hipStream_t st) {
  p.tiles = (p.N + 16 * RT - 1) / (16 * RT);
  const int grid = p.tiles < 256 * per_cu ? p.tiles : 256 * per_cu;
  thin_kernel<T, RT, XP, NW, D><<<grid, 64 * NW, 0, st>>>(p);
  return hipGetLastError();
}

// The tile.  One 16-row tile per step of four waves (two workgroups share a CU) is best or within 3 %
// everywhere at M <= 16, except that long rows of a matrix with few tiles want eight waves (2048 x
// 5632: 8.3 vs 8.4 - 9 us) and the widest long-row matrices want 32-row tiles (22528 x 4096: 31.5 vs
// 32.8 us, x read half as often).  Above 16 rows x costs as much as W: many tiles take 64 rows per x
// fragment (11264 x 2048 at M = 64: 15.3 vs 18.7 us with 32), few tiles need the waves on K instead
// (2048 x 2048: 6.5 us with 16-row tiles of four waves).
template <typename T>
hipError_t pick(const ThinArgs& p, hipStream_t st) {
  const bool wide = p.N >= 8192;
  if (p.M <= 8) {
    if (wide && p.K >= 4096) return run<T, 2, 1, 4, 4>(p, 1, st);
    if (!wide && p.K >= 4608) return run<T, 1, 1, 8, 4>(p, 2, st);
    return run<T, 1, 1, 4, 4>(p, 2, st);
  }
  if (p.M <= 16) {
    if (wide && p.K >= 4096) return run<T, 2, 2, 4, 4>(p, 1, st);
    return run<T, 1, 2, 4, 4>(p, 2, st);
  }
  if (p.M <= 32) {
    if (wide && p.K >= 4096) return run<T, 2, 4, 4, 3>(p, 1, st);
    if (wide) return run<T, 4, 4, 2, 3>(p, 1, st);
    return run<T, 1, 4, 4, 3>(p, 2, st);
  }
  if (wide) return run<T, 4, 8, 2, 3>(p, 1, st);
  return run<T, 1, 8, 4, 3>(p, 1, st);
}

}  // namespace

extern "C" {

// M <= 64, K % 64 == 0, N % 4 == 0; W contiguous, x rows at stride ldx (% 8), y rows at stride ldy
// (% 4); x, W and y aligned to 16 bytes.  bias [N] in the operands' dtype, or null.
hipError_t sm_thin_gemm(int dt, const void* x, long long ldx, const void* W, const void* bias,
                        void* y, long long ldy, int M, int N, int K, int out32, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  if (M < 0 || M > 64 || N < 4 || N % 4 || K < BK || K % BK || ldx < K || ldx % 8 || ldy < N ||
      ldy % 4 ||
      ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W) |
        reinterpret_cast<uintptr_t>(y)) & 15) != 0)
    return hipErrorInvalidValue;
  // lane offsets are 32-bit byte offsets from a tile's first row and from x
  if (64LL * K * 2 >= (1LL << 32) || 64LL * ldx * 2 >= (1LL << 32)) return hipErrorInvalidValue;
  const ThinArgs p{x, W, bias, y, M, N, K, ldx, ldy, 0, out32};
  if (dt == kBF16) return pick<bf16>(p, st);
  if (dt == kF16) return pick<fp16>(p, st);
  return hipErrorInvalidValue;
}

}  // extern "C"
