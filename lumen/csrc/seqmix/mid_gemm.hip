// Projections of up to 64 rows, x [M, K] W [N, K]^T: a decode step of a busy server.
//
// What bounds them: thin_gemm.hip gives every wave a ring of its own, and with 64 rows of x beside 16 weight rows four rings
// fill LDS with two stages each -- most of what is in flight is x, read again by every tile.  Here the four waves
// of a workgroup share a ring: 64 rows of x, 64 of W, 128 k a stage, three of four stages in flight (96 KB a CU), a barrier a
// stage; a wave multiplies 16 rows with all 64 columns.
//  * act: a tile's 64 weight rows are 32 gate and 32 up rows, so the activation is formed from the fp32 sums and the
//    [M, 2 ff] intermediate and its launch are gone;
//  * slabs: few tiles leave most CUs idle, so K is cut and every slice stores its fp32 sums; the norm that follows adds
//    them while it reads its rows (sm_slab_rms), so that costs no launch and y is never rounded.
// Measured in a graph, weights rotated through 600 MB, 64 rows (bf16), us, separate launches -> here: product and norm 2048 x
// 5632 21.7 -> 12.4, 2048 x 2048 11.8 -> 9.7, 1024 x 2816 13.1 -> 8.6, 4096 x 11264 40.7 -> 26.7, 3072 x 8448 31.2 -> 19.7 (8 rows:
// 12.3 -> 10.3, 8.6 -> 7.7, 8.4 -> 7.3, 25.8 -> 24.2, 19.1 -> 17.4); gate, up and activation 5632 x 2048 20.3 -> 15.7, 2816 x 1024
// 13.0 -> 8.8; without a gate 5632 x 2048 16.9 -> 13.6, 11264 x 4096 31.3 -> 27.2.  One round of tiles only: a workgroup
// fills a CU's LDS, so 264 tiles (gated 8448 x 3072) take two, 34.9 -> 38.1, and stay with the separate launches.
#include "mma.h"

using namespace lumen;

namespace {

constexpr int BM = 64, BN = 64, BK = 128, ROWB = 2 * BK;     // a row of a stage: 16 chunks of 16 bytes
constexpr int STAGE = (BM + BN) * ROWB, D = 4;               // 32 KiB
constexpr int PIECES = STAGE / 1024 / 4;                     // LDS-DMA instructions of a wave and stage

struct MidArgs {
  const void *x, *W;
  void* y;                    // act: [M][ff] 16-bit; slabs: [S][M][N] fp32
  long long ldx;
  int M, N, K, tiles, S;      // N: rows of W
  int ff;                     // act: result columns (gated: N = 2 ff)
  GateForm form;
};

// ACT: 0 slabs, 1 activation of the 64 columns, 2 gated
template <typename T, int ACT>
__global__ void __launch_bounds__(256, 1) mid_kernel(const MidArgs p) {
  __shared__ __attribute__((aligned(16))) char lds[D * STAGE];
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slice = (int)blockIdx.x / p.tiles, tile = (int)blockIdx.x - slice * p.tiles;
  const int steps = p.K / BK, k0 = steps * slice / p.S, n = steps * (slice + 1) / p.S - k0;
  const char* xb = (const char*)p.x + (long long)k0 * ROWB;
  // this wave's pieces of a stage: wid, wid + 4, ... of 4 rows each; the first half x, the others W.  A chunk c of stage
  // row r lies at c ^ (r & 15): a fragment read (16 rows at one chunk) touches every bank once.
  const int c0 = ACT == 2 ? tile * (BN / 2) : tile * BN;     // first column of the result
  const char* wb = (const char*)p.W + ((long long)c0 * p.K + (long long)k0 * BK) * 2;
  unsigned off[PIECES];
#pragma unroll
  for (int q = 0; q < PIECES; ++q) {
    const int piece = wid + 4 * q, r = 4 * (piece & 15) + (lane >> 4), c = (lane & 15) ^ (r & 15);
    if (q < PIECES / 2) {
      off[q] = (unsigned)min(r, p.M - 1) * (unsigned)(2 * p.ldx) + 16 * c;
    } else {
      // (a last tile's rows past the end repeat its last one, and are not stored)
      const int row = ACT == 2 ? min(r & 31, p.ff - 1 - c0) + (r < 32 ? 0 : p.ff) : min(r, p.N - 1 - c0);
      off[q] = (unsigned)row * (unsigned)(2 * p.K) + 16 * c;
    }
  }
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds);
  const auto issue = [&](int t) __attribute__((always_inline)) {
    const unsigned dst = __builtin_amdgcn_readfirstlane(lds0 + (t % D) * STAGE + wid * 1024);
    const char *xs = xb + (long long)t * ROWB, *ws = wb + (long long)t * ROWB;
#pragma unroll
    for (int q = 0; q < PIECES; ++q) dma16(q < PIECES / 2 ? xs : ws, off[q], dst + q * 4096);
  };
#pragma unroll
  for (int t = 0; t < D - 1; ++t)
    if (t < n) issue(t);
  f32x4 acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t = 0; t < n; ++t) {
    // stage t has landed (every wave's pieces, after the barrier), and stage t - 1, whose slot is next, has been read
    if (n - t >= D - 1) wait_vm<PIECES * (D - 2)>();
    else if (n - t == 2) wait_vm<PIECES>();
    else wait_vm<0>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + D - 1 < n) issue(t + D - 1);
    const char* st = lds + (t % D) * STAGE;
    const char *xr = st + (16 * wid + lr) * ROWB, *wr = st + (BM + lr) * ROWB;
    uint4 b[BK / 32], a[BK / 32][4];
#pragma unroll
    for (int s = 0; s < BK / 32; ++s) {
      const int at = ((4 * s + lg) ^ lr) << 4;
      b[s] = *reinterpret_cast<const uint4*>(xr + at);
#pragma unroll
      for (int i = 0; i < 4; ++i) a[s][i] = *reinterpret_cast<const uint4*>(wr + 16 * i * ROWB + at);
    }
#pragma unroll
    for (int s = 0; s < BK / 32; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = Mfma<T>::run(a[s][i], b[s], acc[i]);
  }
  const int m = 16 * wid + lr;         // lane (lr, lg): row m, columns 16 i + 4 lg .. of the tile
  if (m >= p.M) return;
  if constexpr (ACT == 0) {
    float* y = (float*)p.y + ((long long)slice * p.M + m) * p.N + c0 + 4 * lg;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c0 + 16 * i + 4 * lg < p.N) *reinterpret_cast<f32x4*>(y + 16 * i) = acc[i];
  } else {
    T* y = (T*)p.y + (long long)m * p.ff + c0 + 4 * lg;
    constexpr int NI = ACT == 2 ? 2 : 4;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (c0 + 16 * i + 4 * lg >= p.ff) continue;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = ACT == 2 ? gated_f(acc[i][e], acc[(i + 2) & 3][e], 1.f, true, p.form) : gate_act(acc[i][e], p.form.act);
      *reinterpret_cast<uint2*>(y + 16 * i) = make_uint2(pk2<T>(o[0], o[1]), pk2<T>(o[2], o[3]));
    }
  }
}

constexpr int kThreads = 512;

// x += the slabs' sum normed in groups, out = x rounded: a row per workgroup, its sums in registers; a wave's 256 columns
// lie in one group.  All parts of a row are asked for together, the norm's weight with them (64 rows of 4096: 8 slabs 4.48 -> 4.23 us,
// 13 slabs 5.71 -> 4.75)
template <typename TO, int N>
__global__ void __launch_bounds__(kThreads)
slab_rms_kernel(const float* __restrict__ y, int S, const float* __restrict__ w, float* __restrict__ x,
                TO* __restrict__ out, int rows, int W, int groups, float eps) {
  __shared__ float s_part[N * kThreads / 64];
  const int r = blockIdx.x, tid = threadIdx.x, gs = W / groups;
  const float* yr = y + (long long)r * W;
  const long long plane = (long long)rows * W;
  float v[N][4], xv[N][4], ww[N][4];             // (the weight with the first loads: it is needed at once after the sums)
  int at[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {                 // (no branch between parts: past the row's end, its first columns again)
    at[i] = 4 * (tid + i * kThreads);
    if (at[i] >= W) at[i] = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[i][e] = xv[i][e] = ww[i][e] = 0.f;
    if (N == 1 && 4 * tid >= W) continue;
    load4<float>(x + (long long)r * W + at[i], xv[i]);
    load4<float>(w + at[i], ww[i]);
    load4<float>(yr + at[i], v[i]);
  }
  int s0 = N == 1 && 4 * tid >= W ? S : 1;
  const auto some = [&](auto count) __attribute__((always_inline)) {      // slabs s0 .. s0 + count - 1, asked for together
    constexpr int B = decltype(count)::value;
    for (; s0 + B <= S; s0 += B) {
      float u[B][N][4];
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < N; ++i) load4<float>(yr + (s0 + b) * plane + at[i], u[b][i]);
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] += u[b][i][e];
    }
  };
  if constexpr (N == 1) some(std::integral_constant<int, 7>());
  some(std::integral_constant<int, 3>());
  some(std::integral_constant<int, 1>());
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += v[i][e] * v[i][e];
    ss = wave_sum(4 * (tid + i * kThreads) < W ? ss : 0.f);
    if ((tid & 63) == 0) s_part[(tid >> 6) + i * (kThreads / 64)] = ss;     // columns 256 x its index on
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = 4 * (tid + i * kThreads);
    if (c >= W) break;
    const int g = c / gs, per = gs >> 8;
    float tot = 0.f;
    for (int k = 0; k < per; ++k) tot += s_part[g * per + k];
    const float inv = 1.f / sqrtf(tot / (float)gs + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) xv[i][e] += v[i][e] * inv * ww[i][e];
    store4<float>(x + (long long)r * W + c, xv[i]);
    if (out) store4<TO>(out + (long long)r * W + c, xv[i]);
  }
}

bool fits(const void* x, long long ldx, const void* W, const void* y, int M, int N, int K) {
  return M >= 1 && M <= BM && N >= 4 && N % 4 == 0 && K >= BK && K % BK == 0 && ldx >= K && ldx % 8 == 0 &&
         64LL * K * 2 < (1LL << 32) && 64LL * ldx * 2 < (1LL << 32) &&
         ((uintptr_t)x | (uintptr_t)W | (uintptr_t)y) % 16 == 0;
}

}  // namespace

extern "C" {

// y [S][M][N] fp32: the sums of x W^T over S slices of K, 1 <= S <= K / 128.  M <= 64, N % 4 == 0, K % 128 == 0; W contiguous,
// x rows at stride ldx (% 8), 16-byte bases.
hipError_t sm_mid_slabs(int dt, const void* x, long long ldx, const void* W, float* y, int M, int N, int K, int S,
                        hipStream_t st) {
  if (!fits(x, ldx, W, y, M, N, K) || S < 1 || S > K / BK || (dt != kBF16 && dt != kF16)) return hipErrorInvalidValue;
  MidArgs p{};
  p.x = x; p.W = W; p.y = y; p.ldx = ldx; p.M = M; p.N = N; p.K = K; p.S = S;
  p.tiles = (N + BN - 1) / BN;
  if (dt == kBF16) mid_kernel<bf16, 0><<<p.tiles * S, 256, 0, st>>>(p);
  else mid_kernel<fp16, 0><<<p.tiles * S, 256, 0, st>>>(p);
  return hipGetLastError();
}

// y [M][ff] = act(x Wg^T) * (x Wu^T), W = [gate ff | up ff rows], or without a gate act(x W^T): GateForm's activations.
// ff % 4; the rest as above; 64 rows of W and 32-bit offsets from a tile's first gate row to its last up row.
hipError_t sm_mid_act(int dt, const void* x, long long ldx, const void* W, void* y, int M, int ff, int K, int gated, int act,
                      float limit, float limit_s, float slope, float shift, hipStream_t st) {
  if (!fits(x, ldx, W, y, M, ff, K) || (dt != kBF16 && dt != kF16) || act < 0 || act > (gated ? 4 : 3) ||
      (gated && (ff + 32LL) * K * 2 >= (1LL << 32)))
    return hipErrorInvalidValue;
  MidArgs p{};
  p.x = x; p.W = W; p.y = y; p.ldx = ldx; p.M = M; p.K = K; p.S = 1; p.ff = ff;
  p.N = gated ? 2 * ff : ff;
  p.tiles = gated ? (ff + BN / 2 - 1) / (BN / 2) : (ff + BN - 1) / BN;
  p.form = GateForm{act, 0, limit, limit_s, slope, shift};
#define GO(T)                                                        \
  if (gated) mid_kernel<T, 2><<<p.tiles, 256, 0, st>>>(p);           \
  else mid_kernel<T, 1><<<p.tiles, 256, 0, st>>>(p)
  if (dt == kBF16) { GO(bf16); } else { GO(fp16); }
#undef GO
  return hipGetLastError();
}

// x [rows][W] fp32 += the RMS norm in `groups` parts of sum_s y[s] (y [S][rows][W] fp32), times w [W]; out (nullable) [rows][W]
// takes the new row in type dt.  W / groups % 256 == 0, W <= 8192, 16-byte bases.
hipError_t sm_slab_rms(int dt, const float* y, int S, const float* w, float* x, void* out, int rows, int W, int groups,
                       float eps, hipStream_t st) {
  if (rows == 0) return hipSuccess;
  if (rows < 0 || S < 1 || groups < 1 || W < 1 || W > 8192 || W % groups || (W / groups) % 256 || !y || !w || !x ||
      ((uintptr_t)y | (uintptr_t)w | (uintptr_t)x | (uintptr_t)out) % 16)
    return hipErrorInvalidValue;
#define GO(T, N) slab_rms_kernel<T, N><<<rows, kThreads, 0, st>>>(y, S, w, x, (T*)out, rows, W, groups, eps)
#define CALL(T)                \
  if (W <= 2048) GO(T, 1);     \
  else if (W <= 4096) GO(T, 2); \
  else GO(T, 4)
  SM_DISPATCH(dt, CALL)
#undef CALL
#undef GO
  return hipGetLastError();
}

}  // extern "C"
