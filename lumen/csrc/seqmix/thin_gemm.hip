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
//   M = 32: 4.8 / 8.6, 12.5 / 16.3, 10.3 / 15.6, 25.5 / 27.4, 9.5 / 12.7, 37.8 / 42.9, 24.7 / 27.3
//   M = 64: 6.1 / 9.0, 15.3 / 17.6, 12.0 / 18.4, 29.4 / 27.9, 13.3 / 14.3, 52.0 / 45.1, 33.9 / 34.9
//   M = 1:  3.8 / 8.3 (GEMV 4.4), 9.8 / 16.1 (10.5), 7.3 / 11.7 (6.6), 22.4 / 32.0 (22.9), 7.5 / 12.1
//           (8.1), 30.7 / 51.6 (28.5), 17.2 / 20.6 (17.2)
// (16-column tiles throughout; matrices of up to 2048 rows now take tiles of eight, see pick)
// The activation form (thin_act): a workgroup's tile is 16 (or 8) activation columns -- their gate rows and
// their up rows -- so act(gate) * up, times the row's routing weight, is formed from the fp32 sums and
// the [M, 2 ff] intermediate and its kernel are gone.  Routed experts: W holds every expert, and a
// step of a few rows uses few of them.  `sparse` reads the routing weights first and streams the
// weights of experts some row chose only -- in the first projection by tile, in the second (K runs
// over [experts x ff]) by k stage; what an unchosen expert would add is zero.
// Measured like the above, a whole feed-forward against two library GEMMs and the activation kernel:
//   dense 2048 -> 5632 (gated): 1 row 18.3 / 28.8 us, 8 rows 22.8 / 31.8, 32 rows 27.9 / 35.8
//   16 experts of 1408, top 3, and a shared one: 1 row 17.5 / 113.9, 8 rows 49.3 / 122.3, 32 rows 88.2 /
//   144.6; width 4096, experts of 2816: 8 rows 189.4 / 269.6, 32 rows 248.4 / 406.8
// The gated form (thin_gate) multiplies gelu(sum) with a row of a per-token table: a launch of 4 us less per layer; thin_tail
// turns a projection's last columns (tanh) or copies them into a cache, likewise.
// From 33 rows on every tile re-reads more x than W, so the widest matrices stay with the library
// there; at M = 1 the GEMV stays ahead on long rows (ops/gemm.py has the rule).
#include "mma.h"

using namespace lumen;

namespace {

constexpr int BK = 64, ROWB = 128;   // k per stage, bytes of an image row
constexpr int kCUs = 256;

// 16-byte chunk c of image row r lives at chunk c ^ swz(r): a fragment read (16 rows at one chunk)
// touches 16 different bank slots
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

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
  int tiles;       // plain: ceil(N / (16 RT))
  int out32;       // fp32 result
  // routed experts: weights [M, E] fp32, blocks of ff columns and a last one of ffs (E = 0: just it)
  const float* wts;
  int E, ff, ffs;
  int sparse;      // skip experts that no row chose
  GateForm form;
  // plain form (or null): y = gelu_tanh(x W^T) * table[token of the row], columns alike
  const void* table; long long ldt; const long long* tokens;
  // plain form: tanh of the columns from tanh_from on; the columns from cache_from on once more, as rounded, to row
  // slots[m] (>= 0) of a cache
  int tanh_from; void* cache; long long ldc; int cache_from; const long long* slots;
};

constexpr int kNoTanh = 0x7fffffff;
constexpr int kMaxWts = 2048;     // routing weights held in LDS (M * E)

// the i-th set bit of a mask
__device__ __forceinline__ int nth_bit(unsigned long long m, int i) {
  for (; i > 0; --i) m &= m - 1;
  return __builtin_ctzll(m);
}

// XP: pieces of 8 x rows (1, 2, 4, 8: groups of up to 8, 16, 32, 64 rows, blockIdx.y names the group).  ACT: 0 plain, 1 activation
// (no gate), 2 gated.  RT: row tiles of W of a product; WP: pieces of 8 W rows, 2 RT or fewer: plain 1 of an RT of 1 (the product's upper
// half repeats the lower one, never stored); gated half of them gate and half up rows (WP 2: the two halves of one row tile).
template <typename T, int RT, int XP, int NW, int D, int ACT, int WP>
__global__ void __launch_bounds__(64 * NW, 1) thin_kernel(const ThinArgs p) {
  constexpr int MT = XP < 2 ? 1 : XP / 2;
  constexpr int WB = WP * 8 * ROWB, SB = WB + XP * 8 * ROWB;
  constexpr int G = WP + XP;                       // DMA instructions of a stage
  constexpr int TC = ACT == 2 ? 4 * WP : 8 * WP;   // result columns of a tile
  constexpr int PB = RT * MT * 1024;               // a wave's partial tile
  constexpr int WTS = XP <= 4 ? kMaxWts * 4 : 0;
  static_assert(G * (D - 1) < 64, "stages in flight");
  static_assert(WP == 2 * RT || (RT == 1 && WP == 1 && ACT == 0) || (RT == 1 && WP == 2 && ACT == 2), "pieces of a tile");
  static_assert(NW * D * SB + 2 * NW * PB + WTS <= 163840, "LDS");
  __shared__ __attribute__((aligned(16))) char lds[NW * D * SB + 2 * NW * PB + WTS];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* ring = lds + wid * D * SB;
  char* part = lds + NW * D * SB;                  // [2][NW][PB]: this tile's and the last one's
  float* wts = reinterpret_cast<float*>(part + 2 * NW * PB);
  const int m0 = blockIdx.y * (8 * XP), M = min(p.M - m0, 8 * XP);       // this workgroup's rows
  const T* x = (const T*)p.x + (long long)m0 * p.ldx;
  const T* W = (const T*)p.W;

  // experts some row chose (every one of them unless `sparse`)
  unsigned long long chosen = 0;
  int n_chosen = 0;
  if (WTS > 0 && p.E > 0) {
    if (p.wts != nullptr) {
      for (int i = threadIdx.x; i < M * p.E; i += 64 * NW) wts[i] = p.wts[m0 * p.E + i];
      __syncthreads();
    }
    if (p.sparse) {
      bool on = false;
      if (lane < p.E)
        for (int m = 0; m < M; ++m) on |= !(wts[m * p.E + lane] == 0.f);
      chosen = __ballot(on);
      n_chosen = __popcll(chosen);
    }
  }
  int tiles = p.tiles, kt = p.K / BK;
  const int per = p.ff / TC, ks = p.ff >> 6;       // tiles / k stages of an expert
  if (p.sparse) {
    if (ACT) tiles = n_chosen * per + p.ffs / TC;
    else kt = n_chosen * ks + (p.ffs >> 6);
  }
  const int k0 = kt * wid / NW, nk = kt * (wid + 1) / NW - k0;
  // The groups of a tile's rows on one XCD (workgroups are dealt out over eight, one after the other), so that its W comes from HBM once:
  // where the tiles are no multiple of eight the later groups start some tiles on (64 rows in two groups: 7040 x 2048 12.2 -> 11.3 us, 3104 x 4096 10.2 -> 8.5)
  int bx = blockIdx.x;
  if (blockIdx.y > 0 && gridDim.x >= 8) {
    bx += gridDim.x * blockIdx.y & 7;
    if (bx >= (int)gridDim.x) bx -= gridDim.x;
  }
  const int mine = max(0, (tiles - bx + (int)gridDim.x - 1) / (int)gridDim.x);
  const int total = mine * nk;                     // stages this wave streams
  const int rr = lane >> 3, c = lane & 7;          // row within a piece, LDS chunk
  // expert (E: the last block) and column of activation tile t
  const auto block_of = [&](int t, int& e, int& col) {
    const int i = per > 0 ? t / per : 0;
    const int n = p.sparse ? n_chosen : p.E;
    if (p.E > 0 && i < n) {
      e = p.sparse ? nth_bit(chosen, i) : i;
      col = (t - i * per) * TC;
    } else {
      e = p.E;
      col = (t - n * per) * TC;
    }
  };
  int at_t = bx, at_k = 0, issued = 0, put = 0;
  int left = 0, seg = 0, kk = 0;                   // sparse second projection: place in the k walk
  const auto seek = [&]() {                        // to this wave's first stage
    if (ACT || !p.sparse) { kk = k0 * BK; return; }
    seg = ks > 0 ? min(k0 / ks, n_chosen) : 0;
    const int in = k0 - seg * ks;
    left = seg < n_chosen ? ks - in : 0x7fffffff;
    kk = (seg < n_chosen ? nth_bit(chosen, seg) : p.E) * p.ff + in * BK;
  };
  const T *Wa = W, *Wb = W;                        // first row of the tile's (gate | up) rows
  int last = 0;
  const auto seat = [&]() {
    if constexpr (ACT == 0) {
      Wa = W + (long long)at_t * TC * p.K;
      last = min(TC, p.N - at_t * TC) - 1;
    } else {
      int e, col;
      block_of(at_t, e, col);
      Wa = W + ((long long)e * ACT * p.ff + col) * p.K;
      Wb = Wa + (long long)(e < p.E ? p.ff : p.ffs) * p.K;
      last = 8 * WP - 1;
    }
  };
  seek();
  if (total > 0) seat();
  const auto issue = [&]() {
    char* img = ring + put * SB;
#pragma unroll
    for (int q = 0; q < WP; ++q) {
      const int r = 8 * q + rr;
      const T* base = ACT == 2 && q >= WP / 2 ? Wb : Wa;
      const int row = ACT == 2 && q >= WP / 2 ? r - 4 * WP : min(r, last);
      dma16(base, ((unsigned)row * (unsigned)p.K + kk + 8 * (c ^ swz(r))) * 2u, img + 8 * q * ROWB);
    }
#pragma unroll
    for (int q = 0; q < XP; ++q) {
      const int r = 8 * q + rr;
      dma16(x, ((unsigned)min(r, M - 1) * (unsigned)p.ldx + kk + 8 * (c ^ swz(r))) * 2u,
            img + WB + 8 * q * ROWB);
    }
    put = put + 1 == D ? 0 : put + 1;
    ++issued;
    if (++at_k == nk) {
      at_k = 0;
      at_t += gridDim.x;
      seek();
      if (issued < total) seat();
    } else {
      kk += BK;
      if (ACT == 0 && p.sparse && --left == 0) {
        ++seg;
        left = seg < n_chosen ? ks : 0x7fffffff;
        kk = (seg < n_chosen ? nth_bit(chosen, seg) : p.E) * p.ff;
      }
    }
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d)
    if (issued < total) issue();
  const int lr = lane & 15, lg = lane >> 4;
  int get = 0, done = 0, buf = 0;
  for (int t = bx; t < tiles; t += gridDim.x) {
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
          const int r = (16 * i + lr) & (8 * WP - 1);
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
    const auto sum = [&](int q) {
      f32x4 v = *reinterpret_cast<const f32x4*>(pb + q * 1024 + lane * 16);
#pragma unroll
      for (int w = 1; w < NW; ++w)
        v += *reinterpret_cast<const f32x4*>(pb + w * PB + q * 1024 + lane * 16);
      return v;
    };
    if constexpr (ACT == 0) {
      for (int q = wid; q < RT * MT; q += NW) {
        const int i = q / MT, j = q - i * MT;
        f32x4 v = sum(q);
        const int m = m0 + 16 * j + lr, n = t * TC + 16 * i + 4 * lg;
        if (m >= p.M || 16 * j + lr >= M || n >= p.N || 4 * lg >= TC) continue;
        if (p.bias != nullptr) {
          const T* b = (const T*)p.bias + n;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += to_f32(b[e]);
        }
        if (p.table != nullptr) {
          const T* e4 = (const T*)p.table + p.tokens[m] * p.ldt + n;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f(v[e]) * to_f32(e4[e]);
        }
        if (n + 3 >= p.tanh_from) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e >= p.tanh_from) v[e] = tanhf(v[e]);
        }
        if (p.cache != nullptr && n >= p.cache_from) {
          const long long sl = p.slots[m];
          if (sl >= 0)
            *reinterpret_cast<uint2*>((T*)p.cache + sl * p.ldc + (n - p.cache_from)) =
                make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
        }
        if (p.out32)
          *reinterpret_cast<f32x4*>((float*)p.y + (long long)m * p.ldy + n) = v;
        else
          *reinterpret_cast<uint2*>((T*)p.y + (long long)m * p.ldy + n) =
              make_uint2(pk2<T>(v[0], v[1]), pk2<T>(v[2], v[3]));
      }
    } else {
      int e, col;
      block_of(t, e, col);
      for (int j = wid; j < MT; j += NW) {
        const int m = 16 * j + lr;
        f32x4 g = sum(j), u = f32x4{1.f, 1.f, 1.f, 1.f};
        if constexpr (ACT == 2 && RT == 1) {       // up rows in the lanes of the tile's upper half
#pragma unroll
          for (int i = 0; i < 4; ++i) u[i] = __shfl(g[i], (lane + 32) & 63, 64);
        } else if constexpr (ACT == 2) {
          u = sum(MT + j);
        }
        if (m >= M || 4 * lg >= TC) continue;
        const float w = e < p.E ? wts[m * p.E + e] : 1.f;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          o[i] = w == 0.f ? 0.f
                 : ACT == 2 ? gated_f(g[i], u[i], w, e == p.E, p.form)
                            : gate_act(g[i], p.form.act) * w;
        *reinterpret_cast<uint2*>((T*)p.y + (long long)(m0 + m) * p.ldy + e * p.ff + col + 4 * lg) =
            make_uint2(pk2<T>(o[0], o[1]), pk2<T>(o[2], o[3]));
      }
    }
    buf ^= 1;
  }
}

template <typename T, int RT, int XP, int NW, int D, int ACT = 0, int WP = 2 * RT>
hipError_t run(ThinArgs p, int per_cu, hipStream_t st) {
  constexpr int TC = ACT == 2 ? 4 * WP : 8 * WP;
  p.tiles = ACT ? (p.E * p.ff + p.ffs) / TC : (p.N + TC - 1) / TC;
  const dim3 grid(p.tiles < 256 * per_cu ? p.tiles : 256 * per_cu, (p.M + 8 * XP - 1) / (8 * XP));
  thin_kernel<T, RT, XP, NW, D, ACT, WP><<<grid, 64 * NW, 0, st>>>(p);
  return hipGetLastError();
}

// The tile.  One 16-row tile per step of four waves (two workgroups share a CU) is best or within 3 %
// everywhere at M <= 16, except that long rows want eight waves at M <= 8 (one row of 2112 x 5632 8.0 vs 9.6 us, of 4096 x 8192 13.4 vs
// 16.1; 6144 x 5632 would be 14.3 for 15.4) and the widest long-row matrices want 32-row tiles (22528 x 4096: 31.5 vs
// 32.8 us, x read half as often).  Above 16 rows x costs as much as W: many tiles take all rows of x, 64 to an x
// fragment (11264 x 2048 at M = 64: 15.3 vs 18.7 us with 32); where that leaves CUs idle the rows are cut into groups of 32 or
// 16, each with workgroups of its own that hold more of W in flight.  All rows -> groups, us, 64 rows: 128 x 2048 6.1 -> 3.8, 256 x
// 4096 9.5 -> 4.9 (16 and eight waves; of 32 4.7, 6.9), 2048 x 2048 7.8 -> 6.1, 2048 x 5632 17.1 -> 12.0 (32), 3072 x 2048 8.1 -> 7.5
// (32, 32-row tiles; 16-row ones 9.6), 4096 x 4096 14.2 -> 13.8, 6144 x 2048 13.3 -> 11.8 (past 4096 columns two groups are more than a
// round: of k below 1024 or past 7680 columns all rows, 33 - 64 rows of 5504 x 256 4.2 us, 5.1 in groups, 7040 x 512 5.7 and 6.2, 8176 x 1792 1 : 1.04 - 1.08; 5504 x 2048 11.2 and 10.2); 32 rows: 128 x 2048 4.5 -> 3.6, 2048 x 2048
// 6.2 -> 5.1, 2048 x 5632 12.4 -> 10.3 (16: two groups of 2048 columns' tiles are a workgroup a CU; 2112 would go x 512 3.0 -> 3.3, x 1024 4.1
// -> 4.4, x 2048 6.0 -> 6.1, 3072 x 2048 6.5 -> 7.0).  The eight waves of up to 256 columns have use for more than three stages of k for every two
// of them (64 rows of 256 columns, four waves over eight: k 64 - 256 0.88, 320 - 768 0.95, 832 1.02, 1536 1.05).
// Up to 16 rows of a matrix of up to 2048 rows take tiles of eight columns, eight waves and the stages that fit: as many CUs as
// there are (16-column tiles of 2048 leave half of them idle).  us, 16-column tiles -> these, 1 / 8 / 16 rows: 2048 x 2048 4.7 / 5.0 /
// 5.2 -> 4.3 / 4.4 / 4.8, 2048 x 5632 8.2 / 8.5 / 9.9 -> 6.9 / 7.2 / 8.5, 2048 x 12672 12.9 / 15.1 / 18.0 -> 11.0 / 12.2 / 14.8 (8 rows, 4.2 TB/s),
// 1024 x 2816 5.2 / 5.4 / 6.0 -> 4.2 / 4.7 / 5.4, 256 x 4096 5.3 / 6.1 / 7.0 -> 4.5 / 5.0 / 6.0; the chosen of 16 experts of 1408, 2048 rows of W, 8
// rows 25.5 -> 20.1, one row 6.9 -> 6.5.  Short rows have no use for eight waves (2048 x 512 3.1 -> 3.2), larger matrices none for
// half tiles (2112 x 2048, 8 rows 4.9 -> 5.4).
template <typename T>
hipError_t pick(const ThinArgs& p, hipStream_t st) {
  const bool wide = p.N >= 8192;
  if (p.N <= 8 * kCUs && p.K >= 1024 && p.M <= 16)
    return p.M <= 8 ? run<T, 1, 1, 8, 5, 0, 1>(p, 1, st) : run<T, 1, 2, 8, 4, 0, 1>(p, 1, st);
  if (p.M <= 8) {
    if (wide && p.K >= 4096) return run<T, 2, 1, 4, 4>(p, 1, st);
    if (!wide && p.K >= 4608) return run<T, 1, 1, 8, 4>(p, 2, st);
    return run<T, 1, 1, 4, 4>(p, 2, st);
  }
  if (p.M <= 16) {
    if (wide && p.K >= 4096) return run<T, 2, 2, 4, 4>(p, 1, st);
    return run<T, 1, 2, 4, 4>(p, 2, st);
  }
  if (p.N <= 256 && p.E == 0) return p.K > 768 ? run<T, 1, 2, 8, 4>(p, 1, st) : run<T, 1, 2, 4, 4>(p, 2, st);
  if (p.M <= 32) {
    if (wide && p.K >= 4096) return run<T, 2, 4, 4, 3>(p, 1, st);
    if (wide) return run<T, 4, 4, 2, 3>(p, 1, st);
    if (p.N <= 8 * kCUs && p.E == 0) return run<T, 1, 2, 4, 4>(p, 2, st);   // rows in two groups of 16
    return run<T, 1, 4, 4, 3>(p, 2, st);
  }
  if (wide) return run<T, 4, 8, 2, 3>(p, 1, st);
  if (p.N <= 2048) return run<T, 1, 4, 4, 3>(p, 2, st);                  // in groups of 32
  return p.N <= 16 * kCUs || (p.K >= 1024 && p.N <= 30 * kCUs) ? run<T, 2, 4, 4, 3>(p, 1, st) : run<T, 1, 8, 4, 3>(p, 1, st);
}

template <typename T>
hipError_t pick_act(const ThinArgs& p, int gated, hipStream_t st) {
  // Tiles of eight columns, two workgroups a CU, where tiles of 16 are one or two rounds of the CUs and at most half of another
  // (5632 columns of 2048, 1.4 rounds, 8 rows 12.7 -> 11.7 us, 5632 of 4096 21.4 -> 18.9, 10240 of 2048 18.6 -> 17.5; 1.6 rounds would go
  // 13.3 -> 14.6, one whole one 14.4 -> 15.0, 2.75 33.0 -> 34.5, 1.4 of 512 6.5 -> 7.1).  Tiles of experts depend on the choice: 16.
  const int t = p.N / 16, rest = t % kCUs;
  if (gated && p.E == 0 && p.K >= 1024 && p.M <= 16 && t > kCUs && t < 3 * kCUs && rest > 0 && 2 * rest <= kCUs)
    return p.M <= 8 ? run<T, 1, 1, 4, 5, 2, 2>(p, 2, st) : run<T, 1, 2, 4, 4, 2, 2>(p, 2, st);
  if (gated) {
    if (p.M <= 8) return run<T, 2, 1, 4, 4, 2>(p, 1, st);
    if (p.M <= 16) return run<T, 2, 2, 4, 4, 2>(p, 1, st);
    return run<T, 2, 4, 4, 3, 2>(p, 1, st);
  }
  if (p.M <= 8) return run<T, 1, 1, 4, 4, 1>(p, 2, st);
  if (p.M <= 16) return run<T, 1, 2, 4, 4, 1>(p, 2, st);
  return run<T, 1, 4, 4, 3, 1>(p, 1, st);
}

bool aligned(const void* x, const void* W, const void* y) {
  return ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(W) |
           reinterpret_cast<uintptr_t>(y)) & 15) == 0;
}

}  // namespace

extern "C" {

// M <= 64, K % 64 == 0, N % 4 == 0; W contiguous, x rows at stride ldx (% 8), y rows at stride ldy
// (% 4); x, W and y aligned to 16 bytes.  bias [N] in the operands' dtype, or null.  wts (or null):
// K is E blocks of ff and one of ffs (both % 64), and blocks whose column of wts [M, E] is zero add
// nothing and are not read (M <= 32, M * E <= 2048, E <= 64).
hipError_t sm_thin_gemm(int dt, const void* x, long long ldx, const void* W, const void* bias,
                        void* y, long long ldy, int M, int N, int K, int out32, const float* wts,
                        int E, int ff, int ffs, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  if (M < 0 || M > 64 || N < 4 || N % 4 || K < BK || K % BK || ldx < K || ldx % 8 || ldy < N ||
      ldy % 4 || !aligned(x, W, y))
    return hipErrorInvalidValue;
  // lane offsets are 32-bit byte offsets from a tile's first row and from x
  if (64LL * K * 2 >= (1LL << 32) || 64LL * ldx * 2 >= (1LL << 32)) return hipErrorInvalidValue;
  if (wts != nullptr && (M > 32 || E < 1 || E > 64 || M * E > kMaxWts || ff < 64 || ff % 64 ||
                         ffs < 0 || ffs % 64 || (long long)E * ff + ffs != K))
    return hipErrorInvalidValue;
  ThinArgs p{};
  p.tanh_from = kNoTanh;
  p.x = x; p.W = W; p.bias = bias; p.y = y;
  p.M = M; p.N = N; p.K = K; p.ldx = ldx; p.ldy = ldy; p.out32 = out32;
  if (wts != nullptr) { p.wts = wts; p.E = E; p.ff = ff; p.ffs = ffs; p.sparse = 1; }
  if (dt == kBF16) return pick<bf16>(p, st);
  if (dt == kF16) return pick<fp16>(p, st);
  return hipErrorInvalidValue;
}

// y [M, N] = gelu_tanh(x @ W^T) * table[tokens[m]][n], the table's rows at stride ldt; the rest as sm_thin_gemm.
hipError_t sm_thin_gate(int dt, const void* x, long long ldx, const void* W, void* y, int M, int N, int K,
                        const void* table, long long ldt, const long long* tokens, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  if (M < 0 || M > 64 || N < 4 || N % 4 || K < BK || K % BK || ldx < K || ldx % 8 || !aligned(x, W, y) || !table ||
      !tokens || ldt < N || 64LL * K * 2 >= (1LL << 32) || 64LL * ldx * 2 >= (1LL << 32))
    return hipErrorInvalidValue;
  ThinArgs p{};
  p.tanh_from = kNoTanh;
  p.x = x; p.W = W; p.y = y;
  p.M = M; p.N = N; p.K = K; p.ldx = ldx; p.ldy = N;
  p.table = table; p.ldt = ldt; p.tokens = tokens;
  if (dt == kBF16) return pick<bf16>(p, st);
  if (dt == kF16) return pick<fp16>(p, st);
  return hipErrorInvalidValue;
}

// y [M, N] = x @ W^T, the columns from tanh_from on through tanh, those from cache_from on (cache given)
// also to row slots[m] >= 0 of cache, rows at stride ldc.  cache_from, ldc % 4, cache at 8 bytes; the rest as above.
hipError_t sm_thin_tail(int dt, const void* x, long long ldx, const void* W, void* y, int M, int N, int K, int tanh_from,
                        void* cache, long long ldc, int cache_from, const long long* slots, hipStream_t st) {
  if (M == 0 || N == 0) return hipSuccess;
  if (M < 0 || M > 64 || N < 4 || N % 4 || K < BK || K % BK || ldx < K || ldx % 8 || !aligned(x, W, y) ||
      tanh_from < 0 || 64LL * K * 2 >= (1LL << 32) || 64LL * ldx * 2 >= (1LL << 32) ||
      (cache && (!slots || cache_from < 0 || cache_from % 4 || cache_from >= N || ldc % 4 || ldc < N - cache_from ||
                 (uintptr_t)cache % 8)))
    return hipErrorInvalidValue;
  ThinArgs p{};
  p.tanh_from = kNoTanh;
  p.x = x; p.W = W; p.y = y;
  p.M = M; p.N = N; p.K = K; p.ldx = ldx; p.ldy = N;
  p.tanh_from = tanh_from; p.cache = cache; p.ldc = ldc; p.cache_from = cache_from; p.slots = slots;
  if (dt == kBF16) return pick<bf16>(p, st);
  if (dt == kF16) return pick<fp16>(p, st);
  return hipErrorInvalidValue;
}

// y [M, E ff + ffs] = the activation of x @ W^T: W [E (1 + gated) ff + (1 + gated) ffs, K] holds per block
// the gate rows then the up rows (or up rows alone), expert e's block weighed by wts [M, E] (see
// GateForm), the last one not.  ff, ffs % 16; M <= 32, M * E <= 2048, E <= 64; the rest as above.
// sparse: blocks of experts that no row chose are not written (ff, ffs % 64).
hipError_t sm_thin_act(int dt, const void* x, long long ldx, const void* W, const float* wts, void* y,
                       int M, int K, int E, int ff, int ffs, int gated, int sparse, int act,
                       int weigh_in, float limit, float limit_s, float slope, float shift,
                       hipStream_t st) {
  if (M == 0) return hipSuccess;
  const long long out = (long long)E * ff + ffs;
  if (M < 0 || M > 32 || K < BK || K % BK || ldx < K || ldx % 8 || E < 0 || E > 64 || ff < 0 ||
      ff % 16 || ffs < 0 || ffs % 16 || out < 16 || out >= (1LL << 27) || M * E > kMaxWts ||
      (E > 0 && (wts == nullptr || ff < 16)) || (E == 0 && ff != 0) || act < 0 ||
      act > (gated ? 4 : 3) || (weigh_in && !gated) || !aligned(x, W, y))
    return hipErrorInvalidValue;
  if (sparse && (E < 1 || ff % 64 || ffs % 64)) return hipErrorInvalidValue;
  if (64LL * K * 2 >= (1LL << 32) || 64LL * ldx * 2 >= (1LL << 32)) return hipErrorInvalidValue;
  ThinArgs p{};
  p.tanh_from = kNoTanh;
  p.x = x; p.W = W; p.y = y;
  p.M = M; p.N = (int)out; p.K = K; p.ldx = ldx; p.ldy = out;
  p.wts = wts; p.E = E; p.ff = ff; p.ffs = ffs; p.sparse = sparse;
  p.form = GateForm{act, weigh_in, limit, limit_s, slope, shift};
  if (dt == kBF16) return pick_act<bf16>(p, gated, st);
  if (dt == kF16) return pick_act<fp16>(p, gated, st);
  return hipErrorInvalidValue;
}

}  // extern "C"
