// Attention with mixed heads over a step's prompt portions: what sm_row_attn (row_attention.hip) computes with `talk`
//   s_h(i, j) = (q_h(i) . k_g(j)) * scale * temp(p_i);  s_h <- cap * tanh(s_h / cap);
//   s_h <- s_h - r1_h * log(1 + r2_h * (i - j));        s'_h = sum_h' talk[h, h'] s_h'
//   o_h(i) = sum_{j <= i} exp(s'_h) v_g(j) / (sum_{j <= i} exp(s'_h) + exp(sink_h))
// for 16-bit caches, heads of 128 and up to 32 of them, on the matrix cores.
//
// What bounded the row kernel on prompts: a workgroup was one row, so every row pulled its whole key and value range
// through L2 and formed the mixed scores, H^2 per key, on the vector units.  Here a workgroup of eight waves is 16
// consecutive rows of a segment and ALL heads (the mixing needs them together); per tile of 32 keys
//   1. wave w forms the scores of its HPW heads: S^T = K Q^T (v_mfma_f32_16x16x32, the keys straight from the cache
//      one tile ahead, since a wave's heads share a key head), shaped in registers, fp32 into LDS;
//   2. wave w mixes the heads of its 4 keys: S' = talk S per key with v_mfma_f32_16x16x4_f32 -- the products stay
//      in fp32 -- in place;
//   3. wave w takes the softmax of its heads with lane (row, 8 keys): exactly the operand of O^T += V^T P^T, so
//      the weights feed it from registers, the fp32 ones in three 16-bit parts; the values lie row-major in LDS
//      (LDS-DMA, issued before step 1) and are read transposed (ds_read_b64_tr_b16).
// A hidden key has weight 0, but 0 times an infinite or NaN value is NaN: in the tiles where some row's keys end (a
// workgroup's last one or two) such values are blanked in LDS, and added at the end to the rows that do see them (a
// weight is positive, so the value itself is the result).
// The score of (key, head, row) lies at ((key Hp + (head ^ head/4 ^ key/4 ^ key/16) mod 4 in the low bits) 16 + row):
// all three steps touch four different groups of 16 banks at a time.
// Bound by the chain of tiles at two waves per SIMD (~14000 cycles per 32 keys, a third of it the shaping's
// transcendentals).  Measured against the row kernel (us, bf16, one key head per four heads, everything on): 16 heads,
// 14 prompts of 63 - 509 tokens 515 -> 107, 1 x 512 148 -> 101, 1 x 24 22 -> 15; 8 heads, 1 x 2048 755 -> 275; 32 heads, 8
// of 32 - 256 316 -> 130, 1 x 2048 5248 -> 930.  Few rows behind many keys have short work in a long chain and stay with
// the row kernel (16 heads, 16 rows behind 1024 keys: 31 us there, 198 here).
// Error: the row kernel's.  Share of results that are not float64's rounded, row kernel / here: bf16 0.0003 / 0.0003,
// fp16 0.0022 / 0.0022.  (Two parts and the hardware's exponential, logarithm and reciprocal as they are: 0.0025 and
// 0.0115, at 100 us for the 14 prompts; three parts alone 104; expf, logf and tanhf 117, with the same error.)
#include "mma.h"

using namespace lumen;

namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
constexpr int kD = 128, kRows = 16, kKeys = 32, kTbl = 512;
// fp16: weights up to e^kRise times this fit, and the parts of small ones stay above its subnormals' grain
template <typename T> constexpr float kUp = 1.f;
template <> constexpr float kUp<fp16> = 128.f;

template <typename T> struct TalkArgs {
  const T* q; long long qr, qh;
  const T *kc, *vc;                          // [blocks][bs][G][kD]
  T* out; long long our, ouh;
  const int* tables; int maxb;
  const int *q_tiles, *cu, *start;           // [n][2] (segment, first row); tiles of tile_rows rows
  int n_tiles, subs, tile_rows;
  int H, G, bs;
  float scale, softcap, tcoef; int tevery;
  const float *r1, *r2, *talk, *sink;
};

// image of 32 value rows of 256 bytes: 16-byte chunk c of row r lies at chunk c ^ vswz(r)
__device__ __forceinline__ int vswz(int r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

__device__ __forceinline__ uint2 tr_read(const char* p) {
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

// LDS-DMA of 16 bytes per lane; ordered by the kernel's waits
__device__ __forceinline__ void dma16(const void* src, const char* lds_wave_base) {
  const unsigned m0 = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const char*)(lds_wave_base))));
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(m0) : "memory", "m0");
}

// HPW: heads of a wave (consecutive ones of one key head); MT: 16-head blocks of the mixing
template <typename T, int HPW, int MT>
__global__ void __launch_bounds__(512, 2) talk_tile_kernel(const TalkArgs<T> a) {
  constexpr int Hp = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* s_s = reinterpret_cast<float*>(smem);                         // [kKeys][Hp][16]
  char* s_v = smem + kKeys * Hp * 16 * 4;                              // [G][kKeys][256 bytes]
  int* s_tbl = reinterpret_cast<int*>(s_v + a.G * kKeys * 256);        // [kTbl], then: were values blanked?
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // every tile's last rows first: consecutive workgroups belong to different tiles
  const int sub = a.subs - 1 - blockIdx.x / a.n_tiles, tile = blockIdx.x % a.n_tiles;
  const int seg = a.q_tiles[2 * tile], first = a.q_tiles[2 * tile + 1] + kRows * sub;
  const int end = min(a.cu[seg + 1], a.q_tiles[2 * tile + 1] + a.tile_rows);
  if (first >= end) return;
  const int p0 = a.start[seg] - a.cu[seg];                             // position = row + p0
  const int kend = min(first + kRows, end) - 1 + p0;                   // the workgroup's last key
  const int row = min(first + lr, end - 1), pos = row + p0;
  const int* tbl = a.tables + (long long)seg * a.maxb;
  const int nblk = kend / a.bs + 1;
  const bool in_lds = nblk <= kTbl;
  if (in_lds)
    for (int i = threadIdx.x; i < nblk; i += 512) s_tbl[i] = tbl[i];
  if (threadIdx.x == 0) s_tbl[kTbl] = 0;
  // heads past the last one: scores of zero, never written again
  for (int i = threadIdx.x; i < kKeys * Hp * 4; i += 512)
    reinterpret_cast<f32x4*>(s_s)[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int hw = w * HPW;
  const bool on = hw < a.H;
  const int g = on ? hw / (a.H / a.G) : 0;
  const int bshift = (a.bs & (a.bs - 1)) == 0 ? __ffs(a.bs) - 1 : -1;
  const auto cache_row = [&](int j) -> long long {
    j = min(j, kend);
    const int jb = bshift >= 0 ? j >> bshift : j / a.bs;
    const int blk = in_lds ? s_tbl[jb] : tbl[jb];
    return (long long)blk * a.bs + (j - jb * a.bs);
  };
  float temp = 1.f;
  if (a.tevery > 0 && a.tcoef != 0.f) temp = 1.f + a.tcoef * logf((float)((pos + 1) / a.tevery) + 1.f);
  const float qs = a.scale * temp, cap = a.softcap, rcap = cap > 0.f ? 1.f / cap : 0.f;
  constexpr bool QREG = HPW <= 2;            // queries in registers; else read again for every tile
  const T* qp = a.q + (long long)row * a.qr + 8 * lg;
  uint4 qf[QREG ? HPW : 1][4];
  if constexpr (QREG) {
#pragma unroll
    for (int x = 0; x < HPW; ++x)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        qf[x][k] = *reinterpret_cast<const uint4*>(qp + (long long)min(hw + x, a.H - 1) * a.qh + 32 * k);
  }
  float ta[MT][4 * MT];                      // talk[16 mt + lr][4 c + lg]
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int c = 0; c < 4 * MT; ++c) {
      const int i = 16 * mt + lr, j = 4 * c + lg;
      ta[mt][c] = i < a.H && j < a.H ? a.talk[i * a.H + j] : 0.f;
    }
  float m[HPW], l[HPW];
  f32x4 O[HPW][8];
#pragma unroll
  for (int x = 0; x < HPW; ++x) {
    const bool sk = a.sink != nullptr && hw + x < a.H;
    m[x] = sk ? a.sink[hw + x] : -INFINITY;                            // the sink: a key without a value
    l[x] = sk && lg == 0 ? 1.f : 0.f;                                  // (a lane's share of the sum)
#pragma unroll
    for (int n = 0; n < 8; ++n) O[x][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // score (key, h, row r)
  const auto at = [](int key, int h, int r) {
    return (key * Hp + (h ^ ((h >> 2) & 3) ^ (((key >> 2) ^ (key >> 4)) & 3))) * 16 + r;
  };
  uint4 kf[2][4];                            // keys 16 b + lr, entries 32 k + 8 lg
  const auto load_keys = [&](int j0) __attribute__((always_inline)) {
    long long r[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) r[b] = cache_row(j0 + 16 * b + lr);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        kf[b][k] = *reinterpret_cast<const uint4*>(a.kc + (r[b] * a.G + g) * kD + 32 * k + 8 * lg);
  };
  __syncthreads();
  if (QREG && on) load_keys(0);             // (HPW = 4: no registers to hold the next tile's keys)

  for (int j0 = 0; j0 <= kend; j0 += kKeys) {
    // HPW = 4: the LDS addresses are formed again in every tile (kept over the loop they spill)
    int lo = lane;
    if constexpr (HPW > 2) asm volatile("" : "+v"(lo));
    const int xr = lo & 15, xg = lo >> 4;
    {  // the tile's values: wave w rows 4 w .. 4 w + 3 of every value head
      const int r = 4 * w + (lane >> 4);
      const T* src = a.vc + cache_row(j0 + r) * a.G * kD + 8 * ((lane & 15) ^ vswz(r));
      for (int gv = 0; gv < a.G; ++gv) dma16(src + gv * kD, s_v + (gv * kKeys + 4 * w) * 256);
    }
    // 1. scores of the wave's heads
    if (on) {
      if (!QREG) load_keys(j0);
#pragma unroll
      for (int x = 0; x < HPW; ++x) {
        if (hw + x >= a.H) break;
        if constexpr (HPW > 2) __builtin_amdgcn_sched_barrier(0);
        uint4 qx[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          qx[k] = QREG ? qf[QREG ? x : 0][k]
                       : *reinterpret_cast<const uint4*>(qp + (long long)(hw + x) * a.qh + 32 * k);
        const float r1 = a.r1 != nullptr ? a.r1[hw + x] : 0.f, r2 = a.r1 != nullptr ? a.r2[hw + x] : 0.f;
        f32x4 c[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          c[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < 4; ++k) c[b] = Mfma<T>::run(kf[b][k], qx[k], c[b]);
          c[b] *= qs;
        }
        if (cap > 0.f) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) c[b][i] = cap * tanh_near(c[b][i] * rcap);
        }
        if (a.r1 != nullptr) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) {              // (keys past the row's position are masked below)
              const float d = (float)max(pos - (j0 + 16 * b + 4 * lg + i), 0);
              c[b][i] -= r1 * log_near(1.f + r2 * d);
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) s_s[at(16 * b + 4 * xg + i, hw + x, xr)] = c[b][i];
      }
      if (QREG && j0 + kKeys <= kend) load_keys(j0 + kKeys);
    }
    __syncthreads();
    // 2. the heads of keys 4 w .. 4 w + 3 mixed, in place
#pragma unroll
    for (int y = 0; y < 4; ++y) {
      const int key = 4 * w + y;
      float b[4 * MT];
#pragma unroll
      for (int c = 0; c < 4 * MT; ++c) b[c] = s_s[at(key, 4 * c + xg, xr)];
      f32x4 d[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        d[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4 * MT; ++c) d[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[mt][c], b[c], d[mt], 0, 0, 0);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_s[at(key, 16 * mt + 4 * xg + i, xr)] = d[mt][i];
    }
    // the values have landed for every wave (the next tile's keys, asked for after them, too)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (j0 + kKeys - 1 > first + p0) {                  // some row's keys end here: infinite values of the wave's
      for (int gv = 0; gv < a.G; ++gv) {                // value rows are blanked
        uint4* vp = reinterpret_cast<uint4*>(s_v + (gv * kKeys + 4 * w) * 256 + 16 * lo);
        if (odd8<T>(*vp)) {
          *vp = finite8<T>(*vp);
          s_tbl[kTbl] = 1;
        }
      }
    }
    __syncthreads();
    // 3. softmax and values of the wave's heads
    if (on) {
#pragma unroll
      for (int x = 0; x < HPW; ++x) {
        if (hw + x >= a.H) break;
        if constexpr (HPW > 2) __builtin_amdgcn_sched_barrier(0);
        float p[8], mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = s_s[at(8 * xg + e, hw + x, xr)];
          p[e] = j0 + 8 * lg + e <= pos ? v : -INFINITY;
          mx = fmaxf(mx, p[e]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (__any(mx > m[x] + kRise)) {
          const float mn = mx > m[x] + kRise ? mx : m[x];
          const float corr = mn == m[x] ? 1.f : exp_near(m[x] - mn);
          l[x] *= corr;
          m[x] = mn;
#pragma unroll
          for (int n = 0; n < 8; ++n) O[x][n] *= corr;
        }
        const float ms = m[x] == -INFINITY ? 0.f : m[x];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = exp_near(p[e] - ms);
          l[x] += p[e];
        }
        uint4 part[3];                                   // the fp32 weights in three 16-bit parts: all of their bits
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          unsigned u[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (y == 0) { p[2 * e] *= kUp<T>; p[2 * e + 1] *= kUp<T>; }
            u[e] = pk2<T>(p[2 * e], p[2 * e + 1]);
            float h0, h1;
            unpack2<T>(u[e], h0, h1);
            p[2 * e] -= h0;
            p[2 * e + 1] -= h1;
          }
          part[y] = make_uint4(u[0], u[1], u[2], u[3]);
        }
        // lane (lr, lg) of operand n: channel 16 n + lr, keys 8 lg .. 8 lg + 7, from rows 8 lg + lr / 4 (+ 4)
        const char* vb = s_v + g * kKeys * 256;
        const int r = 8 * xg + (xr >> 2), half = 8 * (xr & 1);
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int ch = 2 * n + ((xr >> 1) & 1);
          const uint2 v0 = tr_read(vb + r * 256 + ((ch ^ vswz(r)) << 4) + half);
          const uint2 v1 = tr_read(vb + (r + 4) * 256 + ((ch ^ vswz(r + 4)) << 4) + half);
          const uint4 av = make_uint4(v0.x, v0.y, v1.x, v1.y);
#pragma unroll
          for (int y = 0; y < 3; ++y) O[x][n] = Mfma<T>::run(av, part[2 - y], O[x][n]);
        }
      }
    }
    __syncthreads();
  }
  if (s_tbl[kTbl] != 0 && on) {                          // what was blanked, for the rows that see it
    for (int j = (first + p0 + 1) / kKeys * kKeys; j <= pos; ++j) {      // (from the first such tile on)
      const T* vr = a.vc + (cache_row(j) * a.G + g) * kD + 4 * lg;
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        float v[4];
        odd4<T>(vr + 16 * n, v);
#pragma unroll
        for (int x = 0; x < HPW; ++x)
#pragma unroll
          for (int i = 0; i < 4; ++i) O[x][n][i] += v[i];
      }
    }
  }
  // O[x][n][i]: channel 16 n + 4 lg + i of head hw + x, row lr
#pragma unroll
  for (int x = 0; x < HPW; ++x) {
    float sum = l[x];
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    if (hw + x >= a.H || first + lr >= end) continue;
    const float inv = 1.f / (sum * kUp<T>);
    T* op = a.out + (long long)row * a.our + (long long)(hw + x) * a.ouh + 4 * lg;
#pragma unroll
    for (int n = 0; n < 8; ++n)
      *reinterpret_cast<uint2*>(op + 16 * n) =
          make_uint2(pk2<T>(O[x][n][0] * inv, O[x][n][1] * inv), pk2<T>(O[x][n][2] * inv, O[x][n][3] * inv));
  }
}

inline int heads_per_wave(int H) { return H <= 8 ? 1 : H <= 16 ? 2 : 4; }
inline size_t talk_lds(int H, int G) {
  return (size_t)kKeys * ((H + 15) / 16 * 16) * 16 * 4 + (size_t)G * kKeys * 256 + (kTbl + 4) * 4;
}

template <typename T>
hipError_t launch(const TalkArgs<T>& a, hipStream_t st) {
  const size_t lds = talk_lds(a.H, a.G);
  const dim3 grid((unsigned)(a.n_tiles * a.subs));
  const void* f = a.H <= 8    ? (const void*)talk_tile_kernel<T, 1, 1>
                  : a.H <= 16 ? (const void*)talk_tile_kernel<T, 2, 1>
                              : (const void*)talk_tile_kernel<T, 4, 2>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  if (a.H <= 8) talk_tile_kernel<T, 1, 1><<<grid, 512, lds, st>>>(a);
  else if (a.H <= 16) talk_tile_kernel<T, 2, 1><<<grid, 512, lds, st>>>(a);
  else talk_tile_kernel<T, 4, 2><<<grid, 512, lds, st>>>(a);
  return hipGetLastError();
}

}  // namespace

extern "C" {

// Does sm_talk_tiles have a kernel: heads of 128, up to 32 of them, the heads of a wave on one key head, and the
// scores and values of a tile in LDS.
int sm_talk_tiles_ok(int dt, int H, int G, int D, int Dv) {
  if ((dt != kBF16 && dt != kF16) || D != kD || Dv != kD || H < 1 || H > 32 || G < 1 || H % G) return 0;
  const int hpw = heads_per_wave(H);
  return (H / G) % hpw == 0 && talk_lds(H, G) <= 163840;
}

// The first rows of a step, cut into n_tiles tiles of tile_rows rows (q_tiles [n][2]: segment, first row); caches
// [blocks][bs][G][D]; the other arguments as sm_row_attn; strides of q % 8, of out % 4.
hipError_t sm_talk_tiles(int dt, const void* q, long long qr, long long qh, const void* kc, const void* vc, void* out,
                         long long our, long long ouh, const int* tables, int maxb, const int* q_tiles, int n_tiles,
                         int tile_rows, const int* cu, const int* start, int H, int G, int D, int Dv, int bs,
                         float scale, float softcap, float tcoef, int tevery, const float* r1, const float* r2,
                         const float* talk, const float* sink, hipStream_t st) {
  if (n_tiles == 0) return hipSuccess;
  const auto al = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (!sm_talk_tiles_ok(dt, H, G, D, Dv) || n_tiles < 0 || tile_rows < 1 || tile_rows > 4096 || bs < 1 ||
      talk == nullptr || (r1 != nullptr && r2 == nullptr) || !al(q) || qr % 8 || qh % 8 || !al(kc) || !al(vc) ||
      our % 4 || ouh % 4 || (uintptr_t)out % 8)
    return hipErrorInvalidValue;
#define GO(T)                                                                                                     \
  {                                                                                                               \
    const TalkArgs<T> a{(const T*)q, qr, qh, (const T*)kc, (const T*)vc, (T*)out, our, ouh, tables, maxb, q_tiles, \
                        cu, start, n_tiles, (tile_rows + kRows - 1) / kRows, tile_rows, H, G, bs, scale, softcap,  \
                        tcoef, tevery, r1, r2, talk, sink};                                                       \
    return launch<T>(a, st);                                                                                      \
  }
  if (dt == kBF16) GO(bf16)
  GO(fp16)
#undef GO
}

}  // extern "C"
