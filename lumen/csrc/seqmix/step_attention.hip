// Attention of decoded rows against paged key and value caches, heads of 128: row_attention.hip's scores and weights for
// the sizes that a decode step has, with a shorter chain.
//
// What bounds it: the general row kernel asks for a tile's keys 32 channels at a time and per key head, for its values in
// four rounds, and mixes heads through loads of the mixing matrix, so a step waits for memory ten times and more per tile.
// Here a wave asks for all key and value rows of its tile before the first product (128 - 256 bytes a lane), and for the
// next tile's while it multiplies this one's.
//  * step_attn_kernel: a workgroup serves one row and one key head with its HP query heads; its four waves take 16 keys
//    of a 64-key tile each and run an online softmax of their own -- no barrier in the loop -- that meet once at the end.
//    Scores are S = K Q^T on the matrix cores, the query operand comes straight from memory; weights reach the lanes that
//    own 8 channels of a value row through the wave's own LDS, in fp32.
//  * talk_attn_kernel (mixed heads): a wave per key head, all of a tile's 64 keys; the shaped scores of all heads meet in
//    LDS (a barrier a tile, two buffers), lane = key there, the mixing matrix is read from LDS.
// The accumulators of the 16-lane rows are added by v_permlane32_swap / 16_swap, which halve the registers as they go.
// Keys that a row does not see are not read: the row's own stands in.  Their values are zeros, as 0 times an infinity is NaN.
// Measured in a graph, caches rotated through 700 MB, merge of the splits included, us, the general row kernel -> here (16 heads
// over 4 key heads, bf16): 1 row of 331 tokens 12.0 -> 7.7, of 4000 22.1 -> 13.2; 16 rows of 62 - 500 19.3 -> 10.6; 64 rows of 125 -
// 1000 56 -> 31.5 (its caches at 7 TB/s: 10.7), 200 of 62 - 500 94 -> 44; mixed heads with cap, distance bias and sink: 1 row of
// 331 30.6 -> 12.2, 64 rows of 64 - 514 50 -> 20, 32 heads 104 -> 38.
#include "row_attn_args.h"
#include "mma.h"

namespace lumen {
namespace {

constexpr int D = 128, TILE = 64;

// the cache row of key j, blocks of 1 << sh tokens
__device__ __forceinline__ int cache_row(const int* tbl, int sh, int j) {
  return (tbl[j >> sh] << sh) + (j & ((1 << sh) - 1));
}

// lane l of the result: a(l) + a(l ^ 32) below 32, b's above; 16: a's in even rows of 16 lanes, b's in odd ones
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// acc[h][e] of a lane (row kg of 16 lanes, part): summed over the rows, lane row kg keeps the flat entries (8 h + e) 2 HP kg ..
template <int HP> __device__ __forceinline__ void fold(const float (&acc)[HP][8], float (&o)[2 * HP]) {
  float t[4 * HP];
#pragma unroll
  for (int r = 0; r < 4 * HP; ++r) t[r] = fold32(acc[r / 8][r % 8], acc[(r + 4 * HP) / 8][r % 8]);
#pragma unroll
  for (int r = 0; r < 2 * HP; ++r) o[r] = fold16(t[r], t[r + 2 * HP]);
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
}

// the largest of every head's values over the wave, known to all lanes
template <int CTRL> __device__ __forceinline__ float dpp_max(float v) {
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false)));
}
__device__ __forceinline__ float fold32_max(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float fold16_max(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
template <int HP> __device__ __forceinline__ void wave_maxima(const float (&s)[HP], float (&o)[HP]) {
  static_assert(HP == 2 || HP == 4, "heads of a wave");
  float v = HP == 4 ? fold16_max(fold32_max(s[0], s[HP / 2]), fold32_max(s[1], s[HP - 1])) : fold32_max(s[0], s[1]);
  if (HP == 2) v = fold16_max(v, v);
  v = dpp_max<0x128>(v);                          // rotations within a row of 16 lanes by 8, 4, 2, 1
  v = dpp_max<0x124>(v);
  v = dpp_max<0x122>(v);
  v = dpp_max<0x121>(v);
#pragma unroll
  for (int i = 0; i < HP; ++i)
    o[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 64 / HP * i));
}

// a head's biases, asked for before the keys arrive
struct Bias {
  float r1 = 0.f, r2 = 0.f, slope = 0.f;
  __device__ Bias() {}
  template <typename T>
  __device__ __forceinline__ Bias(const RowAttnArgs<T>& a, int h)
      : r1(a.r1 ? a.r1[h] : 0.f), r2(a.r1 ? a.r2[h] : 0.f), slope(a.slopes ? a.slopes[h] : 0.f) {}
  __device__ __forceinline__ Bias uniform() const {                     // (one head for all lanes)
    const auto first = [](float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v))); };
    Bias b;
    b.r1 = first(r1); b.r2 = first(r2); b.slope = first(slope);
    return b;
  }
};
template <typename T>
__device__ __forceinline__ float shaped(const RowAttnArgs<T>& a, float s, const Bias& b, float dist) {
  if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
  if (a.r1 != nullptr) s -= b.r1 * logf(1.f + b.r2 * dist);
  if (a.slopes != nullptr) s -= b.slope * dist;
  return s;
}
template <typename T> __device__ __forceinline__ float query_scale(const RowAttnArgs<T>& a, int pos) {
  return a.tevery > 0 && a.tcoef != 0.f ? a.scale * (1.f + a.tcoef * logf((float)((pos + 1) / a.tevery) + 1.f)) : a.scale;
}

// does a row see all of the n keys from j0 on (one answer for the wave)
template <typename T> __device__ __forceinline__ bool all_seen(const RowAttnArgs<T>& a, int j0, int n, int pos) {
  return j0 + n - 1 <= pos && (a.window <= 0 || pos - j0 < a.window || j0 + n <= a.keep);
}

// the values of a cache row, or (row < 0) zeros for a key that is not seen.  Mixed heads choose the address: to blank 16 values
// behind their loads is a longer program, and a step of one tile waits for its instructions too (30 rows 8.0 us, blanked 8.7,
// here 8.2; of the four values of a wave of the other kernel, where a branch passes over whole tiles, 4.4 us, blanked 4.45, chosen
// 4.5).  As a number, for the compiler took the choice of two pointers for a flat one, whose loads count as LDS reads too (8.6).
__device__ const uint4 kNoValue = {0u, 0u, 0u, 0u};
template <typename T> __device__ __forceinline__ uint4 values_of(const T* vb, int row, long long ld) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  const uintptr_t at = row < 0 ? reinterpret_cast<uintptr_t>(&kNoValue) : reinterpret_cast<uintptr_t>(vb + (long long)row * ld);
  return __builtin_bit_cast(uint4, *reinterpret_cast<const __attribute__((address_space(1))) u32x4*>(at));
}

// acc += p v of one value chunk of 8 channels
template <typename T, int HP>
__device__ __forceinline__ void add_value(float (&acc)[HP][8], const uint4& v, const float (&p)[HP]) {
  float x[8];
  unpack2<T>(v.x, x[0], x[1]);
  unpack2<T>(v.y, x[2], x[3]);
  unpack2<T>(v.z, x[4], x[5]);
  unpack2<T>(v.w, x[6], x[7]);
#pragma unroll
  for (int h = 0; h < HP; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[h][e] = fmaf(p[h], x[e], acc[h][e]);
}

template <typename T, int HP>
__global__ void __launch_bounds__(256, HP == 8 ? 2 : 3)
step_attn_kernel(const RowAttnArgs<T> a) {
  __shared__ __attribute__((aligned(16))) float s_p[4][4][HP][4];      // wave, its row of 16 lanes, head, key
  __shared__ float s_c[4][HP];
  __shared__ __attribute__((aligned(16))) float s_o[4][HP][D];
  __shared__ float s_m[4][HP], s_l[4][HP];
  const int t = row_of(a, blockIdx.x, gridDim.x), g = blockIdx.y, z = blockIdx.z;
  const int lane = threadIdx.x & 63, lr = lane & 15, kg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pos = a.positions[t];
  const int* tbl = a.tables + (long long)a.row_seg[t] * a.maxb;
  const int sh = 31 - __builtin_clz(a.bs);
  const bool on = lr < HP;
  const int h = g * HP + (on ? lr : 0);
  uint4 qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    qf[s] = on ? *reinterpret_cast<const uint4*>(a.q1 + (long long)t * a.q1r + (long long)h * a.q1h + 32 * s + 8 * kg)
               : make_uint4(0u, 0u, 0u, 0u);
  const TileWalk walk(pos, a.window, a.keep);
  if (z >= walk.count) {                         // no tile (the merge reads no values of it)
    if ((int)threadIdx.x < HP) {
      const long long slot = ((long long)t * a.H + g * HP + threadIdx.x) * a.nsplit + z;
      a.ws_ml[2 * slot] = -INFINITY;
      a.ws_ml[2 * slot + 1] = -1.f;
    }
    return;
  }
  const float qscale = query_scale(a, pos);
  const Bias bias(a, h);
  const bool sk = a.sink != nullptr && z == 0 && w == 0;
  float m = sk ? a.sink[h] : -INFINITY, l = sk && kg == 0 ? 1.f : 0.f;   // l: this lane's keys only
  float acc[HP][8];
#pragma unroll
  for (int i = 0; i < HP; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[i][e] = 0.f;

  const T* kb = a.kc + (long long)g * D + 8 * kg;
  const T* vb = a.vc + (long long)g * D + 8 * lr;
  const auto first = [&](int tv) { return walk.key0(tv) + 16 * w; };   // the wave's first key
  const auto load = [&](int tv, uint4 (&k)[4], uint4 (&v)[4]) {
    const int j0 = first(tv);
    if (j0 > pos) return;
    const int j = j0 + lr;
    const int rb = cache_row(tbl, sh, key_seen(j, pos, a.window, a.keep) ? j : pos);
    const T* kp = kb + (long long)rb * a.krow;
#pragma unroll
    for (int s = 0; s < 4; ++s) k[s] = *reinterpret_cast<const uint4*>(kp + 32 * s);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const uint4*>(vb + (long long)__shfl(rb, 4 * kg + i, 64) * a.vrow);
  };
  const auto use = [&](int tv, const uint4 (&k)[4], uint4 (&v)[4]) {
    const int j0 = first(tv);
    if (j0 > pos) return;
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 4; ++s) c = Mfma<T>::run(k[s], qf[s], c);      // c[i] = S[key 4 kg + i][head lr]
    float sv[4], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = j0 + 4 * kg + i;
      sv[i] = key_seen(j, pos, a.window, a.keep) ? shaped(a, c[i] * qscale, bias, (float)(pos - j)) : -INFINITY;
      mx = fmaxf(mx, sv[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);
    const float corr = m == -INFINITY ? 0.f : expf(m - mn);
    float p[4];
    l *= corr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = sv[i] == -INFINITY ? 0.f : expf(sv[i] - mn);
      l += p[i];
    }
    m = mn;
    if (on) {
      *reinterpret_cast<float4*>(&s_p[w][kg][lr][0]) = make_float4(p[0], p[1], p[2], p[3]);
      if (kg == 0) s_c[w][lr] = corr;
    }
    wave_lds_fence();
    float ph[HP][4];
#pragma unroll
    for (int i = 0; i < HP; ++i) {
      const float4 q = *reinterpret_cast<const float4*>(&s_p[w][kg][i][0]);
      ph[i][0] = q.x; ph[i][1] = q.y; ph[i][2] = q.z; ph[i][3] = q.w;
      const float ci = s_c[w][i];
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i][e] *= ci;
    }
    if (!all_seen(a, j0, 16, pos)) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!key_seen(j0 + 4 * kg + i, pos, a.window, a.keep)) v[i] = make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float pk[HP];
#pragma unroll
      for (int n = 0; n < HP; ++n) pk[n] = ph[n][i];
      add_value<T, HP>(acc, v[i], pk);
    }
    wave_lds_fence();
  };
  uint4 k0[4], v0[4], k1[4], v1[4];
  load(z, k0, v0);
  for (int tv = z; tv < walk.count; tv += 2 * a.nsplit) {
    const int t1 = tv + a.nsplit, t2 = t1 + a.nsplit;
    if (t1 < walk.count) load(t1, k1, v1);
    use(tv, k0, v0);
    if (t1 < walk.count) {
      if (t2 < walk.count) load(t2, k0, v0);
      use(t1, k1, v1);
    }
  }
  // the four waves' states meet
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (kg == 0 && on) {
    s_m[w][lr] = m;
    s_l[w][lr] = l;
  }
  float o[2 * HP];
  fold<HP>(acc, o);
#pragma unroll
  for (int r = 0; r < 2 * HP; ++r) {
    const int at = r + 2 * HP * kg;
    s_o[w][at >> 3][8 * lr + (at & 7)] = o[r];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < HP * (D / 4); i += 256) {
    const int hh = i / (D / 4), d = 4 * (i % (D / 4)), head = g * HP + hh;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) M = fmaxf(M, s_m[q][hh]);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float e = s_m[q][hh] == -INFINITY ? 0.f : expf(s_m[q][hh] - M);
      L += s_l[q][hh] * e;
      sum += *reinterpret_cast<const f32x4*>(&s_o[q][hh][d]) * e;
    }
    if (a.nsplit == 1) {
      float inv = 1.f / L;
      if (a.gate != nullptr) inv *= sigmoid_f(to_f32(a.gate[(long long)t * a.gater + head]));
      *reinterpret_cast<uint2*>(a.out + (long long)t * a.our + (long long)head * a.ouh + d) =
          make_uint2(pk2<T>(sum[0] * inv, sum[1] * inv), pk2<T>(sum[2] * inv, sum[3] * inv));
    } else {
      const long long slot = ((long long)t * a.H + head) * a.nsplit + z;
      if (d == 0) {
        a.ws_ml[2 * slot] = M;
        a.ws_ml[2 * slot + 1] = L;
      }
      *reinterpret_cast<f32x4*>(a.ws_o + slot * D + d) = sum;
    }
  }
}

// LDS of the mixed form: scores of all heads [2][TILE][H + 4] | a wave's scores and weights [G][HP][TILE] | talk [H][H]
__host__ __device__ inline int talk_lds(int H) { return 4 * (2 * TILE * (H + 4) + H * TILE + H * H); }

template <typename T, int HP>
__global__ void __launch_bounds__(512, 2)
talk_attn_kernel(const RowAttnArgs<T> a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int t = row_of(a, blockIdx.x, gridDim.x), z = blockIdx.z, H = a.H, ld = H + 4;
  const int lane = threadIdx.x & 63, lr = lane & 15, kg = lane >> 4;
  const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);      // the wave's key head
  float* s_sc = smem;
  float* s_p = smem + 2 * TILE * ld + g * HP * TILE;                   // [HP][TILE]; raw scores as [TILE][HP]
  float* s_talk = smem + 2 * TILE * ld + H * TILE;
  const int pos = a.positions[t];
  const int* tbl = a.tables + (long long)a.row_seg[t] * a.maxb;
  const int sh = 31 - __builtin_clz(a.bs);
  const bool on = lr < HP;
  uint4 qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s)
    qf[s] = on ? *reinterpret_cast<const uint4*>(a.q1 + (long long)t * a.q1r + (long long)(g * HP + lr) * a.q1h + 32 * s + 8 * kg)
               : make_uint4(0u, 0u, 0u, 0u);
  const TileWalk walk(pos, a.window, a.keep);
  if (z >= walk.count) {
    if (lane < HP) {
      const long long slot = ((long long)t * H + g * HP + lane) * a.nsplit + z;
      a.ws_ml[2 * slot] = -INFINITY;
      a.ws_ml[2 * slot + 1] = -1.f;
    }
    return;
  }
  const float qscale = query_scale(a, pos);
  const T* kb = a.kc + (long long)g * D + 8 * kg;
  const T* vb = a.vc + (long long)g * D + 8 * lr;
  float tk[2];                                    // H^2 <= 16 G^2 entries, 64 G threads
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int at = threadIdx.x + i * blockDim.x;
    tk[i] = a.talk[at < H * H ? at : 0];
  }
  float m[HP], l[HP], acc[HP][8];
  Bias bias[HP];
#pragma unroll
  for (int i = 0; i < HP; ++i) bias[i] = Bias(a, g * HP + i).uniform();
#pragma unroll
  for (int i = 0; i < HP; ++i) {
    const bool sk = a.sink != nullptr && z == 0;
    m[i] = sk ? a.sink[g * HP + i] : -INFINITY;
    l[i] = sk && lane == 0 ? 1.f : 0.f;                                 // this lane's keys only
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[i][e] = 0.f;
  }
  int buf = 0;
  for (int tv = z; tv < walk.count; tv += a.nsplit, buf ^= 1) {
    const int j0 = walk.key0(tv);
    float* sc = s_sc + buf * TILE * ld;
    // the tile's keys and half of its values are asked for at once, the other half when the keys have been multiplied
    uint4 k[4][4], v[4][4];
    int rb[4], rv[4];
    const auto load_values = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[u][i] = values_of(vb, __shfl(rv[u], 4 * kg + i, 64), a.vrow);
    };
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + 16 * u + lr;
      const bool seen = key_seen(j, pos, a.window, a.keep);
      rb[u] = cache_row(tbl, sh, seen ? j : pos);
      rv[u] = seen ? rb[u] : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const T* kp = kb + (long long)rb[u] * a.krow;
#pragma unroll
      for (int s = 0; s < 4; ++s) k[u][s] = *reinterpret_cast<const uint4*>(kp + 32 * s);
    }
    load_values(0);
    load_values(1);
    if (tv == z) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int at = threadIdx.x + i * blockDim.x;
        if (at < H * H) s_talk[at] = tk[i];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) c = Mfma<T>::run(k[u][s], qf[s], c);  // c[i] = S[key 16 u + 4 kg + i][head lr]
      if (on)
#pragma unroll
        for (int i = 0; i < 4; ++i) s_p[(16 * u + 4 * kg + i) * HP + lr] = c[i];
    }
    __builtin_amdgcn_sched_barrier(0);            // (into the registers of the keys)
    load_values(2);
    load_values(3);
    wave_lds_fence();
    // lane = key from here on
    const int j = j0 + lane;
    const bool seen = key_seen(j, pos, a.window, a.keep);
    float s[HP];
#pragma unroll
    for (int i = 0; i < HP; ++i) {
      s[i] = s_p[lane * HP + i];
      s[i] = seen ? shaped(a, s[i] * qscale, bias[i], (float)(pos - j)) : 0.f;
      sc[lane * ld + g * HP + i] = s[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < HP; ++i) s[i] = 0.f;
#pragma unroll 1
    for (int n = 0; n < H; n += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(sc + lane * ld + n);
#pragma unroll
      for (int i = 0; i < HP; ++i) {
        const f32x4 y = *reinterpret_cast<const f32x4*>(s_talk + (g * HP + i) * H + n);
        s[i] += y[0] * x[0];
        s[i] += y[1] * x[1];
        s[i] += y[2] * x[2];
        s[i] += y[3] * x[3];
      }
    }
#pragma unroll
    for (int i = 0; i < HP; ++i) s[i] = seen ? s[i] : -INFINITY;
    float mx[HP];
    wave_maxima<HP>(s, mx);
#pragma unroll
    for (int i = 0; i < HP; ++i) {
      const float mn = fmaxf(m[i], mx[i]);
      const float corr = m[i] == -INFINITY ? 0.f : expf(m[i] - mn);
      const float p = s[i] == -INFINITY ? 0.f : expf(s[i] - mn);
      l[i] = l[i] * corr + p;
      m[i] = mn;
      s_p[i * TILE + lane] = p;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[i][e] *= corr;
    }
    wave_lds_fence();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f32x4 p[HP];
#pragma unroll
      for (int n = 0; n < HP; ++n) p[n] = *reinterpret_cast<const f32x4*>(s_p + n * TILE + 16 * u + 4 * kg);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float pk[HP];
#pragma unroll
        for (int n = 0; n < HP; ++n) pk[n] = p[n][i];
        add_value<T, HP>(acc, v[u][i], pk);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    wave_lds_fence();
  }
  float o[2 * HP];
  fold<HP>(acc, o);
  float L[HP];
#pragma unroll
  for (int i = 0; i < HP; ++i) L[i] = wave_sum(l[i]);
#pragma unroll
  for (int i = 0; i < HP; ++i) {
    // flat entries 8 i .. 8 i + 7 of the wave's heads lie with the lane rows that 8 i / (2 HP) ff. name
    constexpr int per = 2 * HP;                                          // entries of a lane
    if (kg != 8 * i / per && per >= 8) continue;
    const int head = g * HP + i;
    const long long slot = ((long long)t * H + head) * a.nsplit + z;
    float inv = 1.f;
    if (a.nsplit == 1) {
      inv = 1.f / L[i];
      if (a.gate != nullptr) inv *= sigmoid_f(to_f32(a.gate[(long long)t * a.gater + head]));
    } else if (lr == 0 && (per >= 8 || kg == 8 * i / per)) {
      a.ws_ml[2 * slot] = m[i];
      a.ws_ml[2 * slot + 1] = L[i];
    }
    const int r0 = per >= 8 ? 8 * i % per : 0, e0 = per >= 8 ? 0 : per * kg - 8 * i;
    constexpr int n = per < 8 ? per : 8;
    if (e0 < 0 || e0 >= 8) continue;
    if (a.nsplit == 1) {
      T* op = a.out + (long long)t * a.our + (long long)head * a.ouh + 8 * lr + e0;
#pragma unroll
      for (int e = 0; e < n; e += 4)
        *reinterpret_cast<uint2*>(op + e) =
            make_uint2(pk2<T>(o[r0 + e] * inv, o[r0 + e + 1] * inv), pk2<T>(o[r0 + e + 2] * inv, o[r0 + e + 3] * inv));
    } else {
      float* op = a.ws_o + slot * D + 8 * lr + e0;
#pragma unroll
      for (int e = 0; e < n; e += 4)
        *reinterpret_cast<f32x4*>(op + e) = f32x4{o[r0 + e], o[r0 + e + 1], o[r0 + e + 2], o[r0 + e + 3]};
    }
  }
}

}  // namespace

// Heads of 128 over key and value caches with rows of whole heads, 2, 4 or 8 query heads a key head, 16-bit types; mixed
// heads: at most 8 key heads of up to 4.
template <typename T> bool step_attn_ok(const RowAttnArgs<T>& a) {
  const auto al = [](const void* p, int n) { return (uintptr_t)p % n == 0; };
  const int hp = a.H / a.G;
  return a.D1 == D && a.D2 == 0 && a.Dv == D && a.vdiv == 1 && a.sigb == nullptr && a.krow == (long long)a.G * D &&
         a.vrow == (long long)a.G * D && (hp == 2 || hp == 4 || hp == 8) && a.G <= 65535 && a.bs >= 1 &&
         (a.bs & (a.bs - 1)) == 0 && (a.talk == nullptr || (hp <= 4 && a.G <= 8 && a.H % 4 == 0)) && al(a.kc, 16) && al(a.vc, 16) && al(a.q1, 16) &&
         a.q1r % 8 == 0 && a.q1h % 8 == 0 && al(a.out, 8) && a.our % 4 == 0 && a.ouh % 4 == 0 && al(a.ws_o, 16);
}
template <> bool step_attn_ok<float>(const RowAttnArgs<float>&) { return false; }

template <typename T> hipError_t launch_step_attn(const RowAttnArgs<T>& a, int Tn, hipStream_t st) {
  const int hp = a.H / a.G;
  const dim3 grid(Tn, a.talk ? 1 : a.G, a.nsplit);
  if (a.talk) {
    if (hp == 2) talk_attn_kernel<T, 2><<<grid, 64 * a.G, talk_lds(a.H), st>>>(a);
    else talk_attn_kernel<T, 4><<<grid, 64 * a.G, talk_lds(a.H), st>>>(a);
  } else if (hp == 2) {
    step_attn_kernel<T, 2><<<grid, 256, 0, st>>>(a);
  } else if (hp == 4) {
    step_attn_kernel<T, 4><<<grid, 256, 0, st>>>(a);
  } else {
    step_attn_kernel<T, 8><<<grid, 256, 0, st>>>(a);
  }
  return hipGetLastError();
}
template <> hipError_t launch_step_attn<float>(const RowAttnArgs<float>&, int, hipStream_t) { return hipErrorInvalidValue; }

template bool step_attn_ok<bf16>(const RowAttnArgs<bf16>&);
template bool step_attn_ok<fp16>(const RowAttnArgs<fp16>&);
template hipError_t launch_step_attn<bf16>(const RowAttnArgs<bf16>&, int, hipStream_t);
template hipError_t launch_step_attn<fp16>(const RowAttnArgs<fp16>&, int, hipStream_t);

}  // namespace lumen

// 1 when sm_row_attn takes these kernels for the operands (arguments as there; mixed, sigmoid: are `talk`, `sigb` given), which
// want other splits of the keys than the general one
extern "C" int sm_step_attn_ok(int dt, const void* q1, long long q1r, long long q1h, int D1, int D2, const void* kc, long long krow,
                               const void* vc, long long vrow, int Dv, const void* out, long long our, long long ouh, int H,
                               int G, int bs, int mixed, int sigmoid, int vdiv) {
  using namespace lumen;
  if ((dt != kBF16 && dt != kF16) || G < 1 || H % G) return 0;
  static const float given = 0.f;
  RowAttnArgs<bf16> a{};
  a.q1 = (const bf16*)q1; a.q1r = q1r; a.q1h = q1h; a.D1 = D1; a.D2 = D2;
  a.kc = (const bf16*)kc; a.krow = krow; a.vc = (const bf16*)vc; a.vrow = vrow; a.Dv = Dv;
  a.out = (bf16*)out; a.our = our; a.ouh = ouh;
  a.H = H; a.G = G; a.bs = bs; a.vdiv = vdiv;
  a.talk = mixed ? &given : nullptr;
  a.sigb = sigmoid ? &given : nullptr;
  return step_attn_ok(a);
}
