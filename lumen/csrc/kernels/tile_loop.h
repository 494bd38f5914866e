// The main loop of products x w^T on tiles of 32 MJ rows of x and 32 NI rows of w (16-bit operands, fp32 sums), one workgroup of
// four waves per CU; the kernels around it choose the rows and write the results.
//
//  * A wave owns 16 MJ x 16 NI results.  Operands come by LDS-DMA in stages of 64 k under counted waits, as many steps
//    ahead as fit into 160 KiB (six at most); one barrier per step.  256 x 160 and wider keep two slots of x, which comes from
//    L2, and three or four of w: loads return in the order they were sent for, and w from HBM takes longer than a step.
//  * With w from HBM few-row tiles wait for bytes: a CU takes 97 B/ns from L2 and 60 of lines from HBM, however many are in
//    flight (48 KB do), so the tile is as narrow in x as the rows are.  Rows of w some KB apart, read a stage at
//    a time by all workgroups in step, meet in the same memory channels: the caller may have a tile start its walk of k
//    elsewhere (`turn`; a bare stream of rows 8 KB apart 5.0 -> 5.6 TB/s, 4 KB apart 4.45 -> 5.45).
//  * Between two products stands at most one other thing, a fragment read or a DMA: in groups of eight products
//    behind their reads the matrix core waited for the issue (256 x 128: 0.82 -> 0.75 us a step, 256 x 256 1.27 -> 1.0).
//  * The accumulators are named as accumulation registers in the products' assembly.  The compiler, left to place them, splits
//    128 and more over both files and moves them to and fro, or spills (256 x 256).
// On 128 CUs a 256 x 256 step takes 0.95 us, 0.85 being the matrix core's; on all 256 the clock falls with the power of random
// operands: 1.25 us, as in the library (zeros: 0.98; products alone: 2.04 PFLOP/s random, 2.41 zeros).
#pragma once
#include "common.h"

namespace lumen {
namespace tile {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// c += a b.  The compiler sees the operands' waits but not the matrix core's latency: whoever reads c by other means goes
// through settle() and hold() first.
template <typename T>
__device__ __forceinline__ void mfma(f32x4& c, uint4 a, uint4 b) {
  if constexpr (__is_same(T, bf16))
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c)
                 : "v"(__builtin_bit_cast(bf16x8, a)), "v"(__builtin_bit_cast(bf16x8, b)));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c)
                 : "v"(__builtin_bit_cast(f16x8, a)), "v"(__builtin_bit_cast(f16x8, b)));
}
// the last products have left the matrix core
__device__ __forceinline__ void settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }
// a read of c is not moved ahead of this
__device__ __forceinline__ void hold(f32x4& c) { asm volatile("" : "+a"(c)); }

constexpr int BK = 64, ROWB = 128;                       // a row of a stage is 64 elements, 128 bytes
constexpr int CUS = 256;

template <int NI, int MJ>
struct Shape {
  static constexpr int BM = 32 * MJ, BN = 32 * NI, XB = BM * ROWB, WB = BN * ROWB;
  static constexpr bool DEEP = MJ == 8 && NI >= 5;       // two slots of x, more of w
  static constexpr int FIT = DEEP ? (160 * 1024 - 2 * XB) / WB : 160 * 1024 / (XB + WB);
  static constexpr int NST = FIT < 6 ? FIT : 6, NSX = DEEP ? 2 : NST;            // slots of w and x
  static constexpr int LDS = NSX * XB + NST * WB;
  static_assert(NST >= 3, "slots");
  static constexpr int PIECES = MJ + NI;                 // 1-KiB LDS-DMA pieces of a wave and stage: MJ of x, NI of w
};

// 16-byte chunk c of stage row r lies at chunk c ^ swz(r): a fragment read (16 rows at one chunk) and an
// LDS-DMA piece (8 whole rows) are both conflict free
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }

template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0xF70);
}

// all but the last r (R at most) stages have arrived
template <int R, int PIECES>
__device__ __forceinline__ void wait_stages(int r) {
  if constexpr (R <= 0) wait_vm<0>();
  else if (r >= R) wait_vm<R * PIECES>();
  else wait_stages<R - 1, PIECES>(r);
}

// LDS-DMA of 16 bytes per lane into the wave's 1-KiB piece (M0: its LDS address).  Inline asm, so that
// the waits of the loop's own counting order it.
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

// Block b of n -> unit: blocks go to the XCDs in turn, XCD x takes consecutive units.
__device__ __forceinline__ int unit_of(int b, int n) {
  const int xcd = b & 7, q8 = n >> 3, r8 = n & 7;
  return (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + (b >> 3);
}
// Tile -> (row tile, column tile): `group` row tiles by all column tiles, row tiles first, so that the 32 tiles an XCD holds at
// a time read a few panels of both operands from its L2.
__device__ __forceinline__ void tile_at(int tile, int tiles_m, int tiles_n, int group, int& tm, int& tn) {
  const int gsz = group * tiles_n, g = tile / gsz, gr = min(group, tiles_m - g * group), in = tile - g * gsz;
  tn = in / gr;
  tm = g * group + in - tn * gr;
}

// W row of a wave's 16 NI -> column: the fragments of a pair give a lane 8 consecutive columns (the last of an odd
// number of fragments 4)
template <int NI>
__device__ __forceinline__ int colperm(int w) {
  if ((w & ~31) + 32 > 16 * NI) return w;
  return (w & ~31) | (((w >> 2) & 3) << 3) | (((w >> 4) & 1) << 2) | (w & 3);
}

// acc[i][j] = products of fragments i of w and j of x over nk stages (64 k each) from xb and wb, to which off[q] is the
// lane's byte offset of the wave's piece q: stage rows 8 (wid + 4 q) + lane / 8 of x for q < MJ, of w from piece MJ on, chunk
// (lane & 7) ^ swz(row).  APART: the walk starts at stage `turn` < nk and comes round to it.  Lane (lr, lg) holds row 16 j + lr of its
// wave's x, rows 16 i + 4 lg .. + 3 of its w.  HALF: with `odd` the last stage holds 32 k; its lanes of the upper half read the lower
// one again, which is multiplied once.
//
// Step t multiplies stage t; at its start the first half's fragments are in registers.  Behind the first half's products it
// reads the second half's; then stage t + 1 has to be there, and every wave done with stage t, whose slots the second half's
// pieces may take.
//  * NST slots of both: the second half sends for the last pieces of stage t + NST, the next step's first half for its others.
//  * DEEP: the second half sends for all of x of stage t + 2 and then w of stage t + NST, which thus has a step and a half before x of
//    stage t + 3 has to be there, sent for after it.  With three slots of x and two of w it had half a step to one, and the
//    card's memory answered later: 512 rows x 2 x 11264 x 4096 with activation (256 x 192) 89.8 -> 81.6 us, x 18560 (256 x 160) 78 -> 72, x
//    22016 (256 x 192) 83.6 -> 78.8; 4096 x 2 x 11008 x 4096 (256 x 256) 554 -> 535 and 521 -> 515 (two cards).  256 x 128 was no faster so
//    (512 x 16384 61.7 -> 62.6).
template <typename T, int NI, int MJ, bool APART = false, bool HALF = false>
__device__ __forceinline__ void products(char* lds, const char* xb, const char* wb, int nk, int turn,
                                         const unsigned (&off)[Shape<NI, MJ>::PIECES], f32x4 (&acc)[NI][MJ], bool odd = false) {
  using S = Shape<NI, MJ>;
  constexpr int NSX = S::NSX, NST = S::NST, XB = S::XB, WB = S::WB, PIECES = S::PIECES;
  constexpr bool DEEP = S::DEEP;
  static_assert(!DEEP || !APART, "no caller has wide tiles walk apart");
  constexpr int PB = PIECES - PIECES / 2, F = NST - 1;   // !DEEP: pieces [PB, PIECES) go out in a second half, [0, PB) in a first
  struct Slot { int x, w; };
  const int lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds);
  const unsigned upper = HALF && odd && (((lane >> 2) ^ wid) & 1) ? BK : 0;     // (bytes; chunk (lane & 7) ^ swz(row) >= 4)
  // pieces q0 .. q1 - 1 of stage t, of x (q < MJ) to slot.x, of w to slot.w
  auto issue = [&](int t, Slot slot, int q0, int q1) __attribute__((always_inline)) {
    const unsigned back = HALF && t == nk - 1 ? upper : 0;
    const int u = APART ? (t + turn < nk ? t + turn : t + turn - nk) : t;
    const char *xs = xb + (long long)u * (BK * 2), *ws = wb + (long long)u * (BK * 2);
    const unsigned dx = __builtin_amdgcn_readfirstlane(lds0 + slot.x * XB + wid * 1024);
    const unsigned dw = __builtin_amdgcn_readfirstlane(lds0 + NSX * XB + slot.w * WB + wid * 1024);
#pragma unroll
    for (int q = q0; q < q1; ++q) dma16(q < MJ ? xs : ws, HALF ? off[q] - back : off[q], q < MJ ? dx + q * 4096 : dw + (q - MJ) * 4096);
  };
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}, hold(acc[i][j]);
  settle();                                              // (and the products find the zeros written)
  uint4 fa[2][NI], fb[2][MJ];
  const int rb0 = (16 * MJ * (wid >> 1) + lr) * ROWB, ra0 = (16 * NI * (wid & 1) + lr) * ROWB;
  // fragments u0 .. u1 - 1 of half h of a stage (w's, then x's)
  auto frags = [&](int h, Slot slot, int u0, int u1) __attribute__((always_inline)) {
    const int c = ((4 * h + lg) ^ swz(lr)) << 4;
    const char *px = lds + slot.x * XB + c, *pw = lds + NSX * XB + slot.w * WB + c;
#pragma unroll
    for (int u = u0; u < u1; ++u)
      if (u < NI) fa[h][u] = *reinterpret_cast<const uint4*>(pw + ra0 + u * 16 * ROWB);
      else fb[h][u - NI] = *reinterpret_cast<const uint4*>(px + rb0 + (u - NI) * 16 * ROWB);
  };
  // the products of half h; between them the reads of the other half's fragments (from stage slot fs, in the first
  // three quarters) and `send(a, b)` for pieces a .. b - 1 of P
  auto half = [&](int h, Slot fs, int P, auto&& send) __attribute__((always_inline)) {
    constexpr int U = NI * MJ, R = NI + MJ, UR = U * 3 / 4;
#pragma unroll
    for (int j = 0; j < MJ; ++j)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int n = j * NI + i;
        mfma<T>(acc[i][j], fa[h][i], fb[h][j]);
        frags(1 - h, fs, min(R, (n * R + UR - 1) / UR), min(R, ((n + 1) * R + UR - 1) / UR));
        send(n * P / U, (n + 1) * P / U);
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  const auto none = [](int, int) __attribute__((always_inline)) {};
  auto after = [](Slot s) __attribute__((always_inline)) {
    return Slot{s.x == NSX - 1 ? 0 : s.x + 1, s.w == NST - 1 ? 0 : s.w + 1};
  };
  Slot s0{0, 0}, s1{1, 1};                               // slots of stages t, t + 1
  int t = 0;
  if constexpr (DEEP) {
    // sent for in this order: w and x of stage 0, w of the others, x of stage 1, the last slot's w
    issue(0, s0, MJ, PIECES);
    issue(0, s0, 0, MJ);
#pragma unroll
    for (int u = 1; u < NST - 1; ++u)
      if (u < nk) issue(u, Slot{0, u}, MJ, PIECES);
    if (nk > 1) issue(1, s1, 0, MJ);
    if (nk >= NST) issue(NST - 1, Slot{0, NST - 1}, MJ, PIECES), wait_vm<(NST - 1) * NI + MJ>();
    else wait_vm<0>();
  } else {
#pragma unroll
    for (int u = 0; u < F; ++u)
      if (u < nk) issue(u, Slot{u, u}, 0, PIECES);
    if (nk > F) issue(F, Slot{F, F}, PB, PIECES), wait_vm<(F - 1) * PIECES + PIECES - PB>();
    else if (nk == F) wait_vm<(F - 1) * PIECES>();
    else wait_vm<0>();
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  frags(0, s0, 0, NI + MJ);
  if constexpr (DEEP) {
    for (; t + NST < nk; ++t) {
      half(0, s0, 0, none);
      wait_vm<NI>();                                     // (all but w of stage t + NST - 1)
      done_reading();
      half(1, s1, PIECES, [&](int a, int b) __attribute__((always_inline)) {
        issue(t + 2, s0, min(a, MJ), min(b, MJ));
        issue(t + NST, s0, max(a, MJ), max(b, MJ));
      });
      s0 = s1, s1 = after(s1);
    }
    for (; t < nk; ++t) {                                // the last stages
      half(0, s0, 0, none);
      wait_vm<0>();
      done_reading();
      if (!HALF || !odd || t + 1 < nk)                   // (the last step reads a slot that holds an earlier stage: unused)
        half(1, s1, MJ, [&](int a, int b) __attribute__((always_inline)) {
          if (t + 2 < nk) issue(t + 2, s0, a, b);
        });
      s0 = s1, s1 = after(s1);
    }
  } else {
    Slot sf{F, F};                                       // slot of stage t + F
    for (; t + NST < nk; ++t) {
      half(0, s0, PB, [&](int a, int b) __attribute__((always_inline)) { issue(t + F, sf, a, b); });
      wait_vm<(F - 1) * PIECES>();
      done_reading();
      half(1, s1, PIECES - PB, [&](int a, int b) __attribute__((always_inline)) { issue(t + NST, s0, PB + a, PB + b); });
      s0 = s1, s1 = after(s1), sf = after(sf);
    }
    for (; t < nk; ++t) {                                // the last stages
      half(0, s0, PB, [&](int a, int b) __attribute__((always_inline)) { if (t + F < nk) issue(t + F, sf, a, b); });
      wait_stages<F - 1, PIECES>(nk - 2 - t);
      done_reading();
      if (!HALF || !odd || t + 1 < nk) half(1, s1, 0, none);
      s0 = s1, s1 = after(s1), sf = after(sf);
    }
  }
  settle();
}

}  // namespace tile
}  // namespace lumen
