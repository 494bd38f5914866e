// Operands of the attention of single rows against paged caches, shared by its kernels.
#pragma once
#include "seqmix.h"

namespace lumen {

constexpr int kQPad = 8;      // padding of the 16-bit query rows in LDS (bank spread)

// Workgroups are handed to the 8 XCDs round-robin in launch order, and every XCD has an L2 of its
// own.  Rows of a prompt's portion that follow each other belong to one sequence and read the same cache
// blocks, so XCD x takes the x-th CONTIGUOUS eighth of the rows instead of every eighth row:
// workgroup b -> row start(b % 8) + b / 8 (a bijection for any row count).  Decoded rows share nothing, and are
// dealt out as they come: in eighths the longest contexts may all fall to one XCD and its share of the memory's rate (200
// rows of 500 - 62 tokens in that order, 16 heads over 4: 43.7 -> 31.2 us).
__device__ __forceinline__ int xcd_row(int b, int n) {
  const int q = n / 8, r = n % 8, x = b % 8;
  return x * q + min(x, r) + b / 8;
}

template <typename T>
struct RowAttnArgs {
  const T* q1; long long q1r, q1h; int D1;
  const T* q2; long long q2r, q2h; int D2;
  const T* kc; long long krow;
  const T* vc; long long vrow; int Dv;
  T* out; long long our, ouh;
  const int* tables; int maxb;
  const int* row_seg; const int* positions;
  int H, G, HB, bs;
  float scale, softcap, tcoef; int tevery;
  const float *r1, *r2, *talk, *sink;
  const float* slopes; int window, keep;     // linear distance bias; window + kept first keys
  const T* gate; long long gater;            // per-head output gate logits [T][H], row stride
  const float* sigb; int vdiv;               // sigmoid weights' per-head bias; key heads per value head
  int own;                                   // every row is a sequence of its own
  int nsplit; float* ws_ml; float* ws_o;     // key splits: partial (max, sum) and accumulators
};

template <typename T> __device__ __forceinline__ int row_of(const RowAttnArgs<T>& a, int b, int n) {
  return a.own ? b : xcd_row(b, n);
}

// The 64-key tiles a row at position `pos` visits: without a window all of 0 .. pos / 64; with one
// the tiles of the first `keep` keys (as far as they lie below the window) and then those of the
// window [pos - window + 1, pos].  Every visited tile holds at least one key the row sees.
struct TileWalk {
  int head, first, count;                    // tiles 0 .. head - 1, then first, first + 1, ...
  __device__ __forceinline__ TileWalk(int pos, int window, int keep) {
    const int lo = window > 0 ? max(0, pos - window + 1) : 0;
    first = lo / 64;
    head = min((min(keep, lo) + 63) / 64, first);
    count = head + pos / 64 - first + 1;
  }
  __device__ __forceinline__ int key0(int v) const { return 64 * (v < head ? v : first + v - head); }
};
__device__ __forceinline__ bool key_seen(int j, int pos, int window, int keep) {
  return j <= pos && (window <= 0 || pos - j < window || j < keep);
}

// step_attention.hip: does it serve these operands, and its launch (the splits' sums follow in row_attention.hip)
template <typename T> bool step_attn_ok(const RowAttnArgs<T>& a);
template <typename T> hipError_t launch_step_attn(const RowAttnArgs<T>& a, int Tn, hipStream_t st);

}  // namespace lumen
