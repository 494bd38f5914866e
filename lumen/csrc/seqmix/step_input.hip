// sm_fill_step: a decode step's inputs into the static buffers of its captured graph, and the buffers' values
// for the padding rows, in one launch.  Up to three int32 and two int64 rows of n entries (padded to
// `bucket` with a value each) and the block table [n][width] into rows of `ld` entries.  What it replaces
// were five or six device copies and up to four fills of 2.4 - 4 us each, bound by their launches (a step
// of one row: 12 - 24 us; this launch 4.9).
#include <climits>

#include "seqmix.h"

using namespace lumen;

namespace {

constexpr int kKeep = INT_MIN;   // a padding value that stands for "left as it is"

struct FillArgs {
  const int* s32[3]; int* d32[3]; int p32[3];
  const long long* s64[2]; long long* d64[2]; long long p64[2];
  const int* table; int* dst; int width, ld;
  int n, bucket;
};

__global__ void __launch_bounds__(256) fill_step_kernel(const FillArgs a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < a.bucket) {
    const bool live = i < a.n;
#pragma unroll
    for (int k = 0; k < 3; ++k)
      if (a.d32[k] != nullptr && (live || a.p32[k] != kKeep)) a.d32[k][i] = live ? a.s32[k][i] : a.p32[k];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (a.d64[k] != nullptr && (live || k == 1)) a.d64[k][i] = live ? a.s64[k][i] : a.p64[k];
  }
  if (i < a.n * a.width) a.dst[(long long)(i / a.width) * a.ld + i % a.width] = a.table[i];
}

}  // namespace

extern "C" {

// a0 .. b2: three pairs of int32 rows (null: none) with their padding values; tok: int64 token ids (the
// padding rows' stay as they are); slot: int64 cache slots.  n <= bucket, n * width and bucket < 2^30.
hipError_t sm_fill_step(const int* a0, int* b0, int p0, const int* a1, int* b1, int p1, const int* a2,
                        int* b2, int p2, const long long* tok, long long* tok_dst,
                        const long long* slot, long long* slot_dst, long long slot_pad,
                        const int* table, int* dst, int width, int ld, int n, int bucket,
                        hipStream_t st) {
  if (bucket <= 0) return hipSuccess;
  if (n < 0 || n > bucket || width < 0 || width > ld || bucket >= (1 << 30) ||
      (long long)n * width >= (1LL << 30))
    return hipErrorInvalidValue;
  const FillArgs a{{a0, a1, a2}, {b0, b1, b2}, {p0, p1, p2}, {tok, slot}, {tok_dst, slot_dst},
                   {0, slot_pad}, table, dst, width, ld, n, bucket};
  const int most = n * width > bucket ? n * width : bucket;
  fill_step_kernel<<<(most + 255) / 256, 256, 0, st>>>(a);
  return hipGetLastError();
}

}  // extern "C"
