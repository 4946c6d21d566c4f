// Document masks: the [lo, hi) of every position's document, a maximal run of
// equal ids, from the ids themselves (no counterpart in the reference, whose
// README.md:219 lists document masking as future work).
//
// Latency-bound: the data is 8 to 16 bytes a position, but each value depends
// on the whole row.  One workgroup per batch row sweeps it in chunks of
// kThreads x kPer positions, forwards for lo (the last document start at or
// before a position) and backwards for hi (the next start after it), each chunk
// one load, one scan over the workgroup (a wave scan by lane shifts, then the
// wave totals through LDS) and one store.  One row of 8192 int64 ids (a single
// chunk, loaded once) takes 13 us, where the sixteen tensor operations that built
// the same bounds (two of them scans of 23 us) took 95 us of GPU time and about
// 140 us to issue.
#include "flexatt_device.h"
#include "flexatt_kernels.h"

namespace flexatt {

namespace {
constexpr int kThreads = 1024, kPer = 8;
constexpr int kWaves = kThreads / 64;

// Exclusive scan over the workgroup of one int per thread.  DIR +1: max over
// the threads before this one; -1: min over the threads after it; `none` where
// there is no such thread.
template <int DIR>
__device__ __forceinline__ int scan_exclusive(int v, int none, int* tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto op = [](int a, int b) { return DIR > 0 ? max(a, b) : min(a, b); };
  int x = v;
#pragma unroll
  for (int d = 1; d < 64; d *= 2) {
    const int y = DIR > 0 ? __shfl_up(x, d) : __shfl_down(x, d);
    if (DIR > 0 ? lane >= d : lane + d < 64) x = op(x, y);
  }
  __syncthreads();  // the previous use of tot is over
  if (lane == (DIR > 0 ? 63 : 0)) tot[wave] = x;
  int e = DIR > 0 ? __shfl_up(x, 1) : __shfl_down(x, 1);
  if (lane == (DIR > 0 ? 0 : 63)) e = none;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    if (DIR > 0 ? w < wave : w > wave) e = op(e, tot[w]);
  return e;
}

template <class I>
__global__ __launch_bounds__(kThreads) void doc_bounds_kernel(const I* ids, int S, int* bounds) {
  __shared__ int tot[kWaves];
  __shared__ int s_carry;
  ids += (int64_t)blockIdx.x * S;
  bounds += (int64_t)blockIdx.x * S * 2;
  constexpr int CH = kThreads * kPer;
  const int nch = (S - 1) / CH + 1;
  I id[kPer + 1];  // ids of positions p0 - 1 .. p0 + kPer - 1 (clamped into the row)
  auto load = [&](int64_t p0) {
#pragma unroll
    for (int e = 0; e <= kPer; ++e) {
      const int64_t i = p0 + e - 1;
      id[e] = ids[i < 0 ? 0 : i < S ? i : S - 1];
    }
  };
  int carry = 0;  // the last start before this chunk
  for (int c = 0; c < nch; ++c) {
    const int64_t p0 = (int64_t)c * CH + threadIdx.x * kPer;
    load(p0);
    int lo[kPer], last = -1;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
      if (p0 + e < S && p0 + e > 0 && id[e + 1] != id[e]) last = (int)p0 + e;
      lo[e] = last;
    }
    const int before = max(carry, scan_exclusive<1>(last, -1, tot));
#pragma unroll
    for (int e = 0; e < kPer; ++e)
      if (p0 + e < S) bounds[2 * (p0 + e)] = max(lo[e], before);
    if (threadIdx.x == kThreads - 1) s_carry = max(last, before);
    __syncthreads();
    carry = s_carry;
  }
  carry = S;  // the next start after this chunk
  for (int c = nch - 1; c >= 0; --c) {
    const int64_t p0 = (int64_t)c * CH + threadIdx.x * kPer;
    if (nch > 1) load(p0);  // (a single chunk is still in registers)
    int hi[kPer], next = 0x7fffffff;
#pragma unroll
    for (int e = kPer - 1; e >= 0; --e) {
      hi[e] = next;
      if (p0 + e < S && p0 + e > 0 && id[e + 1] != id[e]) next = (int)p0 + e;
    }
    const int after = min(carry, scan_exclusive<-1>(next, 0x7fffffff, tot));
#pragma unroll
    for (int e = 0; e < kPer; ++e)
      if (p0 + e < S) bounds[2 * (p0 + e) + 1] = min(hi[e], after);
    if (threadIdx.x == 0) s_carry = min(next, after);
    __syncthreads();
    carry = s_carry;
  }
}
}  // namespace

hipError_t doc_bounds_run(const void* ids, int ids_bytes, int B, int S, int* bounds, hipStream_t st) {
  const dim3 grid(B), block(kThreads);
  switch (ids_bytes) {
    case 1: hipLaunchKernelGGL(doc_bounds_kernel<uint8_t>, grid, block, 0, st, (const uint8_t*)ids, S, bounds); break;
    case 2: hipLaunchKernelGGL(doc_bounds_kernel<uint16_t>, grid, block, 0, st, (const uint16_t*)ids, S, bounds); break;
    case 4: hipLaunchKernelGGL(doc_bounds_kernel<uint32_t>, grid, block, 0, st, (const uint32_t*)ids, S, bounds); break;
    case 8: hipLaunchKernelGGL(doc_bounds_kernel<uint64_t>, grid, block, 0, st, (const uint64_t*)ids, S, bounds); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace flexatt
