// Row addresses of the elementwise scans' loads (mg_elementwise.h).  Plain integer
// arithmetic, host and device, so that the offsets can be enumerated on a CPU.
//
// Loads are issued unconditionally -- a load under a condition became a branch of its own,
// with a wait for the register it replaced -- so a step past the sequence end loads the
// last row again and is made neutral where its value matters.  (linear_scan forward at
// (16, 4096, 1024) 184 -> 176 us, the signed gates 195 -> 186 us, the MinGRU gates, with one
// exponential where there were two, 193 -> 152 us.)  Every offset handed out here is
// therefore one of a row that exists.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

// The row to load for step t of the batch row whose first row is b0: t, or the last one
// past the sequence end.
__host__ __device__ __forceinline__ int64_t ew_row(int64_t b0, int64_t t, int64_t T) {
  return b0 + (t < T ? t : T - 1);
}

// Element offsets of the rows a wave loads, ew_row(b0, t0, T), ew_row(b0, t0 + 1, T), ...,
// times ld: one scalar add a row instead of a 64-bit product.
struct EwRows {
  int64_t off, ld, left, first;
  __host__ __device__ __forceinline__ EwRows(int64_t b0, int64_t t0, int64_t T, int64_t ld_)
      : off(ew_row(b0, t0, T) * ld_), ld(ld_), left(T - 1 - t0), first(b0 * ld_) {}
  __host__ __device__ __forceinline__ int64_t next() {
    const int64_t o = off;
    off += left > 0 ? ld : 0;
    --left;
    return o;
  }
  // The row before the one at offset `o`, or `o` itself where that is the sequence's first
  // row.  The row decides and not the step: with T = 1 every step past the end loads the
  // first row.
  __host__ __device__ __forceinline__ int64_t before(int64_t o) const {
    return o > first ? o - ld : o;
  }
};
