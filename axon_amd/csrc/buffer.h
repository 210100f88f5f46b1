// Rows of a matrix as a buffer: a lane's load has a place of its own in it, in bytes, and may have a scalar one beside it.
//
// A lane whose own place lies behind the buffer's bytes reads nothing and gets zeros.  What a scalar place counts in that check is
// described in more than one way (not at all, or taken off the bytes, with no word on one that is larger than they are), so nothing
// rests on it: a lane that has something to read finds it within the bytes with its scalar place added, and a lane that
// has not lies behind them without it.  Where lanes read on behind their row (numbers that nobody uses), the buffer itself
// begins further on and the scalar place is 0.  Plain functions: a test on the host goes through the places of every lane.
#pragma once

#include <stddef.h>

#ifdef __HIPCC__
#define AXK_BUFFER_FN __host__ __device__ inline __attribute__((always_inline))
#else
#define AXK_BUFFER_FN inline
#endif

struct BufferRows {
  size_t first;        // the element of the matrix that it begins at
  unsigned bytes;
};

// Rows m .. M - 1 of K elements, `stride` (at least K) apart.  Behind the last row: the last row, for the lanes whose place is in the
// first row; the places of the others lie behind it.
AXK_BUFFER_FN BufferRows buffer_rows(int m, int M, size_t stride, int K, unsigned elem_bytes) {
  const int from = m < M ? m : M - 1;
  const size_t bytes = ((size_t)(M - 1 - from) * stride + K) * elem_bytes;
  return BufferRows{(size_t)from * stride, bytes < 0xfffffff0u ? (unsigned)bytes : 0xfffffff0u};
}
