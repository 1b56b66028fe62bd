// Byte offsets of rows inside one head. Plain C++ beside HIP:
// tests/test_row_offset_cpu.py compiles this header by itself.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define CK_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define CK_HOST_DEVICE inline
#endif

namespace ck {
namespace pd {

// Offset of row min(row0 + step, rows - 1), rows of row_bytes bytes each. A head
// is shorter than 2^31 bytes, but a row past it (row0 runs on by up to a tile)
// may not be: its offset is unsigned, so that the minimum is taken of the value
// and not of its 32-bit wrap. row0 * row_bytes is one product per lane, step *
// row_bytes uniform.
CK_HOST_DEVICE uint32_t clamped_row_offset(int row0, int step, int row_bytes, int rows) {
  const uint32_t n = (uint32_t)row_bytes;
  const uint32_t at = (uint32_t)row0 * n + (uint32_t)step * n, last = (uint32_t)(rows - 1) * n;
  return at < last ? at : last;
}

}  // namespace pd
}  // namespace ck
