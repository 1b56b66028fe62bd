// How large one launch may be. Plain C++: tests/test_launch_limits_cpu.py compiles
// this header by itself.
#pragma once

#include <stdint.h>

namespace ck {

// Workgroups of `threads` threads that one launch may hold: HIP takes fewer than
// 2^32 work items (hip_runtime_api.h, hipModuleLaunchKernel).
constexpr int64_t max_workgroups(int threads) { return (((int64_t)1 << 32) - 1) / threads; }

// launch(first, count) over slices of n parts, each `per_part` workgroups of
// `threads` threads, so that no launch is too large; the first status that is not
// 0 (CK_OK) ends it and is returned.
template <class F>
int launch_slices(int64_t n, int64_t per_part, int threads, F&& launch) {
  const int64_t fit = max_workgroups(threads) / per_part;
  const int64_t step = fit < 1 ? 1 : fit;
  int status = 0;
  for (int64_t i = 0; i < n && status == 0; i += step) status = launch(i, n - i < step ? n - i : step);
  return status;
}

}  // namespace ck
