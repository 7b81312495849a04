// What the two selective-scan kernels share (scan.hip, scan_lanes.hip).
#pragma once

#include "mm_common.h"

namespace mm {
namespace scan {

// delta2 = delta' * log2(e), delta' = x <= cut ? softplus(x) : x.  cut is the reference's
// softplus cutoff 20 when delta_softplus is on, NaN when it is off (every comparison with
// NaN is false: delta' = x), so the flag costs no select of its own.  fp32 inputs keep
// log1p accuracy; fp16/bf16 inputs (whose own rounding is 2^-11 / 2^-8) use
// log2(1 + 2^m) directly.
template <int DT>
__device__ __forceinline__ float delta_log2(float x, float cut) {
  const float m = x * kLog2e;
  float l;
  if constexpr (DT == MM_F32) l = log1p_exp(x) * kLog2e;
  else l = log2_hw(1.0f + exp2_hw(m));
  return x <= cut ? l : m;
}

}  // namespace scan

namespace lscan {

// The scan with time across the lanes (scan_lanes.hip): whether a validated call takes it, and
// its launch.  ctl: the workspace's control block, whose status word the call clears; sum: the
// workspace's sum_bytes for segment summaries (none: time is not split).
bool preferred(const mm_scan_params* a, size_t sum_bytes);
int launch(const mm_scan_params* a, int* ctl, float* sum, size_t sum_bytes, void* stream);
// How it would run: time segments, and the waves per channel (0: scan.hip has the call).
int segments(const mm_scan_params* a, size_t sum_bytes, int* sw);

}  // namespace lscan
}  // namespace mm
