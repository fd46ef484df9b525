// Launches of the AWQ plan kernels that also take flat ranges or by-scale groups
// of other sizes than 128 columns: awq_decode_plan<kRanges> with bits 3 or 4, each
// in a translation unit of its own (awq_decode_flat_<kRanges>.hip), so that they
// compile side by side.
//
// A plan launches the first of them that has all its paths. With one kernel of
// every path for all such plans, the aligned weights beside a ragged one paid for
// it: that kernel's slab decode reloads 8136 spilled scalars (v_readlane), and the
// ones of aligned plans 2387 (<0>) and 2894 (<2>). The sets were chosen by that
// count: 3570, 3392, 3882 and 2668 for the first four below.
#pragma once

#include <hip/hip_runtime.h>

#include "mpserve_amd.h"

namespace mps {

// work: AwqWork records.
struct AwqFlatLaunch {
  const mps_awq_tensor *tensors;
  const void *work;
  int64_t nwork;
  const uint32_t *ckpt;
  uint32_t *status;
  int64_t out_delta;
  uint32_t *queue;
  unsigned grid;
  hipStream_t stream;
};

void launch_awq_flat_13(const AwqFlatLaunch &a);  // flat and row ranges, tiny buckets
void launch_awq_flat_14(const AwqFlatLaunch &a);  // flat ranges, ranges side by side, tiny buckets
void launch_awq_flat_11(const AwqFlatLaunch &a);  // every kind of range, no tiny buckets
void launch_awq_flat_30(const AwqFlatLaunch &a);  // as 14, by-scale groups of any size
void launch_awq_flat_31(const AwqFlatLaunch &a);  // every path

}  // namespace mps

// The body of such a unit (which includes awq_decode_device.h).
#define MPS_AWQ_FLAT_UNIT(MODE)                                                                                  \
  namespace mps {                                                                                                \
  void launch_awq_flat_##MODE(const AwqFlatLaunch &a) {                                                          \
    hipLaunchKernelGGL(awq_decode_plan<MODE>, dim3(a.grid), dim3(kAwqBlock), 0, a.stream, a.tensors,             \
                       static_cast<const AwqWork *>(a.work), a.nwork, a.ckpt, a.status, a.out_delta, a.queue);   \
  }                                                                                                              \
  }
