// The AWQ plan kernel with every path, flat ranges among them (awq_decode_device.h):
// a translation unit of its own, so that it compiles beside the others.
#include "awq_decode_device.h"

namespace mps {

void launch_awq_flat_plan(const mps_awq_tensor *tensors, const void *work, int64_t nwork, const uint32_t *ckpt,
                          uint32_t *status, int64_t out_delta, uint32_t *queue, unsigned grid, hipStream_t stream) {
  hipLaunchKernelGGL(awq_decode_plan<15>, dim3(grid), dim3(kAwqBlock), 0, stream, tensors,
                     static_cast<const AwqWork *>(work), nwork, ckpt, status, out_delta, queue);
}

}  // namespace mps
