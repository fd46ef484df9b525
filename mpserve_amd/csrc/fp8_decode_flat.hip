// The FP8 decode kernels that also take flat buckets: those whose column range
// is no multiple of their substreams (fp8_decode_device.h).
#include "fp8_decode_device.h"
#include "fp8_decode_flat.h"

namespace mps {

void launch_flat_one(const mps_fp8_tensor &tensor, uint32_t *status, int32_t parts, unsigned grid, hipStream_t stream) {
  hipLaunchKernelGGL((fp8_decode_one<true, true>), dim3(grid), dim3(kBlock), 0, stream, tensor, status, parts);
}

void launch_flat_plan(bool end_ticket, const mps_fp8_tensor *tensors, const void *work, int64_t nwork, uint32_t *status,
                      int64_t out_delta, uint32_t *queue, unsigned grid, hipStream_t stream) {
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, stream, tensors, static_cast<const WorkItem *>(work), nwork,
                       status, out_delta, queue);
  };
  if (end_ticket) launch(fp8_decode_plan<true, true, true>);
  else launch(fp8_decode_plan<true, false, true>);
}

}  // namespace mps
