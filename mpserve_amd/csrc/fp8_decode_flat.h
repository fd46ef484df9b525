// Launches of the decode kernels that also take flat buckets
// (fp8_decode_flat.hip, a translation unit of its own: these kernels hold every
// path and compile as long as all the others together).
#pragma once

#include <hip/hip_runtime.h>

#include "mpserve_amd.h"

namespace mps {

// Does a tensor with k substreams and m columns have buckets for these kernels
// when its buckets span whole rows? (Column-range buckets may also be flat.)
inline bool flat_rows(int64_t k, int64_t m) { return (k == 256 || k == 512 || k == 1024) && m % k != 0; }

// fp8_decode_one and fp8_decode_plan (work: WorkItem records), flat items included.
void launch_flat_one(const mps_fp8_tensor &tensor, uint32_t *status, int32_t parts, unsigned grid, hipStream_t stream);
void launch_flat_plan(bool end_ticket, const mps_fp8_tensor *tensors, const void *work, int64_t nwork, uint32_t *status,
                      int64_t out_delta, uint32_t *queue, unsigned grid, hipStream_t stream);

}  // namespace mps
