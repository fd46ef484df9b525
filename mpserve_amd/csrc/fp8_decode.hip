// FP8 + Huffman-sidecar -> BF16 decode: the C entry points, the plans, and the
// launches (device code: fp8_decode_device.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <queue>
#include <numeric>
#include <vector>

#include "fp8_decode_device.h"
#include "fp8_decode_flat.h"
#include "mps_common.h"

namespace mps {

namespace {

// ---------------------------------------------------------------------------
// Lane checkpoints: where each substream of a bucket stands at the first row
// of each of its row ranges, so that a plan can decode the ranges as separate
// work items (more work items than buckets when a plan has few).
//
// One workgroup per bucket to split (k = 1024 and fast paths: substream t's
// i-th element is row i / P, column c0 + t + (i % P) * K; flat ones: element
// t + i K of the rows end to end, ranges of slabs instead of rows). Thread t walks
// substream t through the code lengths only: the FP8 byte picks the table,
// the next 7 bits pick the length nibble, an ESC code skips 16 more bits (the
// lossless decode's semantics). It records its position after each range's
// last element. Row indices and table ids out of range stop the walk and mark
// the job failed (the plan then keeps the bucket whole, and its decode
// reports them).
// ---------------------------------------------------------------------------
struct SplitJob {
  int32_t tensor;
  int32_t K;           // substreams (k_eff)
  int32_t P;           // col_len / K (flat: 1, an element a slab)
  int32_t cl;          // col_len
  int32_t c0;          // first column
  int32_t range_rows;  // rows (flat: slabs) per range (the last range may have fewer)
  int32_t ranges;
  int32_t full;        // also rows 0 (the lanes' start bits) and `ranges` (their end bits)
  int64_t bit_base;
  int64_t out;         // first u32 of the job's checkpoints: [ranges - 1][K], or [ranges + 1][K] when full
  const int32_t *table_ids;
  const uint32_t *startbits;
  const int32_t *row_idx;
};

__global__ __launch_bounds__(kBlock) void fp8_checkpoints(const mps_fp8_tensor *__restrict__ tensors,
                                                          const SplitJob *__restrict__ jobs,
                                                          uint32_t *__restrict__ ckpt, uint32_t *__restrict__ failed) {
  __shared__ int32_t s_gid[256];
  __shared__ uint32_t s_lens[256 * kPacked / 4];  // packed length nibbles of each FP8 byte's table
  const SplitJob J = jobs[blockIdx.x];
  const mps_fp8_tensor &T = tensors[J.tensor];
  const int tid = threadIdx.x;
  if (tid < 256) {
    int32_t g = J.table_ids[tid];
    if (g < -1 || g >= T.num_tables) {
      failed[blockIdx.x] = 1u;
      g = -1;
    }
    s_gid[tid] = g;
  }
  __syncthreads();
  for (int i = tid; i < 256 * kPacked; i += kBlock) {
    const int32_t g = s_gid[i / kPacked];
    reinterpret_cast<uint8_t *>(s_lens)[i] = g >= 0 ? T.decode_lens[(int64_t)g * kPacked + i % kPacked] : 0u;
  }
  __syncthreads();
  if (tid >= J.K) return;
  const bool empty = T.bitstream_words <= 0;
  const uint32_t *__restrict__ bs32 = empty ? g_zero_chunks : reinterpret_cast<const uint32_t *>(T.bitstream);
  const uint64_t nchunks = empty ? 2u : (uint64_t)T.bitstream_words * 2u;
  const uint8_t *lens = reinterpret_cast<const uint8_t *>(s_lens);
  uint64_t pos = (uint64_t)J.bit_base + J.startbits[tid];
  const int64_t row0 = J.out + (J.full ? 0 : -(int64_t)J.K);  // where checkpoint row 0 would go
  if (J.full) {
    ckpt[row0 + tid] = J.startbits[tid];
    ckpt[row0 + (int64_t)J.ranges * J.K + tid] = J.startbits[tid + 1];
  }
  uint64_t cidx = ~0ull;
  uint32_t ca = 0, cb = 0;
  const int64_t per_range = (int64_t)J.range_rows * J.P;
  int64_t next = per_range;
  int32_t row_idx = 0;
  const int32_t dr = J.K / J.cl, dc = J.K - dr * J.cl;
  int32_t rr = tid / J.cl, cc = tid - rr * J.cl, seen = -1;  // element's row and column; the row whose index is held
  for (int j = 1; j < J.ranges; ++j, next += per_range) {
    for (int64_t i = next - per_range; i < next; ++i) {
      if (rr != seen) {
        seen = rr;
        row_idx = J.row_idx[rr];
        if (row_idx < 0 || row_idx >= T.n) {
          failed[blockIdx.x] = 1u;
          return;
        }
      }
      const uint8_t q = T.fp8[(int64_t)row_idx * T.m + J.c0 + cc];
      rr += dr;
      cc += dc;
      if (cc >= J.cl) {
        cc -= J.cl;
        ++rr;
      }
      const uint64_t c = pos >> 5;
      if (c != cidx) {
        cidx = c;
        ca = chunk_at(bs32, nchunks, c);
        cb = chunk_at(bs32, nchunks, c + 1);
      }
      const uint32_t peek = (uint32_t)(((((uint64_t)ca << 32) | cb) << (pos & 31u)) >> 57);
      const uint32_t nib = (lens[q * kPacked + (peek >> 1)] >> ((peek & 1u) * 4u)) & 0xFu;
      pos += (nib & 7u) + ((nib & 8u) ? 16u : 0u);
    }
    ckpt[row0 + (int64_t)j * J.K + tid] = (uint32_t)(pos - (uint64_t)J.bit_base);
  }
}

// ---------------------------------------------------------------------------
// Allocation-free batched decode. Some callers cannot allocate device memory
// (code under graph capture, tight serving loops). For them
// mps_fp8_decode_batch_noalloc decodes a list of tensors in one persistent
// launch, like a plan, with its descriptors and work records in `scratch`, a
// static device array of kScratchBytes that each device holds from module
// load to the end of the process. Buckets are not split into row ranges
// (that needs lane checkpoints, which a plan computes once).
//
// Layout of `scratch`: the descriptors (at most kMaxBatchTensors), then one
// 64-byte work record per bucket (at most kMaxBatchWork), then the decode
// launch's queue words in the last 256 bytes (zero from module load; each
// launch leaves them zero).
// ---------------------------------------------------------------------------
constexpr size_t kScratchBytes = size_t(4) << 20;
constexpr int64_t kMaxBatchTensors = 1024;
constexpr size_t kBatchWorkOff = ((sizeof(mps_fp8_tensor) * kMaxBatchTensors + 255) / 256) * 256;
constexpr size_t kBatchQueueOff = kScratchBytes - 256;
constexpr int64_t kMaxBatchWork = (int64_t)((kBatchQueueOff - kBatchWorkOff) / sizeof(WorkItem));

static __device__ __align__(256) uint8_t scratch[kScratchBytes];

// One work record per bucket, in tensor order. Every workgroup first scans the
// bucket counts of the (at most 1024) tensors in LDS, then each work-item
// writes the record of one bucket from that bucket's metadata.
__global__ __launch_bounds__(256) void fp8_batch_records(const mps_fp8_tensor *__restrict__ tensors, int32_t count,
                                                        int64_t total, WorkItem *__restrict__ work, bool flat_ok) {
  constexpr int kPer = kMaxBatchTensors / 256;  // tensors per work-item in the scan
  __shared__ int64_t s_first[kMaxBatchTensors + 1];
  __shared__ int64_t s_part[256];
  const int t = threadIdx.x;
  int64_t v[kPer], sum = 0;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    const int32_t i = t * kPer + j;
    v[j] = i < count ? tensors[i].num_buckets : 0;
    sum += v[j];
  }
  s_part[t] = sum;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {  // inclusive scan of the 256 partial sums
    const int64_t add = t >= off ? s_part[t - off] : 0;
    __syncthreads();
    s_part[t] += add;
    __syncthreads();
  }
  int64_t acc = s_part[t] - sum;  // exclusive prefix of this work-item's tensors
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    s_first[t * kPer + j] = acc;
    acc += v[j];
  }
  if (t == 255) s_first[kMaxBatchTensors] = acc;
  __syncthreads();
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  int32_t lo = 0, hi = count - 1;  // the tensor i with s_first[i] <= g < s_first[i + 1]
  while (lo < hi) {
    const int32_t mid = (lo + hi + 1) >> 1;
    if (s_first[mid] <= g) lo = mid;
    else hi = mid - 1;
  }
  const mps_fp8_tensor &T = tensors[lo];
  WorkItem w = bucket_item(T, g - s_first[lo], flat_ok);
  w.tensor = lo;
  work[g] = w;
}

// The device address of `scratch` on the current device, looked up once per
// device (the host-side name of a device array is not its address).
int scratch_ptr(uint8_t **out) {
  static std::mutex mu;
  static uint8_t *ptrs[kMaxDevices] = {};
  int dev = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(MPS_ERR_INVALID_ARGUMENT, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    ptrs[dev] = static_cast<uint8_t *>(p);
  }
  *out = ptrs[dev];
  return MPS_OK;
}

// Workgroups of a persistent launch on the current device: one per CU.
int persistent_grid(int64_t items, unsigned *grid) {
  int dev = 0, cus = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  if (cus < 1) cus = 1;
  *grid = (unsigned)(items < cus ? items : cus);
  return MPS_OK;
}

int check_tensor(const mps_fp8_tensor *t) {
  if (!t) return fail(MPS_ERR_INVALID_ARGUMENT, "tensor descriptor is NULL");
  if (t->n <= 0 || t->m <= 0) return fail(MPS_ERR_INVALID_ARGUMENT, "n,m must be > 0");
  if (t->k <= 0 || t->k > 1024)
    return fail(MPS_ERR_INVALID_ARGUMENT, "bucket_thread_startbit_u32 has invalid k (must be 1..1024)");
  if (t->num_buckets < 0 || t->num_buckets > INT32_MAX)
    return fail(MPS_ERR_INVALID_ARGUMENT, "invalid number of buckets");
  if (t->num_buckets > 0 && (!t->fp8 || !t->out || !t->bucket_table || !t->bucket_col_start || !t->bucket_col_len ||
                             !t->bucket_row_offsets || !t->bucket_thread_startbit || !t->bucket_bit_base))
    return fail(MPS_ERR_INVALID_ARGUMENT, "NULL sidecar pointer");
  return MPS_OK;
}

}  // namespace

// The status word of the single-tensor decodes (FP8 and AWQ) on a device: a
// module global, so each device holds its own copy, zero from module load to
// the end of the process, and no decode allocates it. It is per device, not
// per stream: decodes on different streams of one device OR into the same
// word (mps_fp8_read_status reads and clears it). Plans carry a word of their own.
static __device__ __align__(256) uint32_t g_status[64];

int status_word(int device, uint32_t **out) {
  static std::mutex mu;
  static uint32_t *words[kMaxDevices] = {};
  if (device < 0 || device >= kMaxDevices) return fail(MPS_ERR_INVALID_ARGUMENT, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!words[device]) {
    // The host-side name of a device global is not its device address: look
    // it up once per device, with that device current.
    int prev = 0;
    MPS_HIP_CHECK(hipGetDevice(&prev));
    if (prev != device) MPS_HIP_CHECK(hipSetDevice(device));
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(g_status));
    if (prev != device) (void)hipSetDevice(prev);
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(status word)");
    words[device] = static_cast<uint32_t *>(p);
  }
  *out = words[device];
  return MPS_OK;
}

std::string &last_error() {
  static thread_local std::string s;
  return s;
}

// Read a device status word and clear it, after `stream`'s work (synchronous).
int read_and_clear(int device, uint32_t *word, void *stream, const char *what, uint32_t *status_out) {
  int prev = 0;
  MPS_HIP_CHECK(hipGetDevice(&prev));
  if (prev != device) MPS_HIP_CHECK(hipSetDevice(device));
  uint32_t v = 0;
  const uint32_t zero = 0;
  hipError_t e = hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream));
  if (e == hipSuccess) e = hipMemcpy(&v, word, sizeof(v), hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(word, &zero, sizeof(zero), hipMemcpyHostToDevice);
  if (prev != device) (void)hipSetDevice(prev);
  if (e != hipSuccess) return hip_fail(e, what);
  *status_out = v;
  return MPS_OK;
}

}  // namespace mps

using namespace mps;

namespace {
constexpr size_t kAlign = 256;
// Work queues of a plan: one per stream that launches it (two u32 words each,
// 64 bytes apart), so that launches on different streams - a graph replay
// and an eager decode, a prefetch on a side stream - never share one.
constexpr int kPlanQueues = 32;
constexpr size_t kQueueStride = 64;
// A work item's set-up (tables into the LDS, the lanes' first loads, the
// pipeline's fill and drain) costs about as long as decoding this many
// elements; plans weigh items by their elements plus this. (Tuning builds:
// MPS_ITEM_SETUP.)
#ifndef MPS_ITEM_SETUP
#define MPS_ITEM_SETUP 65536
#endif
constexpr int64_t kItemSetup = MPS_ITEM_SETUP;
size_t align_up(size_t x) { return (x + kAlign - 1) & ~(kAlign - 1); }
// When items of these costs end, largest first, each on the CU that frees first.
int64_t greedy_end(std::vector<int64_t> &items, int64_t cus) {
  std::sort(items.begin(), items.end(), std::greater<int64_t>());
  std::priority_queue<int64_t, std::vector<int64_t>, std::greater<int64_t>> cu;
  for (int64_t c = 0; c < cus; ++c) cu.push(0);
  int64_t end = 0;
  for (int64_t x : items) {
    const int64_t t = cu.top() + x;
    cu.pop();
    cu.push(t);
    end = std::max(end, t);
  }
  return end;
}
}  // namespace

// A plan owns one device allocation: its status word, the tensor descriptors,
// the lane checkpoints of the buckets it split, the work records and (during
// creation) the checkpoint jobs and their failure flags.
// Tensors with k 256 or 512 substreams may have buckets for the slab path at that k.
inline bool slab_k(int64_t k) { return k == 256 || k == 512; }

struct mps_fp8_plan {
  void *d_block = nullptr;
  uint32_t *d_status = nullptr;
  // kPlanQueues work queues (work counter and exit count, zero between
  // launches); queue i serves streams[i], assigned at the stream's first launch.
  uint32_t *d_queue = nullptr;
  std::mutex mu;
  std::vector<void *> streams;
  mps_fp8_tensor *d_tensors = nullptr;
  WorkItem *d_work = nullptr;
  uint16_t *first_out = nullptr;  // the first tensor's output at creation (decode_into moves all by one offset)
  int64_t count = 0;
  int64_t work_items = 0;
  int device = 0;
  bool slab_k = false;      // some tensor has k 256 or 512: launch fp8_decode_plan<true, ...>
  bool flat = false;        // some bucket is flat: launch_flat_plan
  bool end_ticket = false;  // few work items a CU: tickets taken as items end (fp8_decode_plan<..., true>)
};

extern "C" {

#if MPS_TRACE_ITEMS
// The item trace's host side (instrumented builds only; not part of the product ABI).
int mps_item_trace_clear(void) {
  void *p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_item_trace)) != hipSuccess) return MPS_ERR_HIP;
  return hipMemset(p, 0, sizeof(g_item_trace)) == hipSuccess ? MPS_OK : MPS_ERR_HIP;
}
int mps_item_trace_read(uint64_t *dst, int64_t words) {
  if (!dst || words < (int64_t)(sizeof(g_item_trace) / 8)) return MPS_ERR_INVALID_ARGUMENT;
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(g_item_trace), sizeof(g_item_trace)) == hipSuccess ? MPS_OK
                                                                                                  : MPS_ERR_HIP;
}
#endif


const char *mps_last_error(void) { return last_error().c_str(); }

int mps_clock_rate_khz(int device, int64_t *khz_out) {
  if (!khz_out) return fail(MPS_ERR_INVALID_ARGUMENT, "khz_out is NULL");
  int v = 0;
  MPS_HIP_CHECK(hipDeviceGetAttribute(&v, hipDeviceAttributeClockRate, device));
  *khz_out = v;
  return MPS_OK;
}

int mps_stream_capture_id(void *stream, uint64_t *id_out) {
  last_error().clear();
  if (!id_out) return fail(MPS_ERR_INVALID_ARGUMENT, "id_out is NULL");
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  MPS_HIP_CHECK(hipStreamGetCaptureInfo(reinterpret_cast<hipStream_t>(stream), &s, &id));
  *id_out = s == hipStreamCaptureStatusActive ? (uint64_t)id : 0u;
  return MPS_OK;
}

int mps_fp8_decode(const mps_fp8_tensor *tensor, int64_t max_len, void *stream) {
  last_error().clear();
  if (max_len != kL) return fail(MPS_ERR_INVALID_ARGUMENT, "decode kernel is specialized: max_len must be 7");
  int rc = check_tensor(tensor);
  if (rc != MPS_OK) return rc;
  if (tensor->num_buckets == 0) return MPS_OK;
  int dev = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  uint32_t *status = nullptr;
  rc = status_word(dev, &status);
  if (rc != MPS_OK) return rc;
  unsigned grid = 0;
  rc = persistent_grid(tensor->num_buckets, &grid);
  if (rc != MPS_OK) return rc;
  // Few buckets for the CUs (k = 1024): each bucket shared by `parts`
  // workgroups, the largest power of two up to 16 (one wave each) that keeps
  // buckets x parts within the CUs.
  int32_t parts = 1;
  {
    int dev2 = 0, cus = 0;
    MPS_HIP_CHECK(hipGetDevice(&dev2));
    MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev2));
    if (tensor->k == kBlock)
      while (parts < kBlock / 64 && tensor->num_buckets * parts * 2 <= (int64_t)cus) parts *= 2;
    if (parts > 1) grid = (unsigned)(tensor->num_buckets * parts);
  }
  if (flat_rows(tensor->k, tensor->m))
    launch_flat_one(*tensor, status, parts, grid, reinterpret_cast<hipStream_t>(stream));
  else if (slab_k(tensor->k))
    hipLaunchKernelGGL((fp8_decode_one<true, false>), dim3(grid), dim3(kBlock), 0, reinterpret_cast<hipStream_t>(stream),
                       *tensor, status, parts);
  else
    hipLaunchKernelGGL((fp8_decode_one<false, false>), dim3(grid), dim3(kBlock), 0, reinterpret_cast<hipStream_t>(stream),
                       *tensor, status, parts);
  MPS_HIP_CHECK(hipGetLastError());
  return MPS_OK;
}

int mps_fp8_plan_create(const mps_fp8_tensor *tensors, int64_t count, void *stream, mps_fp8_plan **plan_out) {
  last_error().clear();
  if (!plan_out) return fail(MPS_ERR_INVALID_ARGUMENT, "plan_out is NULL");
  *plan_out = nullptr;
  if (count < 0 || (count > 0 && !tensors)) return fail(MPS_ERR_INVALID_ARGUMENT, "invalid tensor list");
  for (int64_t i = 0; i < count; ++i) {
    const int rc = check_tensor(&tensors[i]);
    if (rc != MPS_OK) return rc;
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // The sidecars may still be being written by work on the caller's stream:
  // everything below reads them after that work.
  MPS_HIP_CHECK(hipStreamSynchronize(st));
  // One work record per bucket.
  std::vector<WorkItem> bucket;
  std::vector<int64_t> elems;  // elements of each bucket (0: a bad bucket)
  std::vector<int32_t> roff, cstart, clen;
  std::vector<int64_t> bbase;
  for (int64_t i = 0; i < count; ++i) {
    const mps_fp8_tensor &T = tensors[i];
    const int64_t nb = T.num_buckets;
    if (nb == 0) continue;
    roff.resize((size_t)nb + 1);
    cstart.resize((size_t)nb);
    clen.resize((size_t)nb);
    bbase.resize((size_t)nb);
    MPS_HIP_CHECK(hipMemcpy(roff.data(), T.bucket_row_offsets, sizeof(int32_t) * (nb + 1), hipMemcpyDefault));
    MPS_HIP_CHECK(hipMemcpy(cstart.data(), T.bucket_col_start, sizeof(int32_t) * nb, hipMemcpyDefault));
    MPS_HIP_CHECK(hipMemcpy(clen.data(), T.bucket_col_len, sizeof(int32_t) * nb, hipMemcpyDefault));
    MPS_HIP_CHECK(hipMemcpy(bbase.data(), T.bucket_bit_base, sizeof(int64_t) * nb, hipMemcpyDefault));
    for (int64_t b = 0; b < nb; ++b) {
      const BucketShape s = bucket_shape(roff[b], roff[b + 1], cstart[b], clen[b], T, true);
      WorkItem w;
      w.tensor = (int32_t)i;
      w.c0 = cstart[b];
      w.cl = clen[b];
      w.rows = s.path == kPathFlat ? s.rows * clen[b] : s.rows;
      w.k_eff = s.k_eff;
      w.path = s.path;
      w.bit_base = bbase[b];
      w.table_ids = T.bucket_table + b * 256;
      w.startbits = T.bucket_thread_startbit + b * (T.k + 1);
      w.endbits = w.startbits + 1;
      w.row_idx = T.row_indices + (s.path != kPathBad ? roff[b] : 0);
      bucket.push_back(w);
      elems.push_back(s.path != kPathBad ? (int64_t)s.rows * clen[b] : 0);
    }
  }
  if (bucket.size() > (size_t)INT32_MAX) return fail(MPS_ERR_INVALID_ARGUMENT, "too many buckets for one plan");
  // Flat buckets send the whole plan to the kernels that have their path, which run
  // the aligned items 1% slower (more spills). A plan with few and short ones keeps
  // them on the general path: under 1/200 of its elements, at most 24 elements a
  // substream in the longest (the general path takes a bucket's substreams at some
  // 0.3 us an element, behind the larger items). An 8B layer beside a ragged weight,
  // general and flat: 64 x 1000 177.8, 179.5 us; 512 x 1000 178.7, 180.4; 2048 x 1000
  // (0.94%) 189.0, 181.7; 64 x 14000 (0.41%, 28 elements) 190.5, 177.3.
  {
    int64_t all = 0, flat = 0, longest = 0;
    for (size_t i = 0; i < bucket.size(); ++i) {
      all += elems[i];
      if (bucket[i].path != kPathFlat) continue;
      flat += elems[i];
      longest = std::max<int64_t>(longest, (elems[i] + bucket[i].k_eff - 1) / bucket[i].k_eff);
    }
    if (flat * 200 < all && longest <= 24)
      for (WorkItem &w : bucket) {
        if (w.path != kPathFlat) continue;
        w.path = kPathGeneric;
        w.rows /= w.cl;
      }
  }
  int device = 0, cus = 0;
  MPS_HIP_CHECK(hipGetDevice(&device));
  MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));

  // Row ranges. A plan whose buckets are few or uneven for the CUs (a layer,
  // a single tensor) would leave CUs idle behind its largest buckets: buckets
  // on the k = 1024 and fast paths larger than total / (2 * CUs) elements are
  // split into row ranges of at most that size (and at least 64 elements per
  // substream, 16 groups, so that a range's set-up stays small beside its
  // decode; fewer where CUs would be idle, min_lane below). Each range starts from lane checkpoints (fp8_checkpoints).
  //
  // A fast-path bucket with k_eff 256 or 512 fills only k_eff of a
  // workgroup's 1024 work-items, and its tables allow one workgroup per CU. So
  // it is cut into a multiple of S = 1024 / k_eff row ranges, and each work
  // item runs S of them side by side over the same tables (kMultiRange): the
  // unit of splitting is then an item of S ranges.
  //
  // A flat bucket is split the same way, into ranges of slabs instead of rows.
  //
  // An item's cost is the time its work-items take: the elements each one
  // decodes times 1024 (the elements of a k = 1024 item; S ranges side by
  // side cost one range's), plus kItemSetup for its set-up.
  //
  // Then the tail. The launch's queue hands the items out largest first
  // (fp8_decode_plan), and an item handed out when R elements of work remain
  // (it and the items after it) can end up to about its size minus R / CUs
  // after the others. Every item past the first CUs that exceeds
  // kTailRatio * R / CUs has its bucket split twice as fine, until none does
  // or none can be. Coarse items keep the set-ups few (each costs about as
  // much as decoding kItemSetup elements); the fine ones at the end fill the
  // CUs' last gaps.
#ifndef MPS_SPLIT_DIV
#define MPS_SPLIT_DIV 2
#endif
#ifndef MPS_TAIL_RATIO
#define MPS_TAIL_RATIO 3
#endif
  constexpr int64_t kTailRatio = MPS_TAIL_RATIO;
  const int64_t ncu = std::max(cus, 1);
  // Per bucket: ranges per item (1, or S for a multi-range bucket), the most
  // items it may be cut into, and its cost as one item (elements + set-up).
  std::vector<int64_t> per_item(bucket.size(), 1), maxi(bucket.size(), 1), whole_cost(bucket.size());
  // What a split-capable bucket is cut along, rows (flat: slabs), how many it
  // has, and the elements each substream has in one.
  auto is_flat = [&](size_t i) { return bucket[i].path == kPathFlat; };
  auto cuts = [&](size_t i) {
    const WorkItem &w = bucket[i];
    return is_flat(i) ? ((int64_t)w.rows + w.k_eff - 1) / w.k_eff : (int64_t)w.rows;
  };
  auto per_cut = [&](size_t i) { return is_flat(i) ? 1 : bucket[i].cl / bucket[i].k_eff; };
  // cost of `rows` rows (slabs) of split-capable bucket i decoded by one group of work-items
  auto rows_cost = [&](size_t i, int64_t rows) { return rows * (int64_t)per_cut(i) * 1024 + kItemSetup; };
  // Fewest elements per substream of a range: 64 where that gives every CU one
  // (4096 x 4096), fewer below, since a set-up costs a CU that would be idle
  // nothing; at least 16. Measured, k = 1024, a plan of one tensor, with 64 and now:
  // 512 x 4096 15.7 -> 10.0 us, 1024 x 4096 20.0 -> 12.3 (32: 13.5), 1000 x 3000
  // 20.1 -> 12.1, 2048 x 4096 19.6 -> 16.6; 2048 x 2048, k = 256: 20.8 -> 12.4 us.
  const int64_t all = std::accumulate(elems.begin(), elems.end(), (int64_t)0);
  const int64_t min_lane = std::min<int64_t>(64, std::max<int64_t>(16, all / (1024 * ncu)));
  for (size_t i = 0; i < bucket.size(); ++i) {
    const WorkItem &w = bucket[i];
    const int64_t ke = std::max<int64_t>(w.k_eff, 1);
    whole_cost[i] = (elems[i] + ke - 1) / ke * 1024 + kItemSetup;
    if ((w.path != kPathK1024 && w.path != kPathFast && !is_flat(i)) || cuts(i) < 2) continue;
    const int32_t P = per_cut(i);
    const int32_t min_rows = std::max<int32_t>(1, ((int32_t)min_lane + P - 1) / P);
    const int64_t maxr = std::max<int64_t>(1, cuts(i) / min_rows);
    const int64_t S = w.path != kPathK1024 && (w.k_eff == 256 || w.k_eff == 512) ? 1024 / w.k_eff : 1;
    // range rows ride in 8 bits of the work record (fast buckets hold <= 128 rows), slabs in 19
    if (S > 1 && maxr >= S && cuts(i) <= (is_flat(i) ? (1 << 19) - 1 : 255)) {
      per_item[i] = S;
      maxi[i] = maxr / S;
      whole_cost[i] = rows_cost(i, (cuts(i) + S - 1) / S);
    } else {
      maxi[i] = maxr;
    }
  }
  // Items of bucket i cut into ni items: their costs, largest first.
  auto for_items = [&](size_t i, int64_t ni, auto &&emit) {
    const int64_t rows = cuts(i);
    if (ni <= 1 && per_item[i] == 1) {
      emit(whole_cost[i]);
      return;
    }
    const int64_t rr = (rows + ni * per_item[i] - 1) / (ni * per_item[i]);  // rows per range
    const int64_t step = rr * per_item[i];                                    // rows per item
    for (int64_t r0 = 0; r0 < rows; r0 += step) emit(rows_cost(i, std::min(rr, rows - r0)));
  };
  int64_t total = 0;
  for (size_t i = 0; i < bucket.size(); ++i) total += whole_cost[i] - kItemSetup;
  const int64_t cap = std::max<int64_t>(total / (MPS_SPLIT_DIV * ncu), 1024 * min_lane);
  std::vector<int64_t> ni(bucket.size(), 1);  // items of each bucket
  for (size_t i = 0; i < bucket.size(); ++i) {
    const int64_t c = whole_cost[i] - kItemSetup;
    if (c > cap) ni[i] = std::min<int64_t>((c + cap - 1) / cap, maxi[i]);
  }
  {
    struct Piece {
      int64_t cost;
      size_t b;
    };
    std::vector<Piece> pieces;
    std::vector<char> bump(bucket.size());
    for (int iter = 0; iter < 64; ++iter) {
      pieces.clear();
      for (size_t i = 0; i < bucket.size(); ++i) for_items(i, ni[i], [&](int64_t c) { pieces.push_back({c, i}); });
      std::stable_sort(pieces.begin(), pieces.end(), [](const Piece &a, const Piece &c) { return a.cost > c.cost; });
      std::fill(bump.begin(), bump.end(), 0);
      bool changed = false;
      int64_t rest = 0;
      for (size_t q = pieces.size(); q-- > 0;) {
        rest += pieces[q].cost;
        const size_t b = pieces[q].b;
        if ((int64_t)q < ncu || bump[b] || ni[b] >= maxi[b]) continue;
        if ((double)pieces[q].cost * (double)ncu > (double)kTailRatio * (double)rest) {
          bump[b] = 1;
          ni[b] = std::min(maxi[b], ni[b] * 2);
          changed = true;
        }
      }
      if (!changed) break;
    }
  }
  // Splitting pays only where it shortens the launch: a tensor whose buckets
  // about match the CUs (a 70B gate_proj: 224 buckets of 1 M elements for 256
  // CUs) already ends after one bucket per CU, and its ranges would only add
  // set-ups. So the plan predicts both launches (items largest first, each to
  // the CU that frees first) and keeps the buckets whole (multi-range buckets:
  // one item) unless the split one ends sooner.
  {
    auto makespan = [&](const std::vector<int64_t> &items_of) {
      std::vector<int64_t> items;
      for (size_t i = 0; i < bucket.size(); ++i) for_items(i, items_of[i], [&](int64_t c) { items.push_back(c); });
      return greedy_end(items, ncu);
    };
    const std::vector<int64_t> whole(bucket.size(), 1);
    if (std::any_of(ni.begin(), ni.end(), [](int64_t x) { return x > 1; }) && makespan(whole) <= makespan(ni))
      ni = whole;
  }
  // Ranges of each bucket.
  std::vector<int64_t> nr(bucket.size());
  for (size_t i = 0; i < bucket.size(); ++i) nr[i] = ni[i] * per_item[i];
  std::vector<SplitJob> jobs;
  std::vector<size_t> job_of(bucket.size(), SIZE_MAX);
  int64_t ck_words = 0, max_items = 0;
  for (size_t i = 0; i < bucket.size(); ++i) {
    const WorkItem &w = bucket[i];
    ++max_items;
    if (nr[i] < 2) continue;
    int64_t ranges = nr[i];
    const int32_t range_rows = (int32_t)((cuts(i) + ranges - 1) / ranges);
    ranges = (cuts(i) + range_rows - 1) / range_rows;
    if (ranges < 2) continue;
    SplitJob j{};
    j.tensor = w.tensor;
    j.K = w.k_eff;
    j.P = per_cut(i);
    j.cl = w.cl;
    j.c0 = w.c0;
    j.range_rows = range_rows;
    j.ranges = (int32_t)ranges;
    j.bit_base = w.bit_base;
    j.out = ck_words;
    j.table_ids = w.table_ids;
    j.startbits = w.startbits;
    j.row_idx = w.row_idx;
    j.full = per_item[i] > 1 ? 1 : 0;
    job_of[i] = jobs.size();
    jobs.push_back(j);
    ck_words += (per_item[i] > 1 ? ranges + 1 : ranges - 1) * w.k_eff;
    max_items += ranges - 1;
  }

  // The plan's device block: the status word at 0, the work queues from
  // kAlign, then the descriptors, checkpoints, split jobs, their flags and the
  // work records.
  if (max_items >= kMaxQueueItems) return fail(MPS_ERR_INVALID_ARGUMENT, "too many work items for one plan");
  const size_t o_queues = kAlign;
  const size_t o_tensors = o_queues + align_up(kQueueStride * kPlanQueues);
  const size_t o_ckpt = o_tensors + align_up(sizeof(mps_fp8_tensor) * (size_t)count);
  const size_t o_jobs = o_ckpt + align_up(sizeof(uint32_t) * (size_t)ck_words);
  const size_t o_failed = o_jobs + align_up(sizeof(SplitJob) * jobs.size());
  const size_t o_work = o_failed + align_up(sizeof(uint32_t) * jobs.size());
  const size_t bytes = o_work + sizeof(WorkItem) * (size_t)max_items;
  auto *p = new (std::nothrow) mps_fp8_plan();
  if (!p) return fail(MPS_ERR_NO_MEMORY, "out of memory");
  p->count = count;
  p->slab_k = std::any_of(tensors, tensors + count, [](const mps_fp8_tensor &t) { return slab_k(t.k); });
  p->flat = std::any_of(bucket.begin(), bucket.end(), [](const WorkItem &w) { return w.path == kPathFlat; });
  p->device = device;
  p->first_out = count > 0 ? tensors[0].out : nullptr;
  hipError_t e = hipMalloc(&p->d_block, bytes);
  if (e != hipSuccess) {
    delete p;
    return hip_fail(e, "mps_fp8_plan_create");
  }
  auto cleanup = [&](hipError_t err) {
    (void)hipStreamSynchronize(st);
    (void)hipFree(p->d_block);
    delete p;
    return hip_fail(err, "mps_fp8_plan_create");
  };
  char *blk = static_cast<char *>(p->d_block);
  p->d_status = reinterpret_cast<uint32_t *>(blk);
  p->d_queue = reinterpret_cast<uint32_t *>(blk + o_queues);
  p->d_tensors = reinterpret_cast<mps_fp8_tensor *>(blk + o_tensors);
  p->d_work = reinterpret_cast<WorkItem *>(blk + o_work);
  uint32_t *d_ckpt = reinterpret_cast<uint32_t *>(blk + o_ckpt);
  // Status word and queues (zero), descriptors, jobs and their flags (zero): one copy, on the caller's stream.
  std::vector<char> head(o_work, 0);
  if (count > 0) std::memcpy(head.data() + o_tensors, tensors, sizeof(mps_fp8_tensor) * (size_t)count);
  if (!jobs.empty()) std::memcpy(head.data() + o_jobs, jobs.data(), sizeof(SplitJob) * jobs.size());
  e = hipMemcpyAsync(blk, head.data(), head.size(), hipMemcpyHostToDevice, st);
  std::vector<uint32_t> failed(jobs.size(), 0u);
  if (e == hipSuccess && !jobs.empty()) {
    hipLaunchKernelGGL(fp8_checkpoints, dim3((unsigned)jobs.size()), dim3(kBlock), 0, st, p->d_tensors,
                       reinterpret_cast<const SplitJob *>(blk + o_jobs), d_ckpt,
                       reinterpret_cast<uint32_t *>(blk + o_failed));
    e = hipGetLastError();
    if (e == hipSuccess)
      e = hipMemcpyAsync(failed.data(), blk + o_failed, sizeof(uint32_t) * jobs.size(), hipMemcpyDeviceToHost, st);
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  if (e != hipSuccess) return cleanup(e);

  // Runs of small flat buckets with the same tables (kFlatRun): a 128 x 128 block
  // holds 16 elements a substream, decoded in a fraction of its set-up, and the
  // blocks of one scale share their tables. Whole flat buckets of at most
  // kRunElems elements are grouped by table ids (read here, for tensors that
  // have such buckets) and cut into runs of the length whose launch is predicted
  // to end first: long runs save set-ups, short ones fill the CUs. A bucket after
  // a run's first costs about kRunFollow elements beside its own (its records,
  // start bits and first words, one round trip after the other).
  // Measured on 128 x 128 blocks: 4096 x 4096, 1024 buckets of 68 scales: 35 ->
  // 31 us at k = 1024, 90 -> 27 us at 256 (where four buckets run side by side);
  // 14336 x 4096: 145 -> 73 us and 299 -> 50 us.
  constexpr int64_t kRunElems = 65536, kRunFollow = 20480;
  std::vector<std::vector<size_t>> runs;
  std::vector<char> in_run(bucket.size(), 0);
  auto run_cost = [&](const WorkItem &w, int64_t n) {
    const int64_t S = 1024 / w.k_eff, rounds = (n + S - 1) / S;
    return kItemSetup + rounds * (((int64_t)w.rows + w.k_eff - 1) / w.k_eff * 1024) + (rounds - 1) * kRunFollow;
  };
  {
    std::vector<std::vector<size_t>> groups;
    std::vector<int32_t> ids;
    for (size_t i = 0; i < bucket.size();) {
      size_t end = i;
      bool some = false;
      auto small = [&](size_t b) { return is_flat(b) && job_of[b] == SIZE_MAX && bucket[b].rows <= kRunElems; };
      for (; end < bucket.size() && bucket[end].tensor == bucket[i].tensor; ++end) some = some || small(end);
      if (some) {
        const mps_fp8_tensor &T = tensors[bucket[i].tensor];
        ids.resize(256 * (size_t)T.num_buckets);
        e = hipMemcpy(ids.data(), T.bucket_table, sizeof(int32_t) * ids.size(), hipMemcpyDefault);
        if (e != hipSuccess) return cleanup(e);
        std::multimap<int32_t, size_t> by_first;  // a group by its first table id
        for (size_t b = i; b < end; ++b) {
          if (!small(b)) continue;
          const int32_t *row = ids.data() + 256 * (b - i);
          const int32_t *one = std::find_if(row, row + 256, [](int32_t g) { return g >= 0; });
          const int32_t key = one < row + 256 ? *one : -1;
          size_t g = SIZE_MAX;
          for (auto [it, last] = by_first.equal_range(key); it != last; ++it)
            if (std::equal(row, row + 256, ids.data() + 256 * (groups[it->second][0] - i))) g = it->second;
          if (g == SIZE_MAX) {
            by_first.emplace(key, g = groups.size());
            groups.emplace_back();
          }
          groups[g].push_back(b);
        }
      }
      i = end;
    }
    // the other items' costs, then each candidate length's
    std::vector<int64_t> others;
    for (size_t i = 0; i < bucket.size(); ++i)
      if (!(is_flat(i) && job_of[i] == SIZE_MAX && bucket[i].rows <= kRunElems))
        for_items(i, ni[i], [&](int64_t c) { others.push_back(c); });
    auto cut = [](size_t n, size_t len) { return (n + len - 1) / len; };  // runs of a group
    size_t best = 1;
    int64_t best_end = INT64_MAX;
    for (size_t len : {1, 2, 3, 4, 6, 8, 12, 16, 24, 32}) {
      if (groups.empty()) break;
      std::vector<int64_t> items(others);
      for (const auto &g : groups) {
        const size_t n = cut(g.size(), len);
        for (size_t r = 0; r < n; ++r)
          items.push_back(run_cost(bucket[g[0]], (int64_t)(g.size() * (r + 1) / n - g.size() * r / n)));
      }
      const int64_t end = greedy_end(items, ncu);
      if (end < best_end) {
        best_end = end;
        best = len;
      }
    }
    size_t followers = 0;
    for (const auto &g : groups) {
      const size_t n = cut(g.size(), best);
      for (size_t r = 0; r < n && followers < (size_t(1) << 20) - 64; ++r) {
        const size_t from = g.size() * r / n, to = g.size() * (r + 1) / n;
        if (to - from < 2) continue;
        runs.emplace_back(g.begin() + from, g.begin() + to);
        followers += to - from - 1;
        for (size_t b : runs.back()) in_run[b] = 1;
      }
    }
  }

  // Work items (buckets and ranges), largest first, the order in which the
  // launch's queue hands them out, by the cost above; then the runs' other buckets.
  std::vector<WorkItem> work, followers;
  std::vector<int64_t> cost;
  for (const auto &r : runs) {
    WorkItem x = bucket[r[0]];
    x.path = (int32_t)(kPathFlat | kFlatRun | ((uint32_t)r.size() << 8));
    x.k_eff = (int32_t)((uint32_t)x.k_eff | ((uint32_t)followers.size() << kFlatSlabShift));
    for (size_t j = 1; j < r.size(); ++j) followers.push_back(bucket[r[j]]);
    work.push_back(x);
    cost.push_back(run_cost(bucket[r[0]], (int64_t)r.size()));
  }
  for (size_t i = 0; i < bucket.size(); ++i) {
    const WorkItem &w = bucket[i];
    if (in_run[i]) continue;
    if (job_of[i] == SIZE_MAX || failed[job_of[i]]) {
      work.push_back(w);
      cost.push_back(per_item[i] > 1 ? rows_cost(i, cuts(i)) : whole_cost[i]);  // a failed walk: one range
      continue;
    }
    const SplitJob &j = jobs[job_of[i]];
    const uint32_t *ck = d_ckpt + j.out;
    if (is_flat(i)) {
      // slabs [r * range_rows, + S * range_rows) of the bucket: elements, first row and column
      const int64_t S = j.full ? 1024 / j.K : 1, step = (int64_t)j.range_rows * j.K;
      for (int64_t r = 0; r < j.ranges; r += S) {
        WorkItem x = w;
        const int64_t at = r * step;
        x.rows = (int32_t)std::min<int64_t>(S * step, w.rows - at);
        x.row_idx = w.row_idx + at / w.cl;
        x.path = (int32_t)(kPathFlat | (j.full ? kMultiRange : 0) | ((uint32_t)(at % w.cl) << 8));
        x.k_eff = j.full ? w.k_eff | (j.range_rows << kFlatSlabShift) : w.k_eff;
        x.startbits = j.full ? ck + r * j.K : r == 0 ? w.startbits : ck + (r - 1) * j.K;
        x.endbits = j.full ? ck + (r + 1) * j.K : r + 1 == j.ranges ? w.endbits : ck + r * j.K;
        work.push_back(x);
        cost.push_back(rows_cost(i, std::min<int64_t>(j.range_rows, cuts(i) - r * j.range_rows)));
      }
      continue;
    }
    if (j.full) {
      // S ranges an item; range r's start bits are checkpoint row r, its end bits row r + 1
      const int32_t S = 1024 / j.K;
      for (int32_t r = 0; r < j.ranges; r += S) {
        WorkItem x = w;
        x.path = kPathFast | kMultiRange | (j.range_rows << 8);
        x.rows = w.rows - r * j.range_rows;
        x.row_idx = w.row_idx + (int64_t)r * j.range_rows;
        x.startbits = ck + (int64_t)r * j.K;
        x.endbits = ck + (int64_t)(r + 1) * j.K;
        work.push_back(x);
        cost.push_back(rows_cost(i, std::min(j.range_rows, x.rows)));
      }
      continue;
    }
    for (int32_t r = 0; r < j.ranges; ++r) {
      WorkItem x = w;
      x.rows = std::min(j.range_rows, w.rows - r * j.range_rows);
      x.row_idx = w.row_idx + (int64_t)r * j.range_rows;
      x.startbits = r == 0 ? w.startbits : ck + (int64_t)(r - 1) * j.K;
      x.endbits = r + 1 == j.ranges ? w.endbits : ck + (int64_t)r * j.K;
      work.push_back(x);
      cost.push_back(rows_cost(i, x.rows));
    }
  }
  {
    std::vector<size_t> order(work.size());
    for (size_t j = 0; j < order.size(); ++j) order[j] = j;
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t c) { return cost[a] > cost[c]; });
    std::vector<WorkItem> sorted(work.size());
    for (size_t j = 0; j < order.size(); ++j) sorted[j] = work[order[j]];
    work.swap(sorted);
  }
  p->work_items = (int64_t)work.size();
  work.insert(work.end(), followers.begin(), followers.end());
  // Ticket mode. With the ticket taken in an item's set-up, a workgroup holds
  // its next item for the whole current one: right for many items of about one
  // size (a full model: ~100 a CU), where the next record then loads during the
  // drain. With few items a CU (a layer, a tensor: split items of mixed sizes),
  // a workgroup that drew a long item would keep its next one from a workgroup
  // that frees sooner, so the ticket is taken as the item ends (measured: 8B
  // layer -2.5%, 70B layer -4.7%; the full model +0.3% that way).
  p->end_ticket = p->work_items < 16 * (int64_t)ncu;
  if (!work.empty()) {
    e = hipMemcpyAsync(p->d_work, work.data(), sizeof(WorkItem) * work.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return cleanup(e);
  }
  *plan_out = p;
  return MPS_OK;
}

namespace {
// The work queue of `stream` in the plan: the one it was given at its first
// launch, or the next free one. A launch leaves its queue as it found it, so
// launches on one stream (in stream order) can share one; launches on
// different streams may overlap and each has its own. A graph captured on a
// stream replays with that stream's queue.
int plan_queue(mps_fp8_plan *plan, void *stream, uint32_t **queue) {
  std::lock_guard<std::mutex> lock(plan->mu);
  size_t i = 0;
  while (i < plan->streams.size() && plan->streams[i] != stream) ++i;
  if (i == plan->streams.size()) {
    if (i >= (size_t)kPlanQueues)
      return fail(MPS_ERR_RUNTIME, "a decode plan serves at most %d streams", kPlanQueues);
    plan->streams.push_back(stream);
  }
  *queue = plan->d_queue + i * (kQueueStride / sizeof(uint32_t));
  return MPS_OK;
}

int plan_launch(mps_fp8_plan *plan, int64_t out_delta, uint32_t *status, void *stream) {
  if (plan->work_items == 0) return MPS_OK;
  unsigned grid = 0;
  int rc = persistent_grid(plan->work_items, &grid);
  if (rc != MPS_OK) return rc;
  uint32_t *queue = nullptr;
  rc = plan_queue(plan, stream, &queue);
  if (rc != MPS_OK) return rc;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, reinterpret_cast<hipStream_t>(stream), plan->d_tensors,
                       plan->d_work, plan->work_items, status, out_delta, queue);
  };
  if (plan->flat) {
    launch_flat_plan(plan->end_ticket, plan->d_tensors, plan->d_work, plan->work_items, status, out_delta, queue, grid,
                     reinterpret_cast<hipStream_t>(stream));
  } else if (plan->slab_k) {
    if (plan->end_ticket) launch(fp8_decode_plan<true, true, false>);
    else launch(fp8_decode_plan<true, false, false>);
  } else {
    if (plan->end_ticket) launch(fp8_decode_plan<false, true, false>);
    else launch(fp8_decode_plan<false, false, false>);
  }
  MPS_HIP_CHECK(hipGetLastError());
  return MPS_OK;
}
}  // namespace

int mps_fp8_plan_decode(mps_fp8_plan *plan, void *stream) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  return plan_launch(plan, 0, plan->d_status, stream);
}

int mps_fp8_plan_decode_into(mps_fp8_plan *plan, uint16_t *out, void *stream) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (!out) return fail(MPS_ERR_INVALID_ARGUMENT, "out is NULL");
  if (plan->count == 0) return MPS_OK;
  uint32_t *status = nullptr;
  const int rc = status_word(plan->device, &status);
  if (rc != MPS_OK) return rc;
  const intptr_t delta = reinterpret_cast<intptr_t>(out) - reinterpret_cast<intptr_t>(plan->first_out);
  if (delta % (intptr_t)sizeof(uint16_t) != 0)
    return fail(MPS_ERR_INVALID_ARGUMENT, "out must be 2-byte aligned like the plan's outputs");
  return plan_launch(plan, (int64_t)(delta / (intptr_t)sizeof(uint16_t)), status, stream);
}

int mps_fp8_plan_info(const mps_fp8_plan *plan, int64_t *work_items, int64_t *lds_bytes) {
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (work_items) *work_items = plan->work_items;
  if (lds_bytes) *lds_bytes = (int64_t)kLdsWords * 4;
  return MPS_OK;
}

int mps_fp8_plan_read_status(mps_fp8_plan *plan, void *stream, uint32_t *status_out) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (!status_out) return fail(MPS_ERR_INVALID_ARGUMENT, "status_out is NULL");
  return read_and_clear(plan->device, plan->d_status, stream, "mps_fp8_plan_read_status", status_out);
}

int mps_fp8_plan_destroy(mps_fp8_plan *plan) {
  if (!plan) return MPS_OK;
  if (plan->d_block) (void)hipFree(plan->d_block);
  delete plan;
  return MPS_OK;
}

int mps_fp8_read_status(int device, void *stream, uint32_t *status_out) {
  last_error().clear();
  if (!status_out) return fail(MPS_ERR_INVALID_ARGUMENT, "status_out is NULL");
  uint32_t *word = nullptr;
  const int rc = status_word(device, &word);
  if (rc != MPS_OK) return rc;
  return read_and_clear(device, word, stream, "mps_fp8_read_status", status_out);
}


int mps_fp8_decode_batch_noalloc(const mps_fp8_tensor *tensors, int64_t count, int64_t max_len, void *stream) {
  last_error().clear();
  if (max_len != kL) return fail(MPS_ERR_INVALID_ARGUMENT, "decode kernel is specialized: max_len must be 7");
  if (count < 0 || (count > 0 && !tensors)) return fail(MPS_ERR_INVALID_ARGUMENT, "invalid tensor list");
  if (count > kMaxBatchTensors)
    return fail(MPS_ERR_INVALID_ARGUMENT,
                "mps_fp8_decode_batch_noalloc: %lld tensors exceed its static scratch (at most %lld)",
                (long long)count, (long long)kMaxBatchTensors);
  int64_t total = 0;
  for (int64_t i = 0; i < count; ++i) {
    const int rc = check_tensor(&tensors[i]);
    if (rc != MPS_OK) return rc;
    total += tensors[i].num_buckets;
  }
  if (total > kMaxBatchWork)
    return fail(MPS_ERR_INVALID_ARGUMENT,
                "mps_fp8_decode_batch_noalloc: %lld buckets exceed its static scratch (at most %lld)",
                (long long)total, (long long)kMaxBatchWork);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // The descriptors travel by a copy from the caller's host array. Captured
  // into a graph, that copy would re-read the host address on every replay,
  // long after the array is gone: a capturing stream is refused, before any
  // copy or launch.
  {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess || cs != hipStreamCaptureStatusNone)
      return fail(MPS_ERR_INVALID_ARGUMENT,
                  "mps_fp8_decode_batch_noalloc cannot run on a capturing stream (its descriptors are copied "
                  "from host memory); create a decode plan before the capture and launch that instead");
  }
  if (total == 0) return MPS_OK;
  int dev = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  uint32_t *status = nullptr;
  int rc = status_word(dev, &status);
  if (rc != MPS_OK) return rc;
  uint8_t *base = nullptr;
  rc = scratch_ptr(&base);
  if (rc != MPS_OK) return rc;
  auto *d_tensors = reinterpret_cast<mps_fp8_tensor *>(base);
  auto *d_work = reinterpret_cast<WorkItem *>(base + kBatchWorkOff);
  // The descriptors are read from the caller's host array before this returns.
  MPS_HIP_CHECK(hipMemcpyAsync(d_tensors, tensors, sizeof(mps_fp8_tensor) * (size_t)count, hipMemcpyHostToDevice, st));
  const bool flat = std::any_of(tensors, tensors + count, [](const mps_fp8_tensor &t) { return flat_rows(t.k, t.m); });
  hipLaunchKernelGGL(fp8_batch_records, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, d_tensors,
                     (int32_t)count, total, d_work, flat);
  MPS_HIP_CHECK(hipGetLastError());
  unsigned grid = 0;
  rc = persistent_grid(total, &grid);
  if (rc != MPS_OK) return rc;
  const bool sk = std::any_of(tensors, tensors + count, [](const mps_fp8_tensor &t) { return slab_k(t.k); });
  if (flat)
    launch_flat_plan(false, d_tensors, d_work, total, status, 0, reinterpret_cast<uint32_t *>(base + kBatchQueueOff), grid,
                     st);
  else if (sk)
    hipLaunchKernelGGL((fp8_decode_plan<true, false, false>), dim3(grid), dim3(kBlock), 0, st, d_tensors, d_work, total,
                       status, (int64_t)0, reinterpret_cast<uint32_t *>(base + kBatchQueueOff));
  else
    hipLaunchKernelGGL((fp8_decode_plan<false, false, false>), dim3(grid), dim3(kBlock), 0, st, d_tensors, d_work, total,
                       status, (int64_t)0, reinterpret_cast<uint32_t *>(base + kBatchQueueOff));
  MPS_HIP_CHECK(hipGetLastError());
  return MPS_OK;
}

}  // extern "C"
