// AWQ int4 + Huffman-sidecar -> BF16 decode: the C entry points, the plans, and
// the launches (device code: awq_decode_device.h).
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

#include "awq_decode_device.h"
#include "awq_decode_flat.h"
#include "mps_common.h"

namespace mps {
namespace {

template <int kSplit>
__global__ __launch_bounds__(kAwqBlock) void awq_decode_kernel(mps_awq_tensor T, uint32_t *status) {
  // Row offsets (the slab path's queue) first: the tables' base then rides in
  // the LDS instructions' offset field, and the queue's address needs no add.
  __shared__ __attribute__((aligned(16))) uint32_t lds[kRowSlots + kLutEntries];
  uint32_t *s_base = lds, *lut = lds + kRowSlots;
  awq_bucket<kSplit>(T, blockIdx.x / kSplit, (int)(blockIdx.x % kSplit), lut, s_base, status);
}

// Lane checkpoints of a slab-path row bucket split into row ranges: where each
// substream stands at the first row of every range after the first, found by
// walking it through the code lengths once (the int4 value picks the table, the
// next 11 bits the length nibble; a nibble of 15 is an 11-bit ESC code and 16
// raw bits). One workgroup per bucket to split; lane t < k walks substream t,
// whose element (row r, block p) is column c0 + t + k p of the bucket's row r. A
// row index or table id out of range stops the walk and marks the job failed
// (the plan then keeps the bucket whole, and its decode reports them). A `full`
// job (ranges side by side, k 256 or 512) also writes rows 0 (the substreams'
// start bits) and `ranges` (their end bits). A by-scale job's ranges are ranges
// of slabs (`range_rows` slabs of k / group_size groups each; `rows`: the groups).
struct AwqSplitJob {
  int32_t tensor, bucket, P, rows;
  int32_t c0, range_rows, ranges;
  int32_t full;  // 1: also the rows at both ends; 2: so, and the ranges are slabs of a flat bucket
  int64_t out;  // first u32 of the job's checkpoints: [ranges - 1][k], or [ranges + 1][k] when full
};

__global__ __launch_bounds__(kAwqBlock) void awq_checkpoints(const mps_awq_tensor *__restrict__ tensors,
                                                             const AwqSplitJob *__restrict__ jobs,
                                                             uint32_t *__restrict__ ckpt,
                                                             uint32_t *__restrict__ failed) {
  __shared__ int32_t s_gid[16];
  __shared__ uint8_t s_lens[16 * kAwqPacked];  // packed length nibbles of each int4 value's table
  const AwqSplitJob J = jobs[blockIdx.x];
  const mps_awq_tensor &T = tensors[J.tensor];
  const int tid = threadIdx.x;
  if (tid < 16) {
    int32_t g = T.bucket_table[(int64_t)J.bucket * 16 + tid];
    if (g < -1 || g >= T.num_tables) {
      failed[blockIdx.x] = 1u;
      g = -1;
    }
    s_gid[tid] = g;
  }
  __syncthreads();
  for (int i = tid; i < 16 * kAwqPacked; i += kAwqBlock) {
    const int32_t g = s_gid[i / kAwqPacked];
    s_lens[i] = g >= 0 ? T.decode_lens[(int64_t)g * kAwqPacked + i % kAwqPacked] : 0xFFu;  // missing: all ESC
  }
  __syncthreads();
  const bool empty = T.bitstream_words <= 0;
  const uint32_t *__restrict__ bs32 = empty ? g_awq_zero_chunks : reinterpret_cast<const uint32_t *>(T.bitstream);
  const uint64_t nchunks = empty ? 2u : (uint64_t)T.bitstream_words * 2u;
  const int32_t K = (int32_t)T.k;
  if (tid >= K) return;
  const uint64_t bit_base = (uint64_t)T.bucket_bit_base[J.bucket];
  const int32_t ra = T.bucket_row_offsets[J.bucket];
  const uint32_t *sb = T.bucket_thread_startbit + (int64_t)J.bucket * (K + 1);
  const int64_t row0 = J.out - (J.full ? 0 : K);  // where checkpoint row 0 would go
  if (J.full) {
    ckpt[row0 + tid] = sb[tid];
    ckpt[row0 + (int64_t)J.ranges * K + tid] = sb[tid + 1];
  }
  uint64_t pos = bit_base + sb[tid];
  uint64_t cidx = ~0ull;
  uint32_t ca = 0, cb = 0;
  auto step = [&](uint32_t q) {  // past the code of one element with int4 value q
    const uint64_t c = pos >> 5;
    if (c != cidx) {
      cidx = c;
      ca = chunk_at(bs32, nchunks, c);
      cb = chunk_at(bs32, nchunks, c + 1);
    }
    const uint32_t peek = (uint32_t)(((((uint64_t)ca << 32) | cb) << (pos & 31u)) >> (64 - kAwqL));
    const uint32_t nib = (s_lens[q * kAwqPacked + (peek >> 1)] >> ((peek & 1u) * 4u)) & 0xFu;
    pos += nib == 15u ? (uint64_t)kAwqEscLow : (uint64_t)nib;
  };
  if (J.full == 2) {
    // flat (rows or groups of any width cl): substream t's element in slab i is
    // element t + i K of the rows end to end
    const int32_t cl = T.group_col_start ? (int32_t)T.group_size : T.bucket_col_len[J.bucket];
    const int32_t dr = K / cl, dc = K - dr * cl;
    int32_t rr = tid / cl, cc = tid - rr * cl, seen = -1;
    int64_t base = 0;
    // The walk stops at the last range's start; the rows after it are checked here, so that a
    // bucket with a bad one keeps its per-lane record, which drops that row alone.
    for (int32_t r = tid; r < T.bucket_row_offsets[J.bucket + 1] - ra; r += K) {
      const int32_t row = T.row_indices[ra + r], c0 = T.group_col_start ? T.group_col_start[ra + r] : J.c0;
      if (row < 0 || row >= T.n || c0 < 0 || (int64_t)c0 + cl > T.m) failed[blockIdx.x] = 1u;
    }
    for (int j = 1; j < J.ranges; ++j) {
      for (int32_t i = (j - 1) * J.range_rows; i < j * J.range_rows; ++i) {
        if (rr != seen) {
          seen = rr;
          const int32_t row = T.row_indices[ra + rr], c0 = T.group_col_start ? T.group_col_start[ra + rr] : J.c0;
          if (row < 0 || row >= T.n || c0 < 0 || (int64_t)c0 + cl > T.m) {
            failed[blockIdx.x] = 1u;
            return;
          }
          base = (int64_t)row * T.m + c0;
        }
        step(T.int4[base + cc] & 15u);
        rr += dr;
        cc += dc;
        if (cc >= cl) {
          cc -= cl;
          ++rr;
        }
      }
      ckpt[row0 + (int64_t)j * K + tid] = (uint32_t)(pos - bit_base);
    }
    return;
  }
  if (T.group_col_start) {
    // by-scale (J.rows groups of gs columns): ranges of J.range_rows slabs of K / gs
    // groups; substream t's element in slab i is column t % gs of group (K / gs) i + t / gs
    const int32_t gs = (int32_t)T.group_size, gps = K / gs, gsub = tid / gs, col = tid - gsub * gs;
    for (int j = 1; j < J.ranges; ++j) {
      for (int32_t i = (j - 1) * J.range_rows; i < j * J.range_rows; ++i) {
        const int32_t g = gps * i + gsub;
        if (g >= J.rows) break;
        const int32_t row = T.row_indices[ra + g], c0 = T.group_col_start[ra + g];
        if (row < 0 || row >= T.n || c0 < 0 || (int64_t)c0 + gs > T.m) {
          failed[blockIdx.x] = 1u;
          return;
        }
        step(T.int4[(int64_t)row * T.m + c0 + col] & 15u);
      }
      ckpt[row0 + (int64_t)j * K + tid] = (uint32_t)(pos - bit_base);
    }
    return;
  }
  for (int j = 1; j < J.ranges; ++j) {
    for (int32_t r = (j - 1) * J.range_rows; r < j * J.range_rows; ++r) {
      const int32_t row = T.row_indices[ra + r];
      if (row < 0 || row >= T.n) {
        failed[blockIdx.x] = 1u;
        return;
      }
      const uint8_t *qrow = T.int4 + (int64_t)row * T.m + J.c0 + tid;
      for (int32_t p = 0; p < J.P; ++p) step(qrow[(int64_t)p * K] & 15u);
    }
    ckpt[row0 + (int64_t)j * K + tid] = (uint32_t)(pos - bit_base);
  }
}

int check_awq(const mps_awq_tensor *t) {
  if (!t) return fail(MPS_ERR_INVALID_ARGUMENT, "tensor is NULL");
  if (t->n <= 0 || t->m <= 0) return fail(MPS_ERR_INVALID_ARGUMENT, "n,m must be > 0");
  if (t->n * t->m >= ((int64_t)1 << 31)) return fail(MPS_ERR_INVALID_ARGUMENT, "tensor too large (n*m >= 2^31)");
  if (t->k <= 0 || t->k > kAwqBlock)
    return fail(MPS_ERR_INVALID_ARGUMENT, "bucket_thread_startbit_u32 has invalid k (must be 1..1024)");
  if (t->num_buckets < 0 || t->num_buckets >= ((int64_t)1 << 31))
    return fail(MPS_ERR_INVALID_ARGUMENT, "invalid bucket count");
  if (t->num_buckets > 0 && (!t->int4 || !t->bucket_table || !t->bucket_row_offsets || !t->row_indices ||
                             !t->bucket_thread_startbit || !t->bucket_bit_base || !t->out))
    return fail(MPS_ERR_INVALID_ARGUMENT, "NULL sidecar array");
  if (t->group_col_start) {
    if (t->group_size <= 0 || t->group_size > t->m) return fail(MPS_ERR_INVALID_ARGUMENT, "group_size must be in (0,m]");
  } else if (t->num_buckets > 0 && (!t->bucket_col_start || !t->bucket_col_len)) {
    return fail(MPS_ERR_INVALID_ARGUMENT, "NULL sidecar array");
  }
  if (t->num_tables > 0 && (!t->decode_syms || !t->decode_lens))
    return fail(MPS_ERR_INVALID_ARGUMENT, "NULL sidecar array");
  return MPS_OK;
}

}  // namespace
}  // namespace mps

using namespace mps;

// A plan owns one device allocation: its status word, the tensor descriptors,
// the work records, and the split jobs and lane checkpoints of its row ranges.
// Work queues of a plan: one per stream that launches it (two u32 words each,
// 64 bytes apart), so that launches on different streams never share one.
constexpr int kAwqPlanQueues = 32;
constexpr size_t kAwqQueueStride = 64;

struct mps_awq_plan {
  int device = 0;
  int64_t count = 0, nwork = 0;
  // kAwqPlanQueues work queues (zero between launches); queue i serves
  // streams[i], assigned at the stream's first launch
  uint32_t *d_queue = nullptr;
  std::mutex mu;
  std::vector<void *> streams;
  uint16_t *first_out = nullptr;  // the first tensor's output at creation (decode_into moves from it)
  void *d_block = nullptr;
  uint32_t *d_status = nullptr;
  mps_awq_tensor *d_tensors = nullptr;
  AwqWork *d_work = nullptr;
  uint32_t *d_ckpt = nullptr;  // lane checkpoints of the row buckets split into ranges
  int64_t splits = 0;          // row buckets split into ranges
  // bit 0: some work record is a row range (kind 2); bit 1: ranges side by side
  // (kind 3); bit 2: tiny buckets (kind 0 with `tiny`); bit 3: flat ranges (kind 4);
  // bit 4: by-scale groups of other sizes than 128 columns
  int ranges_mode = 0;
};

extern "C" {

#if MPS_TRACE_ITEMS
// The record trace's host side (instrumented builds only; not part of the product ABI).
int mps_awq_trace_clear(void) {
  void *p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(g_awq_trace)) != hipSuccess) return MPS_ERR_HIP;
  return hipMemset(p, 0, sizeof(g_awq_trace)) == hipSuccess ? MPS_OK : MPS_ERR_HIP;
}
int mps_awq_trace_read(uint64_t *dst, int64_t words) {
  if (!dst || words < (int64_t)(sizeof(g_awq_trace) / 8)) return MPS_ERR_INVALID_ARGUMENT;
  return hipMemcpyFromSymbol(dst, HIP_SYMBOL(g_awq_trace), sizeof(g_awq_trace)) == hipSuccess ? MPS_OK : MPS_ERR_HIP;
}
#endif


int mps_awq_decode(const mps_awq_tensor *tensor, int64_t max_len, void *stream) {
  last_error().clear();
  if (max_len != kAwqL) return fail(MPS_ERR_INVALID_ARGUMENT, "AWQ bucket decode kernel is specialized: max_len must be 11");
  int rc = check_awq(tensor);
  if (rc != MPS_OK) return rc;
  if (tensor->num_buckets == 0) return MPS_OK;
  int dev = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  uint32_t *status = nullptr;
  rc = status_word(dev, &status);
  if (rc != MPS_OK) return rc;
  // Fewer buckets than CUs: split each bucket's lanes over 2 workgroups.
  int cus = 0;
  MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int64_t B = tensor->num_buckets;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (B >= cus)
    hipLaunchKernelGGL(awq_decode_kernel<1>, dim3((unsigned)B), dim3(kAwqBlock), 0, s, *tensor, status);
  else
    hipLaunchKernelGGL(awq_decode_kernel<2>, dim3((unsigned)(2 * B)), dim3(kAwqBlock / 2), 0, s, *tensor, status);
  MPS_HIP_CHECK(hipGetLastError());
  return MPS_OK;
}

int mps_awq_plan_create(const mps_awq_tensor *tensors, int64_t count, void *stream, mps_awq_plan **plan_out) {
  last_error().clear();
  if (!plan_out) return fail(MPS_ERR_INVALID_ARGUMENT, "plan_out is NULL");
  *plan_out = nullptr;
  if (count < 0 || count >= ((int64_t)1 << 31) || (count > 0 && !tensors))
    return fail(MPS_ERR_INVALID_ARGUMENT, "invalid tensor list");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // The sidecars may still be being written by work on the caller's stream.
  MPS_HIP_CHECK(hipStreamSynchronize(st));
  int dev = 0, cus = 0;
  MPS_HIP_CHECK(hipGetDevice(&dev));
  MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  // Work records (AwqWork). Slab-eligible buckets get one record each (kind 1),
  // except that by-scale ones take in the following buckets with identical
  // table ids (nsub in all); the others run in runs of up to 1024 / k
  // consecutive buckets of one tensor with identical table ids (one scale) and
  // at most kRowSlots / 4 rows each, so they can share a workgroup's tables
  // (kind 0).
  std::vector<AwqWork> base;
  std::vector<int32_t> roff, clen, cst, btab, gcol, grow;
  // Elements a by-scale slab record's run of buckets may hold: a CU's share
  // of the plan (records go out largest first, so the large ones run early
  // and small ones fill the end; half a share measured 0.9% slower on an 8B
  // layer, a quarter 4.8%).
  int64_t all_elems = 0;
  for (int64_t i = 0; i < count; ++i)
    if (tensors[i].n > 0 && tensors[i].m > 0 && tensors[i].n < ((int64_t)1 << 31) && tensors[i].m < ((int64_t)1 << 31))
      all_elems += tensors[i].n * tensors[i].m;
#ifndef MPS_AWQ_RUN_DIV
#define MPS_AWQ_RUN_DIV 1
#endif
  const int64_t run_cap = std::max<int64_t>(1, all_elems / (MPS_AWQ_RUN_DIV * (int64_t)std::max(cus, 1)));
  // row-layout slab records: rows, P, column start; k for the records of
  // buckets whose ranges may run side by side (0: others)
  std::vector<int32_t> rows_of_rec, p_of_rec, c0_of_rec, k_of_rec, gps_of_rec;
  const char *slab_env = std::getenv("MPSERVE_AWQ_SLAB");
  const bool slab_on = !(slab_env && slab_env[0] == '0');
  int64_t total = 0;
  for (int64_t i = 0; i < count; ++i) {
    const mps_awq_tensor &T = tensors[i];
    int rc = check_awq(&T);
    if (rc != MPS_OK) return rc;
    const int64_t B = T.num_buckets;
    if (B == 0) continue;
    roff.resize((size_t)B + 1);
    btab.resize((size_t)B * 16);
    MPS_HIP_CHECK(hipMemcpy(roff.data(), T.bucket_row_offsets, sizeof(int32_t) * (B + 1), hipMemcpyDefault));
    MPS_HIP_CHECK(hipMemcpy(btab.data(), T.bucket_table, sizeof(int32_t) * B * 16, hipMemcpyDefault));
    if (!T.group_col_start) {
      clen.resize((size_t)B);
      MPS_HIP_CHECK(hipMemcpy(clen.data(), T.bucket_col_len, sizeof(int32_t) * B, hipMemcpyDefault));
    }
    // The slab path (k = 1024: by-scale with groups slab_group takes, or row buckets of
    // 1..128 rows over P >= 4 blocks of 1024 columns) loads int4 bytes as dwords
    // and stores 8 bytes a lane: every group or column range must start on a
    // 4-element boundary and the buffers must be aligned to match.
    bool slab_tensor = slab_on && T.k == kAwqBlock && (!T.group_col_start || slab_group(T.group_size, T.k)) &&
                       T.m % 4 == 0 && (reinterpret_cast<uintptr_t>(T.int4) & 3u) == 0 && (reinterpret_cast<uintptr_t>(T.out) & 7u) == 0;
    // By-scale sidecars with k 256 or 512 and such groups: buckets cut into ranges
    // of slabs (k / group_size groups each), 1024 / k ranges side by side a record.
    bool bmulti_tensor = slab_on && (T.k == 256 || T.k == 512) && T.group_col_start &&
                         slab_group(T.group_size, T.k) && T.m % 4 == 0 && (reinterpret_cast<uintptr_t>(T.int4) & 3u) == 0 &&
                         (reinterpret_cast<uintptr_t>(T.out) & 7u) == 0;
    if ((slab_tensor || bmulti_tensor) && T.group_col_start && T.num_row_indices > 0) {
      gcol.resize((size_t)T.num_row_indices);
      MPS_HIP_CHECK(hipMemcpy(gcol.data(), T.group_col_start, sizeof(int32_t) * T.num_row_indices, hipMemcpyDefault));
      bool aligned = std::all_of(gcol.begin(), gcol.end(), [](int32_t c) { return (c & 3) == 0; });
      // The slab path drops a bucket (a range, a wave's groups) with a bad group. Other sizes than
      // 128 columns came to it from the per-lane path, which drops that group alone: with a bad
      // group among them they stay there.
      if (aligned && T.group_size != 128) {
        grow.resize(gcol.size());
        MPS_HIP_CHECK(hipMemcpy(grow.data(), T.row_indices, sizeof(int32_t) * T.num_row_indices, hipMemcpyDefault));
        for (size_t g = 0; g < grow.size() && aligned; ++g)
          aligned = grow[g] >= 0 && grow[g] < T.n && gcol[g] >= 0 && gcol[g] + T.group_size <= T.m;
      }
      slab_tensor = slab_tensor && aligned;
      bmulti_tensor = bmulti_tensor && aligned;
    }
    // Row buckets with k 256 or 512 and P = col_len / k a multiple of 4: the
    // slab path at stride k, with 1024 / k row ranges side by side a record
    // (kind 3), else a bucket fills only k of the 1024 work-items.
    const bool multi_tensor = slab_on && (T.k == 256 || T.k == 512) && !T.group_col_start && T.m % 4 == 0 &&
                              (reinterpret_cast<uintptr_t>(T.int4) & 3u) == 0 &&
                              (reinterpret_cast<uintptr_t>(T.out) & 7u) == 0;
    // Flat: every other bucket with k 256, 512 or 1024 substreams whose rows (or
    // wide by-scale groups) a range can hold 128 of and still be 32 slabs long.
    const bool flat_tensor = slab_on && (T.k == 256 || T.k == 512 || T.k == 1024) &&
                             (!T.group_col_start || T.group_size >= kAwqBlock);
    if ((slab_tensor || multi_tensor || flat_tensor) && !T.group_col_start) {
      cst.resize((size_t)B);
      MPS_HIP_CHECK(hipMemcpy(cst.data(), T.bucket_col_start, sizeof(int32_t) * B, hipMemcpyDefault));
    }
    auto rows_of = [&](int64_t b) { return std::max<int64_t>(0, (int64_t)roff[(size_t)b + 1] - roff[(size_t)b]); };
    auto elems_of = [&](int64_t b) {
      const int64_t cols = T.group_col_start ? T.group_size : (int64_t)clen[(size_t)b];
      return rows_of(b) * std::max<int64_t>(0, cols);
    };
    const int64_t maxsub = T.k <= kAwqBlock / 4 ? 4 : T.k <= kAwqBlock / 2 ? 2 : 1;
    const int64_t row_cap = kRowSlots / 4;
    // (cst holds the column starts only for a slab-eligible row-layout tensor)
    auto slab_ok = [&](int64_t bb) {
      const bool shape =
          slab_tensor &&
          (T.group_col_start
               ? rows_of(bb) >= T.k / T.group_size && rows_of(bb) <= kSlabMaxSlabs * (T.k / T.group_size)
               : rows_of(bb) >= 1 && rows_of(bb) <= 128 && clen[(size_t)bb] >= 4 * kAwqBlock &&
                     clen[(size_t)bb] % kAwqBlock == 0 && cst[(size_t)bb] >= 0 && (cst[(size_t)bb] & 3) == 0 &&
                     (int64_t)cst[(size_t)bb] + clen[(size_t)bb] <= T.m);
      return shape && roff[(size_t)bb] >= 0 && roff[(size_t)bb + 1] <= T.num_row_indices;
    };
    auto multi_ok = [&](int64_t bb) {
      const int64_t kk = T.k;
      if (roff[(size_t)bb] < 0 || roff[(size_t)bb + 1] > T.num_row_indices) return false;
      // by-scale: at least 32 slabs (below that the set-up outweighs the decode, and
      // runs of same-scale buckets on the per-lane path share one set-up)
      if (T.group_col_start) return bmulti_tensor && rows_of(bb) >= 32 * (kk / T.group_size) && rows_of(bb) <= 1024;
      return multi_tensor && rows_of(bb) >= 1 && rows_of(bb) <= 128 && clen[(size_t)bb] >= 4 * kk &&
             clen[(size_t)bb] % (4 * kk) == 0 && cst[(size_t)bb] >= 0 && (cst[(size_t)bb] & 3) == 0 &&
             (int64_t)cst[(size_t)bb] + clen[(size_t)bb] <= T.m;
    };
    auto flat_slabs = [&](int64_t bb) -> int64_t {  // most slabs a range of the bucket may span
      const int64_t cols = T.group_col_start ? T.group_size : (int64_t)clen[(size_t)bb];
      return (kFlatMaxRows - 2) * cols / T.k;
    };
    auto flat_ok = [&](int64_t bb) {
      if (!flat_tensor || roff[(size_t)bb] < 0 || roff[(size_t)bb + 1] > T.num_row_indices) return false;
      const int64_t cols = T.group_col_start ? T.group_size : (int64_t)clen[(size_t)bb], all = elems_of(bb);
      return cols >= 4 && cols < kFlatMaxCols && all > T.k && all < ((int64_t)1 << 31) &&
             (T.group_col_start || (cst[(size_t)bb] >= 0 && (int64_t)cst[(size_t)bb] + cols <= T.m)) &&
             flat_slabs(bb) >= std::min<int64_t>(32, (all + T.k - 1) / T.k);
    };
    auto same_tables = [&](int64_t x, int64_t y) {
      return std::equal(btab.begin() + x * 16, btab.begin() + x * 16 + 16, btab.begin() + y * 16);
    };
    int64_t b = 0;
    while (b < B) {
      total += elems_of(b);
      if (slab_ok(b)) {
        // by-scale: a run of following buckets with identical table ids (one
        // scale's group-cap chunks) joins the record, up to run_cap elements
        int64_t run = 1, elems = elems_of(b);
        if (T.group_col_start) {
          while (b + run < B && elems + elems_of(b + run) <= run_cap && slab_ok(b + run) && same_tables(b, b + run)) {
            elems += elems_of(b + run);
            total += elems_of(b + run);
            ++run;
          }
        }
        base.push_back(AwqWork{(int32_t)i, (int32_t)b, (int32_t)run, 1, 0, 0, 1, 0, 0, elems});
        rows_of_rec.push_back(T.group_col_start ? 0 : (int32_t)rows_of(b));
        p_of_rec.push_back(T.group_col_start ? 0 : clen[(size_t)b] / kAwqBlock);
        c0_of_rec.push_back(T.group_col_start ? 0 : cst[(size_t)b]);
        k_of_rec.push_back(0);
        gps_of_rec.push_back(0);
        b += run;
        continue;
      }
      if (multi_ok(b)) {
        // a per-lane record (kind 0), replaced by side-by-side ranges once its
        // checkpoint walk succeeds
        base.push_back(AwqWork{(int32_t)i, (int32_t)b, 1, 0, 0, 0, 1, 0, 0, elems_of(b)});
        rows_of_rec.push_back((int32_t)rows_of(b));  // rows, or groups (by-scale: P = 0)
        p_of_rec.push_back(T.group_col_start ? 0 : (int32_t)(clen[(size_t)b] / T.k));
        c0_of_rec.push_back(T.group_col_start ? 0 : cst[(size_t)b]);
        k_of_rec.push_back((int32_t)T.k);
        gps_of_rec.push_back(T.group_col_start ? (int32_t)(T.k / T.group_size) : 0);
        ++b;
        continue;
      }
      if (flat_ok(b)) {
        // likewise; its units are slabs, at most p_of_rec a range (gps -1 marks it)
        base.push_back(AwqWork{(int32_t)i, (int32_t)b, 1, 0, 0, 0, 1, 0, 0, elems_of(b)});
        rows_of_rec.push_back((int32_t)((elems_of(b) + T.k - 1) / T.k));
        p_of_rec.push_back((int32_t)std::min<int64_t>(flat_slabs(b), 1 << 30));
        c0_of_rec.push_back(T.group_col_start ? 0 : cst[(size_t)b]);
        k_of_rec.push_back((int32_t)T.k);
        gps_of_rec.push_back(-1);
        ++b;
        continue;
      }
      int64_t nsub = 1, elems = elems_of(b);
      // Tiny: every bucket of the record codes at most one element a lane (k =
      // 1024 only: with k 256 / 512 such buckets run in same-scale runs that
      // share one table set-up, and the tiny path measured 2.9% slower there)
      bool tiny = T.k == kAwqBlock && elems_of(b) <= T.k;
      if (rows_of(b) <= row_cap) {
        while (nsub < maxsub && b + nsub < B && rows_of(b + nsub) <= row_cap && !multi_ok(b + nsub) &&
               !flat_ok(b + nsub) && same_tables(b, b + nsub)) {
          elems += elems_of(b + nsub);
          total += elems_of(b + nsub);
          tiny = tiny && elems_of(b + nsub) <= T.k;
          ++nsub;
        }
      }
      base.push_back(AwqWork{(int32_t)i, (int32_t)b, (int32_t)nsub, 0, 0, 0, 1, tiny ? 1 : 0, 0, elems});
      rows_of_rec.push_back(0);
      p_of_rec.push_back(0);
      c0_of_rec.push_back(0);
      k_of_rec.push_back(0);
      gps_of_rec.push_back(0);
      b += nsub;
    }
  }
  // Row ranges: a slab-path row bucket with more than total / (2 * CUs) elements
  // is split into row ranges of at least 64 elements a lane, each started from
  // lane checkpoints that one walk over the bucket's substreams finds (16: 1024 x
  // 4096, k = 1024, 20.2 -> 24.0 us: more table set-ups than CUs).
  // A bucket with k 256 or 512 (k_of_rec) is always cut, into up to 1024 / k
  // ranges a record (one record per total / (2 * CUs) elements), which share
  // the record's set-up.
  const int64_t target = std::max<int64_t>(1, total / (2 * (int64_t)std::max(cus, 1)));
  // Fewest elements a lane of a range that shares its record's set-up, or of a flat
  // one: 64 where that gives every CU one (4096 x 4096), fewer in smaller plans,
  // whose idle CUs pay a set-up for nothing; at least 16, below which a range is all
  // set-up. One weight's plan, the per-record rule of 64 and now: 1024 x 4096, k =
  // 256, 27.8 -> 17.7 us; 2048 x 2048, k = 256, 28.0 -> 17.5; 2048 x 4096, k = 512,
  // 26.5 -> 20.6; 128-column groups, 1024 x 4096, k = 256, 25.7 -> 22.6 us.
  const int64_t min_lane =
      std::min<int64_t>(64, std::max<int64_t>(16, total / (kAwqBlock * (int64_t)std::max(cus, 1))));
  std::vector<AwqSplitJob> jobs;
  std::vector<size_t> job_rec;  // the base record each job splits
  int64_t ck_words = 0;
  for (size_t r = 0; r < base.size(); ++r) {
    const AwqWork &w = base[r];
    const int32_t rows = rows_of_rec[r], P = p_of_rec[r];
    if (k_of_rec[r] > 0) {
      // units: rows, or slabs of k / group_size groups (by-scale, at most 128 a range: the
      // slab path keeps a wave's 128 group bases in two registers)
      // More than one record only while each range keeps >= min_lane elements a lane.
      const int64_t S = kAwqBlock / k_of_rec[r];
      // (flat: slabs of k elements, at most P a range)
      const bool flat = gps_of_rec[r] < 0;
      const int64_t gps = gps_of_rec[r];
      const int64_t units = flat || P > 0 ? rows : (rows + gps - 1) / gps;
      const int64_t min_units = P > 0 && !flat ? (min_lane + P - 1) / P : min_lane;
      const int64_t recs = std::min(std::max<int64_t>(1, (w.elems + target - 1) / target),
                                    std::max<int64_t>(1, units / (S * min_units)));
      int64_t ranges = std::min<int64_t>(units, S * recs);
      if (P == 0) ranges = std::max<int64_t>(ranges, (units + 127) / 128);
      if (flat) ranges = std::max<int64_t>(ranges, (units + P - 1) / P);
      const int32_t rr = (int32_t)((units + ranges - 1) / ranges);
      ranges = (units + rr - 1) / rr;
      jobs.push_back(AwqSplitJob{w.tensor, w.bucket, P, rows, c0_of_rec[r], rr, (int32_t)ranges, flat ? 2 : 1, ck_words});
      job_rec.push_back(r);
      ck_words += (ranges + 1) * k_of_rec[r];
      continue;
    }
    if (w.kind != 1 || rows < 2 || w.elems <= target) continue;
    const int64_t want = (w.elems + target - 1) / target;
    int32_t rr = (int32_t)((rows + want - 1) / want);
    rr = std::max<int32_t>(rr, (64 + P - 1) / P);
    const int32_t ranges = (rows + rr - 1) / rr;
    if (ranges < 2) continue;
    jobs.push_back(AwqSplitJob{w.tensor, w.bucket, P, rows, c0_of_rec[r], rr, ranges, 0, ck_words});
    job_rec.push_back(r);
    ck_words += (int64_t)(ranges - 1) * kAwqBlock;
  }
  auto make_records = [&](const std::vector<uint32_t> &failed) {
    std::vector<AwqWork> out;
    std::vector<int> split_of(base.size(), -1);
    for (size_t j = 0; j < jobs.size(); ++j)
      if (failed.empty() || failed[j] == 0u) split_of[job_rec[j]] = (int)j;
    for (size_t r = 0; r < base.size(); ++r) {
      if (split_of[r] < 0) {
        out.push_back(base[r]);
        continue;
      }
      const AwqSplitJob &J = jobs[(size_t)split_of[r]];
      if (J.full) {
        // 1024 / k ranges a record; the cost: one range's elements a work-item, x 1024
        const int32_t S = kAwqBlock / k_of_rec[r];
        const bool flat = J.full == 2;
        const int32_t gps = gps_of_rec[r];
        const int32_t units = flat || J.P > 0 ? J.rows : (J.rows + gps - 1) / gps;
        for (int32_t g = 0; g < J.ranges; g += S) {
          const int32_t n = std::min(J.range_rows, units - g * J.range_rows);
          out.push_back(AwqWork{J.tensor, J.bucket, 1, flat ? 4 : 3, g, J.range_rows, J.ranges, 0, J.out,
                                (int64_t)n * (flat ? 1 : std::max(J.P, 1)) * kAwqBlock});
        }
        continue;
      }
      for (int32_t g = 0; g < J.ranges; ++g) {
        const int32_t nrows = std::min(J.range_rows, J.rows - g * J.range_rows);
        out.push_back(AwqWork{J.tensor, J.bucket, 1, 2, g, J.range_rows, J.ranges, 0, J.out,
                              (int64_t)nrows * J.P * kAwqBlock});
      }
    }
    // largest first, so the launch's last workgroups are its smallest
    std::stable_sort(out.begin(), out.end(), [](const AwqWork &x, const AwqWork &y) { return x.elems > y.elems; });
    return out;
  };
  std::vector<AwqWork> items = make_records({});
  auto plan = new (std::nothrow) mps_awq_plan();
  if (!plan) return fail(MPS_ERR_NO_MEMORY, "out of memory");
  plan->device = dev;
  plan->count = count;
  plan->nwork = (int64_t)items.size();
  plan->first_out = count > 0 ? tensors[0].out : nullptr;
  // status word (zero) | work queues (zero) | descriptors | work records | split jobs | checkpoints | job failure flags
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t o_queues = 256;
  const size_t o_tensors = o_queues + up(kAwqQueueStride * kAwqPlanQueues);
  const size_t o_work = o_tensors + up(sizeof(mps_awq_tensor) * (size_t)count);
  const size_t o_jobs = o_work + up(sizeof(AwqWork) * items.size());
  const size_t o_ckpt = o_jobs + up(sizeof(AwqSplitJob) * jobs.size());
  const size_t o_failed = o_ckpt + up(sizeof(uint32_t) * (size_t)ck_words);
  std::vector<char> host(o_failed + up(sizeof(uint32_t) * jobs.size()), 0);
  if (count > 0) std::memcpy(host.data() + o_tensors, tensors, sizeof(mps_awq_tensor) * (size_t)count);
  if (!items.empty()) std::memcpy(host.data() + o_work, items.data(), sizeof(AwqWork) * items.size());
  if (!jobs.empty()) std::memcpy(host.data() + o_jobs, jobs.data(), sizeof(AwqSplitJob) * jobs.size());
  hipError_t e = hipMalloc(&plan->d_block, host.size());
  if (e == hipSuccess) {
    char *blk = static_cast<char *>(plan->d_block);
    plan->d_status = reinterpret_cast<uint32_t *>(blk);
    plan->d_queue = reinterpret_cast<uint32_t *>(blk + o_queues);
    plan->d_tensors = reinterpret_cast<mps_awq_tensor *>(blk + o_tensors);
    plan->d_work = reinterpret_cast<AwqWork *>(blk + o_work);
    plan->d_ckpt = reinterpret_cast<uint32_t *>(blk + o_ckpt);
    e = hipMemcpyAsync(blk, host.data(), host.size(), hipMemcpyHostToDevice, st);
    if (e == hipSuccess && !jobs.empty()) {
      hipLaunchKernelGGL(awq_checkpoints, dim3((unsigned)jobs.size()), dim3(kAwqBlock), 0, st, plan->d_tensors,
                         reinterpret_cast<const AwqSplitJob *>(blk + o_jobs), plan->d_ckpt,
                         reinterpret_cast<uint32_t *>(blk + o_failed));
      e = hipGetLastError();
      std::vector<uint32_t> failed(jobs.size(), 0u);
      if (e == hipSuccess)
        e = hipMemcpyAsync(failed.data(), blk + o_failed, sizeof(uint32_t) * jobs.size(), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e == hipSuccess && std::any_of(failed.begin(), failed.end(), [](uint32_t f) { return f != 0u; })) {
        // keep the buckets whose walk failed whole (fewer records than before)
        items = make_records(failed);
        plan->nwork = (int64_t)items.size();
        e = hipMemcpyAsync(blk + o_work, items.data(), sizeof(AwqWork) * items.size(), hipMemcpyHostToDevice, st);
      }
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
  }
  if (e != hipSuccess) {
    mps_awq_plan_destroy(plan);
    return hip_fail(e, "mps_awq_plan_create");
  }
  plan->splits = (int64_t)jobs.size();
  plan->ranges_mode = (std::any_of(items.begin(), items.end(), [](const AwqWork &w) { return w.tiny != 0; }) ? 4 : 0) |
                      (std::any_of(items.begin(), items.end(), [](const AwqWork &w) { return w.kind == 2; }) ? 1 : 0) |
                      (std::any_of(items.begin(), items.end(), [](const AwqWork &w) { return w.kind == 3; }) ? 2 : 0) |
                      (std::any_of(items.begin(), items.end(), [](const AwqWork &w) { return w.kind == 4; }) ? 8 : 0) |
                      (std::any_of(items.begin(), items.end(), [&](const AwqWork &w) {
                         return w.kind != 0 && tensors[w.tensor].group_col_start && tensors[w.tensor].group_size != 128;
                       })
                           ? 16
                           : 0);
  *plan_out = plan;
  return MPS_OK;
}

static int awq_plan_launch(mps_awq_plan *plan, int64_t out_delta, uint32_t *status, void *stream) {
  if (plan->nwork == 0) return MPS_OK;
  // The stream's work queue: the one it was given at its first launch, or the
  // next free one. A launch leaves its queue as it found it, so launches on
  // one stream share one; a graph captured on a stream replays with its queue.
  uint32_t *queue = nullptr;
  {
    std::lock_guard<std::mutex> lock(plan->mu);
    size_t i = 0;
    while (i < plan->streams.size() && plan->streams[i] != stream) ++i;
    if (i == plan->streams.size()) {
      if (i >= (size_t)kAwqPlanQueues)
        return fail(MPS_ERR_RUNTIME, "an AWQ decode plan serves at most %d streams", kAwqPlanQueues);
      plan->streams.push_back(stream);
    }
    queue = plan->d_queue + i * (kAwqQueueStride / sizeof(uint32_t));
  }
  int cus = 0;
  MPS_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, plan->device));
  const unsigned grid = (unsigned)std::min<int64_t>(plan->nwork, std::max(cus, 1));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kAwqBlock), 0, reinterpret_cast<hipStream_t>(stream), plan->d_tensors,
                       plan->d_work, plan->nwork, plan->d_ckpt, status, out_delta, queue);
  };
  if (plan->ranges_mode & (8 | 16)) {
    const AwqFlatLaunch a{plan->d_tensors, plan->d_work, plan->nwork, plan->d_ckpt, status, out_delta, queue, grid,
                          reinterpret_cast<hipStream_t>(stream)};
    const int mode = plan->ranges_mode;
    auto within = [&](int paths) { return (mode & ~paths) == 0; };
    if (within(13)) launch_awq_flat_13(a);
    else if (within(14)) launch_awq_flat_14(a);
    else if (within(11)) launch_awq_flat_11(a);
    else if (within(30)) launch_awq_flat_30(a);
    else launch_awq_flat_31(a);
  } else switch (plan->ranges_mode) {
    case 0: launch(awq_decode_plan<0>); break;
    case 1: launch(awq_decode_plan<1>); break;
    case 2: launch(awq_decode_plan<2>); break;
    case 3: launch(awq_decode_plan<3>); break;
    case 4: launch(awq_decode_plan<4>); break;
    case 5: launch(awq_decode_plan<5>); break;
    case 6: launch(awq_decode_plan<6>); break;
    default: launch(awq_decode_plan<7>); break;
  }
  MPS_HIP_CHECK(hipGetLastError());
  return MPS_OK;
}

int mps_awq_plan_decode(mps_awq_plan *plan, void *stream) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  return awq_plan_launch(plan, 0, plan->d_status, stream);
}

int mps_awq_plan_decode_into(mps_awq_plan *plan, uint16_t *out, void *stream) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (!out) return fail(MPS_ERR_INVALID_ARGUMENT, "out is NULL");
  if (plan->count == 0) return MPS_OK;
  uint32_t *status = nullptr;
  const int rc = status_word(plan->device, &status);
  if (rc != MPS_OK) return rc;
  const intptr_t delta = reinterpret_cast<intptr_t>(out) - reinterpret_cast<intptr_t>(plan->first_out);
  // the slab path stores 8 bytes a lane: the moved outputs keep its alignment
  if (delta % 8 != 0) return fail(MPS_ERR_INVALID_ARGUMENT, "out must be aligned like the plan's outputs (8 bytes)");
  return awq_plan_launch(plan, (int64_t)(delta / (intptr_t)sizeof(uint16_t)), status, stream);
}

int mps_awq_plan_info(const mps_awq_plan *plan, int64_t *work_items) {
  if (!plan || !work_items) return fail(MPS_ERR_INVALID_ARGUMENT, "NULL argument");
  *work_items = plan->nwork;
  return MPS_OK;
}

int mps_awq_plan_read_status(mps_awq_plan *plan, void *stream, uint32_t *status_out) {
  last_error().clear();
  if (!plan) return fail(MPS_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (!status_out) return fail(MPS_ERR_INVALID_ARGUMENT, "status_out is NULL");
  return read_and_clear(plan->device, plan->d_status, stream, "mps_awq_plan_read_status", status_out);
}

int mps_awq_plan_destroy(mps_awq_plan *plan) {
  if (!plan) return MPS_OK;
  if (plan->d_block) (void)hipFree(plan->d_block);
  delete plan;
  return MPS_OK;
}

}  // extern "C"
