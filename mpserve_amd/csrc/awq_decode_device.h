// AWQ int4 + Huffman-sidecar -> BF16 decode for MI355X (gfx950).
//
// Format (reference kernel/build_huffman.cu:1075-1580 and :1583-2126): bucket b
// owns a list of rows (row layout: row_indices[row_offsets[b] ..] x columns
// [col_start, col_start + col_len)) or of quantisation groups (by-scale
// layout: group g = row group_rows[g], columns [group_col_start[g],
// + group_size)). Its elements, flattened row (group) major, are dealt
// round-robin to k_eff = min(k, total) lanes; lane t codes e = t, t+k_eff, ...
// as one MSB-first substream from bit bucket_bit_base[b] + startbit[b][t].
// A code is looked up with the next 11 bits in the table of
// (bucket scale, int4 value); a length nibble of 15 marks ESC: the code is
// 11 bits and 16 raw BF16 bits follow (decode_huffman.cu:454-460). A table id
// of -1 decodes as ESC too, as the reference kernel does.
//
// Mapping to CDNA4: one workgroup of 1024 work-items per bucket, one lane per
// work-item. The bucket's 16 tables are expanded once into LDS as 32-bit
// entries {sym:16 | nibble:4} indexed (qv << 11) | peek (128 KiB), and the
// bucket's row (group) start offsets are staged next to them (32 KiB), so an
// element costs one ds_read_b32 for its code and one for its row offset. The
// table fill issues all of a work-item's global loads before its first LDS
// store (one memory round trip per bucket). The bit supply is a 64-bit
// MSB-aligned buffer topped up to >= 32 bits after every element from a
// register queue of 8 32-bit chunks; an aligned quad of 4 chunks (more than a
// block of kDepth = 8 codes can take without ESC) and the block's int4 bytes
// are loaded one block ahead, one 16-byte request per quad. ESC payloads can drain the queue, which then reads a
// chunk straight from memory. A tensor with fewer buckets than CUs runs two
// 512-work-item workgroups per bucket, each with its own copy of the tables.
//
// Included by awq_decode.hip (the host side and the kernels without flat ranges)
// and awq_decode_flat_*.hip (the plan kernels with them, awq_decode_flat.h).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mps_common.h"

namespace mps {
namespace {

constexpr int kAwqL = 11;
constexpr int kAwqTable = 1 << kAwqL;     // 2048 entries per code table
constexpr int kAwqPacked = kAwqTable / 2; // 1024 bytes of packed 4-bit lengths
constexpr int kAwqBlock = 1024;           // work-items per bucket workgroup (>= k)
constexpr int kLutEntries = 16 * kAwqTable;
constexpr int kRowSlots = 8192;           // row (group) start offsets staged in LDS
constexpr uint32_t kBadBase = 0xFFFFFFFFu;
// Elements per block, and the chunk queue: a block of kDepth codes without
// ESC takes at most 3 32-bit chunks from the queue; a quad of kStage chunks is
// staged (loaded) one block ahead, and the queue holds kQueue.
#ifndef MPS_AWQ_DEPTH
#define MPS_AWQ_DEPTH 8
#endif
constexpr int kDepth = MPS_AWQ_DEPTH;
constexpr int kStage = 4;   // chunks staged a block: one 16-byte aligned quad
constexpr int kQueue = 8;
static_assert((kDepth * kAwqL + 31) / 32 <= kQueue - kStage, "a block's codes must fit the queue after an append");

// A global-address-space atomic, not a generic one: an outstanding generic
// (flat) access makes the compiler turn every later memory wait into a full one.
__device__ __forceinline__ void flag(uint32_t *status, unsigned int f) {
  __hip_atomic_fetch_or((__attribute__((address_space(1))) uint32_t *)(status), f, __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_AGENT);
}
// A load through a global pointer, for the same reason.
template <typename V>
__device__ __forceinline__ V gload(const V *p) {
  return *(const __attribute__((address_space(1))) V *)(p);
}

// Stream chunk c (32 bits, stream order) of u64 words stored little-endian:
// word w's first 32 stream bits are u32 2w+1. Past the end the last chunk is
// re-read: a well-formed lane never consumes those bits, and an 11-bit peek
// that runs past its last code selects an entry whose low bits do not matter.
__device__ __forceinline__ uint32_t chunk_at(const uint32_t *__restrict__ bs32, uint64_t nchunks, uint64_t c) {
  const uint64_t cc = c < nchunks ? c : nchunks - 1;
  return bs32[cc ^ 1u];
}

__device__ uint32_t g_awq_zero_chunks[2];

// Element offset (row * m + column start) of row (group) rr of the bucket;
// kStaged: every row of the bucket is staged in LDS.
template <bool kStaged>
__device__ __forceinline__ uint32_t row_base(const mps_awq_tensor &T, const uint32_t *__restrict__ s_base,
                                             int32_t ra, int32_t rr, int32_t c0, int32_t cl) {
  if (kStaged || rr < kRowSlots) return s_base[rr];
  const int64_t row = T.row_indices[ra + rr];
  const int64_t col = T.group_col_start ? (int64_t)T.group_col_start[ra + rr] : (int64_t)c0;
  if (row < 0 || row >= T.n || col < 0 || col + cl > T.m) return kBadBase;
  return (uint32_t)(row * T.m + col);
}

// One lane's substream (the element walk, the bit supply and the stores).
template <bool kStaged>
__device__ __forceinline__ void awq_lane(const mps_awq_tensor &T, const uint32_t *__restrict__ lut,
                                         const uint32_t *__restrict__ s_base, int64_t b, int32_t ra, int32_t c0,
                                         int32_t cl, int64_t total, int32_t k, int32_t k_eff, int lane,
                                         uint32_t *status) {
  const uint32_t *__restrict__ sb = T.bucket_thread_startbit + b * ((int64_t)k + 1);
  const uint64_t pos0 = (uint64_t)T.bucket_bit_base[b] + sb[lane];
  const uint64_t pos_end = (uint64_t)T.bucket_bit_base[b] + sb[lane + 1];
  const bool empty = T.bitstream_words <= 0;
  const uint32_t *__restrict__ bs32 = empty ? g_awq_zero_chunks : reinterpret_cast<const uint32_t *>(T.bitstream);
  const uint64_t nchunks = empty ? 2u : (uint64_t)T.bitstream_words * 2u;

  // Initial fill: buffer from chunks cb, cb+1; queue = the next kQueue chunks.
  const uint64_t cb = pos0 >> 5;
  const int skip = (int)(pos0 & 31u);
  uint64_t buf = (((uint64_t)chunk_at(bs32, nchunks, cb) << 32) | chunk_at(bs32, nchunks, cb + 1)) << skip;
  int cnt = 64 - skip;
  // The queue starts with the chunks up to the next multiple of 4, so that
  // every later stage is one aligned quad.
  uint32_t qq[kQueue];
#pragma unroll
  for (int j = 0; j < kQueue; ++j) qq[j] = j < 3 ? chunk_at(bs32, nchunks, cb + 2 + j) : 0u;
  int qn = (int)((4u - ((cb + 2) & 3u)) & 3u);
  uint64_t tail = cb + 2 + qn;  // index of the first chunk not yet in buf/queue

  // Element walk e = tid + i*k_eff -> (rr, cc) = (e / cl, e % cl), incrementally.
  int32_t rr = lane / cl;
  int32_t cc = lane - rr * cl;
  const int32_t dr = k_eff / cl, dc = k_eff - dr * cl;
  const int32_t count = (int32_t)((total - lane + k_eff - 1) / k_eff);
  const uint8_t *__restrict__ qv = T.int4;
  char *__restrict__ outb = reinterpret_cast<char *>(T.out);
  const uint32_t first = row_base<kStaged>(T, s_base, ra, rr, c0, cl);
  const uint32_t safe = first == kBadBase ? 0u : first + (uint32_t)cc;  // an address every lane may read
  int32_t walked = 0;
  auto next_block = [&](uint32_t (&idx)[kDepth]) {
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      uint32_t v = kBadBase;
      if (walked + j < count) {
        const uint32_t base = row_base<kStaged>(T, s_base, ra, rr, c0, cl);
        if (base != kBadBase) v = base + (uint32_t)cc;
      }
      idx[j] = v;
      cc += dc;
      rr += dr;
      if (cc >= cl) {
        cc -= cl;
        rr += 1;
      }
    }
    walked += kDepth;
  };
  uint32_t ia[kDepth], ib[kDepth], qa[kDepth], qb[kDepth];
  next_block(ia);
#pragma unroll
  for (int j = 0; j < kDepth; ++j) qa[j] = qv[ia[j] == kBadBase ? safe : ia[j]];
  // Chunks tail .. tail+3: one 16-byte load when the quad is aligned and whole
  // (u32 words 4j .. 4j+3 hold chunks 4j+1, 4j, 4j+3, 4j+2), else four loads.
  const bool aligned16 = (reinterpret_cast<uintptr_t>(bs32) & 15u) == 0;
  auto stage = [&](uint32_t (&st)[kStage]) {
    if (aligned16 && (tail & 3u) == 0 && tail + 4 <= nchunks) {
      const uint4 v = *reinterpret_cast<const uint4 *>(bs32 + tail);
      st[0] = v.y;
      st[1] = v.x;
      st[2] = v.w;
      st[3] = v.z;
    } else {
#pragma unroll
      for (int j = 0; j < kStage; ++j) st[j] = chunk_at(bs32, nchunks, tail + j);
    }
  };
  uint32_t st[kStage];
  stage(st);
  bool stale = false;

  auto refill = [&]() {
    if (cnt < 32) {
      if (qn > 0) {
        buf |= (uint64_t)qq[0] << (32 - cnt);
#pragma unroll
        for (int j = 0; j + 1 < kQueue; ++j) qq[j] = qq[j + 1];
        --qn;
      } else {
        // Queue drained by ESC payloads: read the chunk straight from memory.
        const uint32_t ch = chunk_at(bs32, nchunks, tail);
        buf |= (uint64_t)ch << (32 - cnt);
        ++tail;
        stale = true;
      }
      cnt += 32;
    }
  };
  auto decode_one = [&](uint32_t q, uint32_t idx) {
    const uint32_t peek = (uint32_t)(buf >> (64 - kAwqL));
    const uint32_t ent = lut[((q & 15u) << kAwqL) | peek];
    const uint32_t nib = ent & 15u;
    uint32_t sym = ent >> 16;
    if (nib == 15u) {
      // ESC: the code is L bits, then 16 raw bits (decode_huffman.cu:454-460)
      buf <<= kAwqL;
      sym = (uint32_t)(buf >> 48);
      buf <<= 16;
      cnt -= kAwqL + 16;
    } else {
      buf <<= nib;
      cnt -= (int)nib;
    }
    // saddr store: the byte offset fits 32 bits (n*m < 2^31)
    if (idx != kBadBase) *reinterpret_cast<uint16_t *>(outb + (idx << 1)) = (uint16_t)sym;
    refill();
  };
  auto block = [&](int32_t i0, uint32_t (&qc)[kDepth], uint32_t (&ic)[kDepth], uint32_t (&qnx)[kDepth],
                   uint32_t (&inx)[kDepth]) {
    // Append the chunks staged one block ago if they are current and fit.
    if (!stale && qn <= kQueue - kStage) {
#pragma unroll
      for (int j = 0; j < kQueue; ++j)
#pragma unroll
        for (int t = 0; t < kStage; ++t)
          if (j == qn + t) qq[j] = st[t];
      qn += kStage;
      tail += kStage;
    }
    stale = false;
    next_block(inx);
#pragma unroll
    for (int j = 0; j < kDepth; ++j) qnx[j] = qv[inx[j] == kBadBase ? safe : inx[j]];
    stage(st);
    if (i0 + kDepth <= count) {
#pragma unroll
      for (int j = 0; j < kDepth; ++j) decode_one(qc[j], ic[j]);
    } else {
#pragma unroll
      for (int j = 0; j < kDepth; ++j)
        if (i0 + j < count) decode_one(qc[j], ic[j]);
    }
  };
  for (int32_t i0 = 0; i0 < count; i0 += 2 * kDepth) {
    block(i0, qa, ia, qb, ib);
    if (i0 + kDepth >= count) break;
    block(i0 + kDepth, qb, ib, qa, ia);
  }
  // The next unread bit must be where the next lane's substream begins.
  if (tail * 32u - (uint64_t)(cnt + 32 * qn) != pos_end) flag(status, MPS_STATUS_DESYNC);
}

// kSplit workgroups of kAwqBlock / kSplit work-items share a bucket: each
// stages the bucket's tables and decodes its slice of the lanes (launches with
// fewer buckets than CUs use several CUs per bucket).
template <int kSplit>
__device__ __forceinline__ void awq_bucket(const mps_awq_tensor &T, int64_t b, int part, uint32_t *__restrict__ lut,
                                           uint32_t *__restrict__ s_base, uint32_t *status) {
  constexpr int kThreads = kAwqBlock / kSplit;
  const int tid = threadIdx.x;
  const int lane = part * kThreads + tid;
  // Bucket geometry (decode_huffman.cu:417-444, :528-545).
  const int32_t ra = T.bucket_row_offsets[b], rb = T.bucket_row_offsets[b + 1];
  const int32_t rows = rb - ra;
  if (rows <= 0) return;
  const bool by_scale = T.group_col_start != nullptr;
  const int32_t c0 = by_scale ? 0 : T.bucket_col_start[b];
  const int32_t cl = by_scale ? (int32_t)T.group_size : T.bucket_col_len[b];
  if (cl <= 0 || ra < 0 || (int64_t)rb > T.num_row_indices ||
      (!by_scale && (c0 < 0 || (int64_t)c0 + cl > T.m))) {
    if (tid == 0) flag(status, MPS_STATUS_BAD_BUCKET);
    return;
  }
  const int64_t total = (int64_t)rows * cl;
  const int32_t k = (int32_t)T.k;
  const int32_t k_eff = total < k ? (int32_t)total : k;

  // Tables: entry (q << 11) | p = sym << 16 | nibble; a missing table (id -1)
  // is all ESC entries, as the reference decodes it. The 16 table ids are
  // bucket-uniform (scalar loads); every work-item then fills 32 entries, two
  // per table, with all 64 global loads issued before the first LDS store
  // (addresses of missing tables are clamped to table 0 and the entry selected
  // afterwards), so the fill costs one memory round trip, not 32.
  int32_t gid[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) gid[q] = T.bucket_table[b * 16 + q];
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 16; ++q)
      if (gid[q] < -1 || gid[q] >= T.num_tables) flag(status, MPS_STATUS_BAD_TABLE);
  }
  const int64_t G = T.num_tables;
  if (G <= 0) {
    for (int i = tid; i < kLutEntries; i += kThreads) lut[i] = 15u;
  } else for (int part = 0; part < kSplit; ++part) {  // kSplit rounds of 32 entries a work-item
    uint32_t sy[32], ln[32];
#pragma unroll
    for (int it = 0; it < 32; ++it) {
      const int i = (part * 32 + it) * kThreads + tid;
      const int q = i >> kAwqL, p = i & (kAwqTable - 1);
      const uint32_t g = (gid[q] >= 0 && gid[q] < G) ? (uint32_t)gid[q] : 0u;  // table 0 exists: G > 0
      sy[it] = T.decode_syms[(size_t)g * kAwqTable + p];
      ln[it] = T.decode_lens[(size_t)g * kAwqPacked + (p >> 1)];
    }
#pragma unroll
    for (int it = 0; it < 32; ++it) {
      const int i = (part * 32 + it) * kThreads + tid;
      const int q = i >> kAwqL, p = i & (kAwqTable - 1);
      const bool ok = gid[q] >= 0 && gid[q] < G;
      lut[i] = ok ? (sy[it] << 16) | ((p & 1) ? (ln[it] >> 4) : (ln[it] & 15u)) : 15u;
    }
  }
  const int32_t staged = rows < kRowSlots ? rows : kRowSlots;
  for (int r = tid; r < staged; r += kThreads) {
    const int64_t row = T.row_indices[ra + r];
    const int64_t col = by_scale ? (int64_t)T.group_col_start[ra + r] : (int64_t)c0;
    uint32_t base = kBadBase;
    if (row >= 0 && row < T.n && col >= 0 && col + cl <= T.m) base = (uint32_t)(row * T.m + col);
    else flag(status, MPS_STATUS_BAD_ROW);
    s_base[r] = base;
  }
  __syncthreads();
  if (lane >= k_eff) return;

  if (rows <= kRowSlots) awq_lane<true>(T, lut, s_base, b, ra, c0, cl, total, k, k_eff, lane, status);
  else awq_lane<false>(T, lut, s_base, b, ra, c0, cl, total, k, k_eff, lane, status);
}

// ---------------------------------------------------------------------------
// Slab path, told here for k = 1024 substreams and groups of 128 columns (other
// sizes, slab_group, and k 256 and 512 likewise): by-scale buckets with groups of 128
// columns (8 to 1024 groups). Element e of such a bucket is column e % 128 of
// its group e / 128, and substream t codes e = t, t + 1024, ...: the i-th
// element of every substream lies in *slab* i, the bucket's groups 8i .. 8i+7.
// Lane l = 16R + v of wave w decodes substream t = 64w + 4v + R, four elements
// (slabs 4g .. 4g+3) per step, in the register layout of the FP8 slab decode:
//  - lane (R, v) loads one dword of int4 bytes, columns 64(w & 1) + 4v .. +3 of
//    slab 4g+R's group 8(4g+R) + w/2, so each 16-lane row reads 64 contiguous
//    bytes; a 4x4 byte transpose across lanes (0,v) .. (3,v) gives every lane
//    its own four bytes;
//  - the inverse transpose of the BF16 symbols gives lane (R, v) those columns'
//    values for one 8-byte store (a 128-byte segment per 16-lane row);
//  - the wave's group bases (row * m + column start + 64(w & 1)) for slabs
//    l and l + 64 sit in lane l of two VGPRs and are fetched with ds_bpermute;
//  - the bit supply is the FP8 slab path's: an 8-chunk LDS queue per lane fed
//    from a register reserve that requests aligned 64-byte blocks.
// Codes are up to 11 bits, so a step cuts two 32-bit windows, two codes each.
// An ESC entry's low bits are 27 (its 11-bit code and the 16 raw bits), so bit
// 4 flags it and the running shift steps over the raw bits; a step holding an
// ESC code is decoded again code by code, reading the raw symbol.
// ---------------------------------------------------------------------------
// A plan's work record (a workgroup decodes one at a time, taking them from
// the plan's queue: awq_decode_plan).
//  kind 0: buckets bucket .. bucket + nsub - 1 on the per-lane path (one scale, shared tables;
//          with `tiny`, buckets of one code a lane that look their codes up in the global tables);
//  kind 1: slab-path buckets bucket .. bucket + nsub - 1 with identical table ids (a by-scale run);
//  kind 2: rows [range * range_rows, +range_rows) of a slab-path row bucket split into
//          `ranges` ranges, starting from the lane checkpoints at ckpt + (range - 1) * 1024
//          and ending at ckpt + range * 1024 (the bucket's own start and end bits at its ends);
//  kind 4: ranges range .. range + 1024 / k - 1 of a flat bucket (k 256, 512 or 1024, rows
//          of any width), side by side as kind 3's; a range is range_rows slabs of k elements;
//  kind 3: ranges range .. range + 1024 / k - 1 of a row bucket with k 256 or 512 split into
//          `ranges` ranges, side by side on the slab path: range r starts at checkpoint row
//          r and ends at row r + 1 of ckpt ([ranges + 1][k]).
struct AwqWork {
  int32_t tensor, bucket, nsub, kind;
  int32_t range, range_rows, ranges;
  int32_t tiny;  // kind 0: 1 when every bucket codes at most one element a lane (awq_tiny_lane)
  int64_t ckpt;
  int64_t elems;  // (the plan's ordering key)
};
static_assert(sizeof(AwqWork) == 48, "work record layout");

constexpr uint32_t kAwqEscBit = 1u << 4;
constexpr uint32_t kAwqEscLow = 27u;          // 11 + 16: an ESC entry's low bits
constexpr int kSlabQSlots = 8;                // LDS queue chunks per lane
constexpr uint32_t kSlabBsPast = 0x80000000u; // bitstream offset beyond every bucket's range
constexpr uint32_t kSlabOutPast = 0xFFFFFFF0u;  // BF16 byte offset beyond every output (2*n*m < 2^32)
constexpr uint32_t kSlabInPast = 0x80000000u;   // int4 byte offset beyond every input (n*m < 2^31)
constexpr int kSlabCacheNT = 2;               // buffer cache-policy bits: non-temporal
constexpr int kSlabMaxSlabs = 128;              // a wave's slab bases: two registers of 64
constexpr int kFlatMaxRows = 128;               // a flat range's row bases, likewise
constexpr int64_t kFlatMaxCols = 1 << 24;
// By-scale groups the slab path takes: a power of two of 64 columns or more
// (a wave's 64 columns lie in one group), and whole groups a slab of k.
__host__ __device__ inline bool slab_group(int64_t group_size, int64_t k) {
  return group_size >= 64 && group_size <= k && (group_size & (group_size - 1)) == 0;
}
constexpr uint32_t kRunTables = 1u << 8;        // run_flags: a run's tables are in the LDS
static_assert(kSlabQSlots * kAwqBlock <= kRowSlots, "the slab queue lives in the row-offset region");

// Buffer resource over [base, base + bytes): raw buffer loads past the end
// return 0 and stores past the end are dropped (gfx9 V# with stride 0).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t awq_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint32_t awq_uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// Slab layouts: by-scale groups, or row buckets whose column range is P blocks
// of 1024 (P >= 4) with P % 4 == 0 (a step's four slabs in one row) or not (a
// step can straddle two rows; each lane picks its row's offset).
// Flat layouts: slab i is the k elements from i * k on in the range's row-major
// order, whatever its rows' width (the FP8 slab decode's kWrap 3 and 4): `count`
// is then the range's elements, `P` the width, `fcol` the first element's column;
// kLayFlat for widths that are multiples of 4, kLayFlatSplit for the others,
// where a lane's four elements may continue in the next row. Measured, as plans,
// against the per-lane path: row buckets of 3001 x 5000, k = 1024: 243 -> 34 us;
// 3001 x 5001, k = 256: 662 -> 40 us.
enum : int { kLayGroups = 0, kLayRows = 1, kLayRowsWrap = 2, kLayFlat = 3, kLayFlatSplit = 4 };

// base_lo / base_hi: lane l holds slab l's and l + 64's base (groups), or row
// l's and l + 64's offset (rows, column start included); rows and P describe a
// row bucket (rows x P elements per lane).
// kShift: log2 of the substream count k (the row layouts' block stride), 10,
// or 0 for the run-time `kshift` (kLayRows with k 256 or 512, several row
// ranges side by side: `lane` is the work-item's substream within its range's
// group of k, `qlane` the work-item, whose LDS queue column it owns).
template <bool kEsc, int kLay, int kShift = 10>
__device__ __forceinline__ void awq_slab_decode(const mps_awq_tensor &T, const uint32_t *__restrict__ lut,
                                                uint32_t *__restrict__ queue, uint32_t qlane, uint32_t lane,
                                                uint32_t kshift, uint32_t count,
                                                uint32_t base_lo, uint32_t base_hi, uint32_t rows, uint32_t P,
                                                uint64_t bucket_bit, const uint2 (&first)[4], uint32_t pos,
                                                uint32_t pos_end, uint32_t *status, uint32_t fcol = 0) {
#ifndef MPS_AWQ_SLAB_PREFETCH
#define MPS_AWQ_SLAB_PREFETCH 8
#endif
#ifndef MPS_AWQ_FEED_EVERY
#define MPS_AWQ_FEED_EVERY 2
#endif
  constexpr bool kFlat = kLay >= kLayFlat;
  constexpr int DF = kLay == kLayFlatSplit ? 4 : MPS_AWQ_SLAB_PREFETCH;  // int4 prefetch distance (steps)
  constexpr int FE = MPS_AWQ_FEED_EVERY;     // steps per bitstream feed (16 bytes: 2 x 44 bits fit)
  static_assert(DF % FE == 0 && (FE == 1 || FE == 2), "a feed every one or two steps");
#ifndef MPS_AWQ_RB
#define MPS_AWQ_RB 4
#endif
  constexpr int RB = MPS_AWQ_RB;  // 16-byte blocks per bitstream request
  static_assert(kShift == 10 || (kShift == 0 && kLay != kLayRowsWrap), "k < 1024: no aligned steps across rows");
  count = awq_uni(count);
  kshift = kShift ? (uint32_t)kShift : awq_uni(kshift);
  bucket_bit = ((uint64_t)awq_uni((uint32_t)(bucket_bit >> 32)) << 32) | awq_uni((uint32_t)bucket_bit);
  const uint32_t nfull = kFlat ? count >> (kshift + 2u) : count >> 2;
  uint32_t tail = count & 3u;  // elements of the last, partial step (flat: by lane)
  uint32_t gall = nfull + (tail ? 1u : 0u);
  if constexpr (kFlat) {
    const uint32_t rest = count - (nfull << (kshift + 2u));
    const uint32_t t = (lane & ~63u) | ((lane & 15u) << 2) | ((lane >> 4) & 3u);  // the lane's substream
    tail = rest > t ? (rest - t + (1u << kshift) - 1u) >> kshift : 0u;
    gall = nfull + (rest ? 1u : 0u);
  }
  const uint32_t nm = (uint32_t)(T.n * T.m);
  const __amdgpu_buffer_rsrc_t r_q = awq_rsrc(T.int4, nm);
  const __amdgpu_buffer_rsrc_t r_out = awq_rsrc(T.out, 2u * nm);
  const uint64_t bs_bytes = T.bitstream_words > 0 ? (uint64_t)T.bitstream_words * 8u : 0u;
  const uint64_t base_byte = bucket_bit >> 3;
  const uint32_t win_bytes = base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
  const __amdgpu_buffer_rsrc_t r_bs =
      awq_rsrc(reinterpret_cast<const uint8_t *>(T.bitstream) + (base_byte < bs_bytes ? base_byte : 0), win_bytes);

  const uint32_t lane4 = qlane << 2;
  const uint32_t R = (lane >> 4) & 3u;
  const uint32_t R4 = R << 2;
  const uint32_t v4 = (lane & 15u) << 2;
  const char *qbytes = reinterpret_cast<const char *>(queue);
  const char *lbytes = reinterpret_cast<const char *>(lut);
  // byte selectors of the int4-byte transpose (v_perm: 0-3 pick the second operand's bytes, 4-7 the first's)
  const uint32_t selA = (R & 2u) ? 0x07060302u : 0x05040100u;
  const uint32_t selB = (R & 1u) ? 0x07030501u : 0x06020400u;

  // --- bitstream queue: chunk h (32 stream bits) of this lane in slot (~h) & 7 ---
  auto chunk_mem = [&](uint32_t h) -> uint32_t {  // biased chunk h from memory (h < 2: zeros)
    return __builtin_amdgcn_raw_buffer_load_b32(r_bs, ((h - 2u) ^ 1u) << 2, 0, 0);
  };
  auto put_pair = [&](uint32_t h, uint32_t hi, uint32_t lo) {  // chunks h (even) and h + 1
    uint32_t *slot = queue + (((~h << 10) & 0x1800u) | qlane);
    slot[0] = lo;
    slot[1024] = hi;
  };
  const uint32_t phase =
      ((uint32_t)reinterpret_cast<uintptr_t>(T.bitstream) + (uint32_t)(bucket_bit >> 3)) & (16u * RB - 1u);
  const uint32_t rq0 = ((pos >> 5) & ~1u) + 2u;
  const uint32_t nfirst = ((phase + 4u * (rq0 - 2u)) & 15u) ? 6u : 8u;
#pragma unroll
  for (int i = 0; i < 3; ++i) put_pair(rq0 + 2 * i, first[i].y, first[i].x);
  if (nfirst == 8u) put_pair(rq0 + 6u, first[3].y, first[3].x);
  uint32_t wqb = (rq0 + nfirst) << 5;  // 32 x (first chunk not yet written)
  uint32_t rqb = wqb;                  // 32 x (first chunk not yet requested)
  uint32_t np = 0u - (pos + 64u);      // negated biased position

  auto window = [&](uint32_t npv) -> uint32_t {  // 32 stream bits at -npv
    const uint32_t t7 = npv << 7;
    const uint32_t c0 = *reinterpret_cast<const uint32_t *>(qbytes + ((t7 & 0x7000u) | lane4));
    const uint32_t c1 = *reinterpret_cast<const uint32_t *>(qbytes + (((t7 - 4096u) & 0x7000u) | lane4));
    uint32_t w = __builtin_amdgcn_alignbit(c0, c1, npv);
    const bool dry = (int32_t)(wqb + npv) <= 31;
    if (__builtin_amdgcn_ballot_w64(dry)) {
      if (dry) {
        const uint32_t h = (~npv) >> 5;
        w = __builtin_amdgcn_alignbit(chunk_mem(h), chunk_mem(h + 1u), npv);
        __asm__ volatile("" ::"v"(w));  // wait for the loads here, not at a later join
      }
    }
    return w;
  };
  // 64 stream bits at -npv as {hi, lo}: three queue chunks, or memory for
  // lanes whose queue lacks the third.
  auto window64 = [&](uint32_t npv, uint32_t &hi, uint32_t &lo) {
    const uint32_t t7 = npv << 7;
    uint32_t c0 = *reinterpret_cast<const uint32_t *>(qbytes + ((t7 & 0x7000u) | lane4));
    uint32_t c1 = *reinterpret_cast<const uint32_t *>(qbytes + (((t7 - 4096u) & 0x7000u) | lane4));
    uint32_t c2 = *reinterpret_cast<const uint32_t *>(qbytes + (((t7 - 8192u) & 0x7000u) | lane4));
    const bool dry = (int32_t)(wqb + npv) <= 63;
    if (__builtin_amdgcn_ballot_w64(dry)) {
      if (dry) {
        const uint32_t h = (~npv) >> 5;
        c0 = chunk_mem(h);
        c1 = chunk_mem(h + 1u);
        c2 = chunk_mem(h + 2u);
        __asm__ volatile("" ::"v"(c0), "v"(c1), "v"(c2));  // wait for the loads here, not at a later join
      }
    }
    hi = __builtin_amdgcn_alignbit(c0, c1, npv);
    lo = __builtin_amdgcn_alignbit(c1, c2, npv);
  };
  // Register reserve of up to RB 16-byte blocks after the queue's last chunk,
  // refilled by aligned 64-byte requests that land in inb.
  uint4 rv[RB], inb[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) rv[i] = inb[i] = make_uint4(0u, 0u, 0u, 0u);
  uint32_t rcnt = 0, ninb = 0;
  bool ifl = false;
  // A feed writes chunks h .. h + 3 (h = wqb / 32, even) as two slot pairs,
  // ((~h) >> 1) & 3 and the one below; the next feed's h is 4 more, so both
  // pair indices flip bit 1: their byte addresses are kept and XORed with 0x4000.
  char *const qw = reinterpret_cast<char *>(queue);
  uint32_t fa = ((((~(wqb >> 5)) << 10) & 0x1800u) | qlane) << 2;
  uint32_t fb = ((((~((wqb >> 5) + 2u)) << 10) & 0x1800u) | qlane) << 2;
  auto feed = [&]() {
    const bool f = rcnt != 0u && (int32_t)(wqb + np) < 128;
    if (f) {
      *reinterpret_cast<uint32_t *>(qw + fa) = rv[0].x;          // chunk h + 1
      *reinterpret_cast<uint32_t *>(qw + fa + 4096u) = rv[0].y;  // chunk h
      *reinterpret_cast<uint32_t *>(qw + fb) = rv[0].z;          // chunk h + 3
      *reinterpret_cast<uint32_t *>(qw + fb + 4096u) = rv[0].w;  // chunk h + 2
#pragma unroll
      for (int i = 0; i + 1 < RB; ++i) rv[i] = rv[i + 1];
    }
    const uint32_t flip = f ? 0x4000u : 0u;
    fa ^= flip;
    fb ^= flip;
    wqb += f ? 128u : 0u;
    rcnt -= f ? 1u : 0u;
  };
  // The first request (is_first) runs up to the next 16 RB-byte boundary of the
  // bitstream; every later one is RB whole blocks from that boundary on.
  auto land = [&]() {
    const bool l = ifl && rcnt == 0u;
    if (l) {
#pragma unroll
      for (int i = 0; i < RB; ++i) rv[i] = inb[i];
    }
    rcnt = l ? ninb : rcnt;
    ifl = ifl && !l;
  };
  auto reserve = [&](auto is_first) {
    constexpr bool kFirst = decltype(is_first)::value;
    const bool req = !ifl && rcnt <= 1u && (int32_t)(rqb - (pos_end + 192u)) < 0;
    const uint32_t off = (rqb >> 3) - 8u;
    const uint32_t nreq = kFirst ? (16u * RB - ((phase + off) & (16u * RB - 1u))) >> 4 : (uint32_t)RB;
    if (req) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(
            r_bs, (!kFirst || (uint32_t)i < nreq) ? off + 16u * (uint32_t)i : kSlabBsPast, 0, 0);
        inb[i] = make_uint4(v[0], v[1], v[2], v[3]);
      }
      ninb = nreq;
    }
    ifl = ifl || req;
    rqb += req ? nreq << 7 : 0u;
  };
  // after every second step: a 16-byte feed covers the 2 x 44 bits two steps can take.
  // Requests are considered at every MPS_AWQ_REQ_EVERY-th of these: lanes reach
  // the request point on different steps, so a request's loads carry few
  // active lanes, and asking less often gathers more of them into each load.
#ifndef MPS_AWQ_REQ_EVERY
#define MPS_AWQ_REQ_EVERY 2
#endif
  static_assert(MPS_AWQ_REQ_EVERY >= 1 && (MPS_AWQ_REQ_EVERY & (MPS_AWQ_REQ_EVERY - 1)) == 0, "a power of two");
  uint32_t bstep = 0;  // bitstream steps taken (uniform)
  auto bitstream_step = [&]() {
    land();
    if ((bstep & (MPS_AWQ_REQ_EVERY - 1)) == 0u) reserve(std::false_type{});
    bstep = awq_uni(bstep + 1u);
    feed();
  };

  // --- walker: the int4 load of step g; returns its BF16 store byte offset
  // (kLayRows: the step's uniform element offset; the lane adds its own) ---
  rows = awq_uni(rows);
  P = awq_uni(P);
  uint32_t w_g = 0, w_row = 0, w_blk = 0;
  auto row_offset = [&](uint32_t r) -> uint32_t {
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)base_lo, (int)(r & 63u));
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)base_hi, (int)(r & 63u));
    return r < 64u ? a : b;
  };
  uint32_t w_off = 0, w_next = 0;
  if constexpr (kLay == kLayRows || kLay == kLayRowsWrap) {
    w_off = row_offset(0);
    w_next = row_offset(rows > 1u ? 1u : 0u);  // offset of row w_row + 1 (kLayRowsWrap)
  }
  const uint32_t colw = (lane & ~63u) | v4;    // 64w + 4v: the lane's columns within a k-block
  const uint32_t vf_al = (R << kshift) + colw;  // ... and its block within an aligned step
  auto load_step = [&](uint32_t &F) -> uint32_t {
    uint32_t ret;
    if constexpr (kLay == kLayGroups) {
      // this lane's slab is 4 w_g + R: its base sits in lane (4 w_g + R) & 63 of
      // base_lo (slabs below 64) or base_hi (the four slabs are all below or all above)
      const bool hi = w_g >= 16u;
      const uint32_t src = hi ? base_hi : base_lo;
      const uint32_t base = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(((w_g << 4) + R4) & 0xFCu), (int)src);
      const bool ok = (int32_t)R < (int32_t)awq_uni(count - 4u * w_g);
      const uint32_t off = base + v4;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_q, ok ? off : kSlabInPast, 0, 0);
      ret = ok ? off << 1 : kSlabOutPast;
    } else if constexpr (kLay == kLayRows) {
      const uint32_t so = awq_uni(w_off + (w_blk << kshift));
      F = __builtin_amdgcn_raw_buffer_load_b32(r_q, vf_al, so, 0);
      ret = so;
    } else {
      const uint32_t b = w_blk + R;
      const bool wrap = b >= P;
      const bool ok = !wrap || w_row + 1u < rows;
      const uint32_t off = (wrap ? w_next : w_off) + ((wrap ? b - P : b) << kshift) + colw;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_q, ok ? off : kSlabInPast, 0, 0);
      ret = ok ? off << 1 : kSlabOutPast;
    }
    const bool more = w_g + 1u < gall;
    if constexpr (kLay != kLayGroups) {
      // advance the row walk (past the last step it stays there)
      const uint32_t nb = w_blk + 4u;
      const bool wr = nb >= P;
      const uint32_t nrow = w_row + ((more && wr) ? 1u : 0u);
      const uint32_t noff = row_offset(nrow);
      const uint32_t nnext = row_offset(nrow + 1u < rows ? nrow + 1u : nrow);
      w_blk = awq_uni(more ? (wr ? nb - P : nb) : w_blk);
      w_off = awq_uni(nrow != w_row ? noff : w_off);
      w_next = awq_uni(nrow != w_row ? nnext : w_next);
      w_row = awq_uni(nrow);
    }
    w_g = awq_uni(w_g + (more ? 1u : 0u));
    return ret;
  };

  // Flat: the lane's four elements of the step, their row and column; then 4k elements on.
  uint32_t f_at = 0, f_row = 0, f_col = 0;
  const uint32_t f_dr = kFlat ? awq_uni((4u << kshift) / P) : 0u, f_dc = kFlat ? awq_uni((4u << kshift) - f_dr * P) : 0u;
  const bool f_hi = kFlat && awq_uni((fcol + count + P - 1u) / P) > 64u;
  if constexpr (kFlat) {
    f_at = (R << kshift) + colw;
    const uint32_t x = fcol + f_at;
    f_row = x / P;
    f_col = x - f_row * P;
  }
  auto lane_row_offset = [&](uint32_t r) -> uint32_t {  // every lane of the wave takes part
    uint32_t o = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(r << 2), (int)base_lo);
    if (f_hi) {
      const uint32_t h = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(r << 2), (int)base_hi);
      o = r < 64u ? o : h;
    }
    return o;
  };
  // As the FP8 slab decode's load_flat: sh is 4 - the lane's elements in its row
  // (kLayFlatSplit), F the dword that ends with the row, F2 the next row's first.
  auto load_flat = [&](uint32_t &F, uint32_t &F2, uint32_t &sh) -> uint32_t {
    const bool ok = f_at < count;
    const uint32_t off = lane_row_offset(f_row) + f_col;
    uint32_t so = ok ? off << 1 : kSlabOutPast;
    if constexpr (kLay == kLayFlat) {
      F = __builtin_amdgcn_raw_buffer_load_b32(r_q, ok ? off : kSlabInPast, 0, 0);
    } else {
      const uint32_t left = P - f_col;  // columns to the row's end
      sh = ok && left < 4u ? 4u - left : 0u;
      const bool more = sh != 0u && f_at + left < count;
      const uint32_t next = __builtin_amdgcn_ballot_w64(more) ? lane_row_offset(f_row + 1u) : 0u;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_q, ok ? off - sh : kSlabInPast, 0, 0);
      F2 = __builtin_amdgcn_raw_buffer_load_b32(r_q, more ? next : kSlabInPast, 0, 0);
      so = sh ? kSlabOutPast : so;
    }
    f_at += 4u << kshift;
    f_row += f_dr;
    f_col += f_dc;
    const bool carry = f_col >= P;
    f_row += carry ? 1u : 0u;
    f_col -= carry ? P : 0u;
    return so;
  };

  auto lookup = [&](uint32_t qb, uint32_t x) -> uint32_t {  // entry of int4 value qb at peek bits x[12:2]
    return *reinterpret_cast<const uint32_t *>(lbytes + ((qb & 15u) << 13 | (x & 0x1FFCu)));
  };
  // sh, gi (kLayFlatSplit): the step's sh as load_flat gave it, and its number.
  auto step = [&](auto is_tail, uint32_t F, uint32_t so, uint32_t sh = 0, uint32_t gi = 0) {
    constexpr bool kTail = decltype(is_tail)::value;
    const auto p1 = __builtin_amdgcn_permlane32_swap(F, F, false, false);
    const uint32_t gq = __builtin_amdgcn_perm(p1[1], p1[0], selA);
    const auto p2 = __builtin_amdgcn_permlane16_swap(gq, gq, false, false);
    const uint32_t fq = __builtin_amdgcn_perm(p2[1], p2[0], selB);  // byte j = element j's int4 byte
    const uint32_t np0 = np;
    uint32_t e[4];
    {
      // 64 stream bits at -np: the first two codes come from the high word; the
      // second window starts where they end, cut from the same two words.
      uint32_t hi, lo;
      window64(np, hi, lo);
      uint32_t s = 19u;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (kFlat || !kTail || (uint32_t)j < tail) {
          e[j] = lookup(fq >> (8 * j), __builtin_amdgcn_alignbit(hi, hi, s));
          if (kFlat && kTail) e[j] = (uint32_t)j < tail ? e[j] : 0u;  // by lane
          s -= e[j];
        } else {
          e[j] = 0u;
        }
      }
      // the window 19 - s bits on: ({hi, lo} >> (32 - (19 - s)))[31:0] (the
      // shift is taken mod 32, so the entries' high bits in s do not matter)
      const uint32_t win = __builtin_amdgcn_alignbit(hi, lo, s + 13u);
      uint32_t s2 = 19u;
#pragma unroll
      for (int j = 2; j < 4; ++j) {
        if (kFlat || !kTail || (uint32_t)j < tail) {
          e[j] = lookup(fq >> (8 * j), __builtin_amdgcn_alignbit(win, win, s2));
          if (kFlat && kTail) e[j] = (uint32_t)j < tail ? e[j] : 0u;
          s2 -= e[j];
        } else {
          e[j] = 0u;
        }
      }
      np += (uint32_t)((int32_t)(s << 16) >> 16) + (uint32_t)((int32_t)(s2 << 16) >> 16) - 38u;
    }
    if constexpr (kEsc) {
      // A wave with an ESC code in the step decodes the step again one code at
      // a time, every lane: the slow decode gives the fast one's result where
      // there is no ESC, so no lane needs to be masked off.
      if (__builtin_amdgcn_ballot_w64(((e[0] | e[1] | e[2] | e[3]) & kAwqEscBit) != 0u)) {
        uint32_t p = np0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (!kTail || (uint32_t)j < tail) {
            const uint32_t w = window(p);
            uint32_t ent = lookup(fq >> (8 * j), w >> 19);
            p -= ent & 15u;
            if (ent & kAwqEscBit) {
              ent = window(p) & 0xFFFF0000u;  // the symbol: the 16 raw bits after the code
              p -= 16u;
            }
            e[j] = ent;
          }
        }
        np = p;
      }
    }
    const auto t0 = __builtin_amdgcn_permlane32_swap(e[0], e[2], false, false);
    const auto t1 = __builtin_amdgcn_permlane32_swap(e[1], e[3], false, false);
    const uint32_t a = __builtin_amdgcn_perm(t0[1], t0[0], 0x07060302u);
    const uint32_t b = __builtin_amdgcn_perm(t1[1], t1[0], 0x07060302u);
    const auto t2 = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    const v2u o = {__builtin_amdgcn_perm(t2[1], t2[0], 0x05040100u), __builtin_amdgcn_perm(t2[1], t2[0], 0x07060302u)};
    if constexpr (kLay == kLayRows) __builtin_amdgcn_raw_buffer_store_b64(o, r_out, vf_al << 1, awq_uni(so) << 1, kSlabCacheNT);
    else __builtin_amdgcn_raw_buffer_store_b64(o, r_out, so, 0, kSlabCacheNT);
    if constexpr (kLay == kLayFlatSplit) {
      if (__builtin_amdgcn_ballot_w64(sh != 0u)) {
        const uint32_t f = (((gi << 2) + R) << kshift) + colw, x = fcol + f;
        const uint32_t row = x / P, in_row = 4u - sh;
        const uint32_t o0 = lane_row_offset(row) + (x - row * P), o1 = lane_row_offset(row + 1u) - in_row;
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
          const bool ok = sh != 0u && f + j < count;
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o[j / 2u] >> (16u * (j & 1u))), r_out,
                                                ok ? ((j < in_row ? o0 : o1) + j) << 1 : kSlabOutPast, 0, 0);
        }
      }
    }
  };

  uint32_t Fr[DF], SOr[DF];
  uint32_t F2r[kLay == kLayFlatSplit ? DF : 1], SHr[kLay == kLayFlatSplit ? DF : 1];
  auto load_ring = [&](int u) {
    if constexpr (kFlat) SOr[u] = load_flat(Fr[u], F2r[kLay == kLayFlatSplit ? u : 0], SHr[kLay == kLayFlatSplit ? u : 0]);
    else SOr[u] = load_step(Fr[u]);
  };
  auto ring_bytes = [&](int u) -> uint32_t {
    if constexpr (kLay == kLayFlatSplit) return __builtin_amdgcn_alignbit(F2r[u], Fr[u], SHr[u] << 3);
    return Fr[u];
  };
#pragma unroll
  for (int u = 0; u < DF; ++u) load_ring(u);
  reserve(std::true_type{});  // the first request (nothing to feed yet)
  // Wave priorities, as in the FP8 slab decode: the issue arbiter favours the
  // oldest ready wave, so a wave lowers its priority by one level per quarter
  // of its steps, counted from a head start that grows with its age.
#ifndef MPS_AWQ_PRIO
#define MPS_AWQ_PRIO 1
#endif
#ifndef MPS_AWQ_PRIO_LEAD
#define MPS_AWQ_PRIO_LEAD 16
#endif
  const uint32_t quarter = awq_uni(nfull / 4u > 0u ? nfull / 4u : 1u);
  const uint32_t lead = (3u - (awq_uni(qlane) >> 8)) * (quarter * MPS_AWQ_PRIO_LEAD / 16u);  // head start (steps)
  uint32_t prio = 3u - (lead / quarter < 3u ? lead / quarter : 3u);
  uint32_t prio_at = (lead / quarter + 1u) * quarter - lead;  // steps done when the priority next drops
  if (MPS_AWQ_PRIO) {
    if (prio == 3u) __builtin_amdgcn_s_setprio(3);
    else if (prio == 2u) __builtin_amdgcn_s_setprio(2);
    else if (prio == 1u) __builtin_amdgcn_s_setprio(1);
    else __builtin_amdgcn_s_setprio(0);
  }
  uint32_t g = 0;
  for (; g + (uint32_t)DF <= nfull; g += (uint32_t)DF) {
    if (MPS_AWQ_PRIO && g >= prio_at) {
      prio_at += quarter;
      --prio;
      if (prio == 2u) __builtin_amdgcn_s_setprio(2);
      else if (prio == 1u) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
    }
#pragma unroll
    for (int u = 0; u < DF; ++u) {
      if constexpr (kLay == kLayFlatSplit) {
        const uint32_t F = ring_bytes(u), so = SOr[u], sh = SHr[u];
        load_ring(u);
        step(std::false_type{}, F, so, sh, g + (uint32_t)u);
      } else {
        const uint32_t F = Fr[u], so = SOr[u];
        load_ring(u);  // the step DF ahead
        step(std::false_type{}, F, so);
      }
      if (u % FE == FE - 1) bitstream_step();
    }
  }
  if (MPS_AWQ_PRIO) __builtin_amdgcn_s_setprio(0);
  // the last (fewer than DF) full steps and the partial one; their bytes are already loaded
#pragma unroll
  for (int u = 0; u < DF; ++u) {
    if (g + (uint32_t)u < gall) {
      if constexpr (kLay == kLayFlatSplit) {
        if (g + (uint32_t)u < nfull) step(std::false_type{}, ring_bytes(u), SOr[u], SHr[u], g + (uint32_t)u);
        else step(std::true_type{}, ring_bytes(u), SOr[u], SHr[u], g + (uint32_t)u);
      } else {
        if (g + (uint32_t)u < nfull) step(std::false_type{}, Fr[u], SOr[u]);
        else step(std::true_type{}, Fr[u], SOr[u]);
      }
      if (u % FE == FE - 1) bitstream_step();
    }
  }
  if (0u - np - 64u != pos_end) flag(status, MPS_STATUS_DESYNC);
}

// One slab-path bucket, checked by the plan: by-scale with one to 128 slabs of
// whole groups, or a row bucket of 1 .. 128 rows whose column range is P >= 4
// blocks of k, or flat (kRanged 3). Set-up in two levels of loads,
// each issued in full before any result is used: (1) the table ids, the
// wave's group rows and column starts (or the bucket's rows), the lane's start
// and end bits; (2) the tables' slices and the lane's first bitstream words.
// Thread tid expands entries 32c .. 32c+31 of the table of int4 value tid / 64
// (c = tid % 64).
// kRanged: 0 a whole bucket, 1 a row range (kind 2), 2 row ranges side by side
// (kind 3: k 256 or 512, the work-items [s k, (s + 1) k) decode range
// wk.range + s, from checkpoint rows range + s and range + s + 1 of a full
// [ranges + 1][k] set), 3 flat ranges side by side (kind 4: k 256, 512 or 1024,
// rows of any width, a range being slabs [range * range_rows, + range_rows) of
// the bucket); whole buckets compile without the range logic.
// A by-scale record may hold a run of buckets b with identical table ids: the
// first that gets past its checks (`tables`) loads and expands the tables and
// records in run_flags that it did (kRunTables) and whether they have an ESC
// entry (bit 1); the others reuse both.
// kAnyGroup: by-scale groups of any size slab_group allows; else 128 columns, as
// constants (with the size a variable the kernels' scalar registers spill more).
template <int kRanged, bool kAnyGroup>
__device__ __forceinline__ void awq_slab_bucket(const mps_awq_tensor &T, const AwqWork &wk, int64_t b, bool tables,
                                                uint32_t &run_flags, const uint32_t *__restrict__ ckpt,
                                                uint32_t *__restrict__ lut, uint32_t *__restrict__ region,
                                                uint32_t *status) {
  int tid;
  __asm__ volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"((int)threadIdx.x));
  const bool by_scale = T.group_col_start != nullptr;
  const int32_t ra = T.bucket_row_offsets[b], rb = T.bucket_row_offsets[b + 1];
  const int32_t groups = rb - ra;  // groups (by-scale) or rows
  const int32_t c0 = by_scale ? 0 : T.bucket_col_start[b];
  const int32_t cl = by_scale ? (kAnyGroup ? (int32_t)T.group_size : 128) : T.bucket_col_len[b];
  constexpr bool kFlat = kRanged == 3;
  constexpr bool kMulti = kRanged >= 2;
  const int32_t K = kMulti ? (int32_t)T.k : kAwqBlock;  // substreams (the block stride)
  const uint32_t ks = K == 256 ? 8u : K == 512 ? 9u : 10u;
  // by-scale: log2 of the group's columns and of a slab's groups
  uint32_t gsh = 7u;
  if constexpr (kAnyGroup) {
    const uint32_t z = by_scale ? (uint32_t)__builtin_ctz((uint32_t)cl | 0x400u) : 10u;
    gsh = z < 6u ? 6u : z > ks ? ks : z;
  }
  const uint32_t gpsh = ks - gsh;
  const bool shape_ok =
      kFlat ? groups >= 1 && cl >= 4 && cl < kFlatMaxCols && (int64_t)groups * cl < ((int64_t)1 << 31) && c0 >= 0 &&
                  (int64_t)c0 + cl <= T.m
      : by_scale ? ((kAnyGroup ? slab_group(cl, K) : T.group_size == 128) && groups >= (kMulti ? 1 : 1 << gpsh) && groups <= (kMulti ? 1024 : kSlabMaxSlabs << gpsh))
               : (groups >= 1 && groups <= 128 && cl >= 4 * K && cl % (kMulti ? 4 * K : K) == 0 && c0 >= 0 &&
                  (int64_t)c0 + cl <= T.m);
  const bool k_ok = kMulti ? (K == 256 || K == 512 || (kFlat && K == 1024)) : T.k == kAwqBlock;
  if (!shape_ok || !k_ok || ra < 0 || (int64_t)rb > T.num_row_indices) {
    if (tid == 0) flag(status, MPS_STATUS_BAD_BUCKET);
    return;
  }
  const uint32_t P = by_scale || kFlat ? 0u : (uint32_t)cl >> ks;
  // a row range (kinds 2, 3): its first row and row count; its lanes start and
  // end at checkpoints. Kind 3: this work-item's group of K (uniform per wave)
  // and its range; a last record's spare groups have no rows and only take
  // part in the barriers. A by-scale kind 3 range is a range of slabs (K / 128
  // groups each): [s0, s0 + ns) of the bucket's slabs.
  const bool ranged = kRanged != 0 && !by_scale && !kFlat;
  const bool from_ckpt = ranged || kMulti;  // lanes start (and end) at checkpoints
  const int32_t sub = kMulti ? (int32_t)awq_uni((uint32_t)tid >> ks) : 0;
  const int32_t range = wk.range + sub;
  // flat: the range's elements, its first row and that element's column there
  uint32_t f_elems = 0, f_row = 0, f_col = 0;
  if constexpr (kFlat) {
    const uint64_t step = (uint64_t)wk.range_rows << ks, at = (uint64_t)range * step, all = (uint64_t)groups * (uint32_t)cl;
    if (range < wk.ranges && at < all) {
      f_elems = awq_uni((uint32_t)(step < all - at ? step : all - at));
      f_row = awq_uni((uint32_t)at / (uint32_t)cl);
      f_col = awq_uni((uint32_t)at - f_row * (uint32_t)cl);
    }
  }
  const int32_t f_rows = f_elems ? (int32_t)awq_uni((f_col + f_elems + (uint32_t)cl - 1u) / (uint32_t)cl) : 0;
  const int32_t first_row = kFlat ? (int32_t)f_row : ranged ? range * wk.range_rows : 0;
  const int32_t nr_all = ranged ? (groups - first_row < wk.range_rows ? groups - first_row : wk.range_rows) : groups;
  const int32_t gps = kAnyGroup ? 1 << gpsh : K >> 7;  // by-scale: groups per slab
  const int32_t s0 = kMulti && by_scale ? range * wk.range_rows : 0;
  const int32_t ns_all = (groups + gps - 1) / gps - s0;
  const int32_t ns = kMulti && by_scale ? (ns_all < wk.range_rows ? ns_all : wk.range_rows) : 0;
  // rows of the range (rows), or the bucket's groups (by-scale); 0 for a spare group
  const int32_t nr = kFlat ? f_rows : kMulti ? (range < wk.ranges && (by_scale ? ns > 0 : nr_all > 0) ? nr_all : 0) : nr_all;
  if (!kMulti && nr <= 0) {
    if (tid == 0) flag(status, MPS_STATUS_BAD_BUCKET);
    return;
  }
  const uint32_t lane = kMulti ? (uint32_t)tid & (uint32_t)(K - 1) : (uint32_t)tid;  // within the group of K
  const uint32_t w = lane >> 6, wl = (uint32_t)tid & 63u;  // wave within the group of K, lane within the wave
  const uint32_t t = (w << 6) | (((uint32_t)tid & 15u) << 2) | (((uint32_t)tid >> 4) & 3u);  // substream
  const int q = tid >> 6, c = tid & 63;
  // level 1
  const __amdgpu_buffer_rsrc_t r_tab = awq_rsrc(T.bucket_table + b * 16, 64u);
  const int32_t gq = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_tab, (uint32_t)q * 4u, 0, 0);
  const __amdgpu_buffer_rsrc_t r_grow = awq_rsrc(T.row_indices + ra + first_row, (uint32_t)(nr > 0 ? nr : 0) * 4u);
  const __amdgpu_buffer_rsrc_t r_gcol =
      awq_rsrc(by_scale ? T.group_col_start + ra + (kFlat ? first_row : 0) : nullptr,
               by_scale ? (uint32_t)(kFlat ? nr : groups) * 4u : 0u);
  // by-scale: groups gps (s0 + wl) + wg and gps (s0 + wl + 64) + wg (slabs s0 + wl and s0 + wl + 64), where
  // wg is the wave's group within a slab, and its 64 columns start at wcol there; rows: rows wl and wl + 64
  const bool slabs = by_scale && !kFlat;
  const uint32_t wg = w >> (gsh - 6u), wcol = (w & ((1u << (gsh - 6u)) - 1u)) << 6;
  const uint32_t gi0 = slabs ? (uint32_t)gps * ((uint32_t)s0 + wl) + wg : wl;
  const uint32_t gi1 = slabs ? (uint32_t)gps * ((uint32_t)s0 + wl + 64u) + wg : wl + 64u;
  const int32_t row0 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_grow, gi0 * 4u, 0, 0);
  const int32_t col0 = by_scale ? (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_gcol, gi0 * 4u, 0, 0) : c0;
  const int32_t row1 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_grow, gi1 * 4u, 0, 0);
  const int32_t col1 = by_scale ? (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_gcol, gi1 * 4u, 0, 0) : c0;
  const __amdgpu_buffer_rsrc_t r_sb = awq_rsrc(T.bucket_thread_startbit + b * (kAwqBlock + 1), (kAwqBlock + 1) * 4u);
  // kind 2: ranges - 1 checkpoint rows (between ranges); kind 3: ranges + 1 (the ends too)
  const uint32_t ck_rows = !from_ckpt ? 0u : kMulti ? (uint32_t)wk.ranges + 1u : (uint32_t)wk.ranges - 1u;
  const __amdgpu_buffer_rsrc_t r_ck = awq_rsrc(from_ckpt ? ckpt + wk.ckpt : nullptr, ck_rows * (uint32_t)K * 4u);
  // one unconditional load each from the chosen array (a load under a branch is
  // waited for where the branch joins, which would serialise the set-up's loads)
  const bool from_ck = from_ckpt && (kMulti || wk.range > 0), to_ck = from_ckpt && (kMulti || wk.range + 1 < wk.ranges);
  const __amdgpu_buffer_rsrc_t r_pos = from_ck ? r_ck : r_sb;
  const __amdgpu_buffer_rsrc_t r_end = to_ck ? r_ck : r_sb;
  const uint32_t ck0 = kMulti ? (uint32_t)range : (uint32_t)(wk.range - 1);  // checkpoint row of the range's start
  const uint32_t live = kMulti && nr <= 0 ? kSlabBsPast : 0u;               // spare groups load nothing
  const uint32_t pos = __builtin_amdgcn_raw_buffer_load_b32(
      r_pos, live | (from_ck ? ((ck0 << ks) + t) * 4u : t * 4u), 0, 0);
  const uint32_t pos_end = __builtin_amdgcn_raw_buffer_load_b32(
      r_end, live | (to_ck ? (((ck0 + 1u) << ks) + t) * 4u : (t + 1u) * 4u), 0, 0);
  const uint64_t bucket_bit = (uint64_t)T.bucket_bit_base[b];
  // Offset of the lane's first bitstream words and the descriptor's bitstream
  // fields, computed here, before the table loads (the words themselves are
  // loaded after the table expansion).
  uint32_t off0 = ((pos >> 5) & ~1u) * 4u;
  __asm__ volatile("" : "+v"(off0));
  const uint8_t *bs_ptr = reinterpret_cast<const uint8_t *>(T.bitstream);
  int64_t bs_words = T.bitstream_words;
  __asm__ volatile("" : "+s"(bs_ptr), "+s"(bs_words));
  // level 2
  const bool tab_ok = gq >= 0 && gq < T.num_tables;
  const bool tab_load = tables && tab_ok;
  const uint32_t G = (uint32_t)(T.num_tables > 0 ? T.num_tables : 0);
  const __amdgpu_buffer_rsrc_t r_syms = awq_rsrc(T.decode_syms, G * (uint32_t)(kAwqTable * 2));
  const __amdgpu_buffer_rsrc_t r_lens = awq_rsrc(T.decode_lens, G * (uint32_t)kAwqPacked);
  uint4 sv[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto x = __builtin_amdgcn_raw_buffer_load_b128(
        r_syms, tab_load ? (uint32_t)gq * (uint32_t)(kAwqTable * 2) + (uint32_t)c * 64u + 16u * (uint32_t)i : kSlabBsPast,
        0, 0);
    sv[i] = make_uint4(x[0], x[1], x[2], x[3]);
  }
  const auto ln = __builtin_amdgcn_raw_buffer_load_b128(
      r_lens, tab_load ? (uint32_t)gq * (uint32_t)kAwqPacked + (uint32_t)c * 16u : kSlabBsPast, 0, 0);
  if (tables && tid == 0) {
    bool bad = false;
#pragma unroll
    for (int qq = 0; qq < 16; ++qq) {
      const int32_t id = gload(T.bucket_table + b * 16 + qq);
      bad |= id < -1 || id >= T.num_tables;
    }
    if (bad) flag(status, MPS_STATUS_BAD_TABLE);
  }
  // expansion: entry p of value q = sym << 16 | (nibble 15 ? 27 : nibble); a
  // missing table is all ESC entries, as the reference decodes it. The
  // nibbles go to bytes (even entries in `fl`, odd ones in `fh`); a byte b
  // becomes b + 12 when it is 15 (the carry of b + 1 into bit 4, times 3/4
  // of 16), and one byte permute per entry joins it with its symbol.
  uint32_t esc_seen = tab_ok ? 0u : 1u;
  if (tables) {
    const uint32_t nib32[4] = {ln[0], ln[1], ln[2], ln[3]};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = nib32[i] & 0x0F0F0F0Fu, hi = (nib32[i] >> 4) & 0x0F0F0F0Fu;
      const uint32_t el = ((lo + 0x01010101u) & 0x10101010u) >> 2, eh = ((hi + 0x01010101u) & 0x10101010u) >> 2;
      esc_seen |= el | eh;
      const uint32_t fl = tab_ok ? lo + el + (el << 1) : 0x1B1B1B1Bu;
      const uint32_t fh = tab_ok ? hi + eh + (eh << 1) : 0x1B1B1B1Bu;
      const uint32_t w4[4] = {sv[i].x, sv[i].y, sv[i].z, sv[i].w};  // zero for a missing table
      uint32_t e[8];
#pragma unroll
      for (int cc = 0; cc < 4; ++cc) {
        e[2 * cc] = __builtin_amdgcn_perm(w4[cc], fl, 0x05040C00u | (uint32_t)cc);
        e[2 * cc + 1] = __builtin_amdgcn_perm(w4[cc], fh, 0x07060C00u | (uint32_t)cc);
      }
      uint4 *dst = reinterpret_cast<uint4 *>(lut + (q << kAwqL) + 32 * c + 8 * i);
      dst[0] = make_uint4(e[0], e[1], e[2], e[3]);
      dst[1] = make_uint4(e[4], e[5], e[6], e[7]);
    }
  }
  // The lane's first four bitstream words (two 16-byte loads), issued once the
  // wave's own tables are in LDS: issued before, these scattered loads (64
  // lines a wave) queued ahead of the other waves' table loads; here they
  // overlap the other waves' expansion and the barriers, and the decode waits
  // for them after issuing its first int4 loads.
  __builtin_amdgcn_sched_barrier(0);
  uint2 first[4];
  {
    const uint64_t bs_bytes = bs_words > 0 ? (uint64_t)bs_words * 8u : 0u;
    const uint64_t base_byte = bucket_bit >> 3;
    const uint32_t win_bytes = base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
    const __amdgpu_buffer_rsrc_t r_bs = awq_rsrc(bs_ptr + (base_byte < bs_bytes ? base_byte : 0), win_bytes);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(r_bs, off0 + 16u * (uint32_t)i, 0, 0);
      first[2 * i] = make_uint2(x[0], x[1]);
      first[2 * i + 1] = make_uint2(x[2], x[3]);
    }
  }
  // group bases of this wave for slabs wl and wl + 64 (by-scale), or the
  // offsets of rows wl and wl + 64 with the column start (rows)
  const uint32_t m = (uint32_t)T.m;
  auto gbase = [&](uint32_t gi, int32_t row, int32_t col, bool &bad) -> uint32_t {
    if (gi >= (uint32_t)nr) return 0u;
    bad |= row < 0 || (int64_t)row >= T.n || col < 0 || (int64_t)col + cl > T.m;
    // (128 columns spelt out: what this lambda captures moves the compiler's register choices, and
    // with wcol in every kernel awq_decode_plan<3> and <5> reloaded 5788 and 5314 spilled scalars
    // instead of 3554 and 3370: layers that mix row ranges with k = 256 or tiny buckets 238 -> 229 us.)
    if constexpr (kAnyGroup) return (uint32_t)row * m + (uint32_t)col + (slabs ? wcol : 0u);
    else return (uint32_t)row * m + (uint32_t)col + (by_scale ? ((w & 1u) << 6) : 0u);
  };
  bool bad_row = kFlat && nr > kFlatMaxRows;
  const uint32_t base_lo = gbase(gi0, row0, col0, bad_row);
  const uint32_t base_hi = gbase(gi1, row1, col1, bad_row);
  uint32_t *s_wflag = region + 5 * kAwqBlock;  // queue slot 5 until the decode starts
  {
    const uint32_t wf = (__builtin_amdgcn_ballot_w64(bad_row) ? 1u : 0u) |
                        (__builtin_amdgcn_ballot_w64(esc_seen != 0u) ? 2u : 0u);
    if (wl == 0) s_wflag[tid >> 6] = wf;  // one word per wave of the workgroup
  }
  __syncthreads();
  uint32_t bflags = 0;
#pragma unroll
  for (int i = 0; i < kAwqBlock / 64; ++i) bflags |= s_wflag[i];
  __syncthreads();  // the flag words belong to the queue from here on
  bflags = awq_uni(bflags);
  if (tables) run_flags = (bflags & 2u) | kRunTables;
  else bflags = (bflags & ~2u) | (run_flags & 2u);
  if (bflags & 1u) {
    if (tid == 0) flag(status, MPS_STATUS_BAD_ROW);
    return;
  }
  // this wave's elements per lane: by-scale, every full slab and the partial
  // last one when its group wg exists; rows, rows x P
  const uint32_t count = by_scale ? ((uint32_t)groups >> gpsh) + (wg < ((uint32_t)groups & ((uint32_t)gps - 1u)) ? 1u : 0u)
                                  : (uint32_t)nr * P;
  const bool esc = (bflags & 2u) != 0u;
  if constexpr (kMulti) {
    if (nr <= 0) return;  // a spare group
    if constexpr (kFlat) {
#define MPS_AWQ_FLAT(ESC, LAY)                                                                                     \
  awq_slab_decode<ESC, LAY, 0>(T, lut, region, (uint32_t)tid, lane, ks, f_elems, base_lo, base_hi, (uint32_t)nr,    \
                               (uint32_t)cl, bucket_bit, first, pos, pos_end, status, f_col)
      if (cl % 4 == 0) {
        if (esc) MPS_AWQ_FLAT(true, kLayFlat);
        else MPS_AWQ_FLAT(false, kLayFlat);
      } else {
        if (esc) MPS_AWQ_FLAT(true, kLayFlatSplit);
        else MPS_AWQ_FLAT(false, kLayFlatSplit);
      }
#undef MPS_AWQ_FLAT
      return;
    }
    if (by_scale) {
      // this wave's slabs in the range: those whose group gps i + wg exists
      const int32_t cw = groups > (int32_t)wg ? (groups - (int32_t)wg + gps - 1) / gps : 0;
      const int32_t cnt = cw - s0 < 0 ? 0 : cw - s0 < ns ? cw - s0 : ns;
      if (esc)
        awq_slab_decode<true, kLayGroups, 0>(T, lut, region, (uint32_t)tid, lane, ks, (uint32_t)cnt, base_lo,
                                             base_hi, (uint32_t)groups, 0u, bucket_bit, first, pos, pos_end, status);
      else
        awq_slab_decode<false, kLayGroups, 0>(T, lut, region, (uint32_t)tid, lane, ks, (uint32_t)cnt, base_lo,
                                              base_hi, (uint32_t)groups, 0u, bucket_bit, first, pos, pos_end, status);
      return;
    }
    if (esc)
      awq_slab_decode<true, kLayRows, 0>(T, lut, region, (uint32_t)tid, lane, ks, count, base_lo, base_hi,
                                         (uint32_t)nr, P, bucket_bit, first, pos, pos_end, status);
    else
      awq_slab_decode<false, kLayRows, 0>(T, lut, region, (uint32_t)tid, lane, ks, count, base_lo, base_hi,
                                          (uint32_t)nr, P, bucket_bit, first, pos, pos_end, status);
    return;
  }
#define MPS_AWQ_SLAB(ESC, LAY)                                                                               \
  awq_slab_decode<ESC, LAY>(T, lut, region, (uint32_t)tid, (uint32_t)tid, 10u, count, base_lo, base_hi,       \
                            (uint32_t)nr, P, bucket_bit, first, pos, pos_end, status)
  if (by_scale) {
    if (esc) MPS_AWQ_SLAB(true, kLayGroups);
    else MPS_AWQ_SLAB(false, kLayGroups);
  } else if (P % 4u == 0u) {
    if (esc) MPS_AWQ_SLAB(true, kLayRows);
    else MPS_AWQ_SLAB(false, kLayRows);
  } else {
    if (esc) MPS_AWQ_SLAB(true, kLayRowsWrap);
    else MPS_AWQ_SLAB(false, kLayRowsWrap);
  }
#undef MPS_AWQ_SLAB
}

// A later bucket of a by-scale run, once the run's tables are in the LDS:
// each wave sets up and decodes its own part without meeting the others. A
// lane's queue slots and a wave's group bases are its own, so nothing here
// needs the workgroup: a wave that ends one bucket starts the next one's
// loads while the others still decode, and their latency hides behind them.
// A row or column out of range in a wave's groups flags and skips that
// wave's part (its groups only). 128-column groups only: kernels of other sizes
// run such buckets through awq_slab_bucket, after a barrier (as a template over
// the size, this function cost awq_decode_plan<2>, which it serves too, 1400
// reloads of spilled scalar registers: a 30 us launch of row buckets took 33).
__device__ __forceinline__ void awq_slab_bucket_wave(const mps_awq_tensor &T, int64_t b, uint32_t run_flags,
                                                     const uint32_t *__restrict__ lut,
                                                     uint32_t *__restrict__ region, uint32_t *status) {
  int tid;
  __asm__ volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"((int)threadIdx.x));
  const int32_t ra = T.bucket_row_offsets[b], rb = T.bucket_row_offsets[b + 1];
  const int32_t groups = rb - ra;
  if (!(groups >= 8 && groups <= 8 * kSlabMaxSlabs && T.group_size == 128) || ra < 0 ||
      (int64_t)rb > T.num_row_indices || T.k != kAwqBlock) {
    if (tid == 0) flag(status, MPS_STATUS_BAD_BUCKET);
    return;
  }
  const uint32_t w = (uint32_t)tid >> 6, wl = (uint32_t)tid & 63u;
  const uint32_t t = (w << 6) | (((uint32_t)tid & 15u) << 2) | (((uint32_t)tid >> 4) & 3u);  // substream
  // level 1: this wave's groups 8 wl + w/2 and 8 (wl + 64) + w/2, the lane's start and end bits
  const __amdgpu_buffer_rsrc_t r_grow = awq_rsrc(T.row_indices + ra, (uint32_t)groups * 4u);
  const __amdgpu_buffer_rsrc_t r_gcol = awq_rsrc(T.group_col_start + ra, (uint32_t)groups * 4u);
  const uint32_t gi0 = 8u * wl + (w >> 1), gi1 = 8u * (wl + 64u) + (w >> 1);
  const int32_t row0 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_grow, gi0 * 4u, 0, 0);
  const int32_t col0 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_gcol, gi0 * 4u, 0, 0);
  const int32_t row1 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_grow, gi1 * 4u, 0, 0);
  const int32_t col1 = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_gcol, gi1 * 4u, 0, 0);
  const __amdgpu_buffer_rsrc_t r_sb = awq_rsrc(T.bucket_thread_startbit + b * (kAwqBlock + 1), (kAwqBlock + 1) * 4u);
  const uint32_t pos = __builtin_amdgcn_raw_buffer_load_b32(r_sb, t * 4u, 0, 0);
  const uint32_t pos_end = __builtin_amdgcn_raw_buffer_load_b32(r_sb, (t + 1u) * 4u, 0, 0);
  const uint64_t bucket_bit = (uint64_t)T.bucket_bit_base[b];
  // level 2: the lane's first bitstream words
  uint2 first[4];
  {
    const uint64_t bs_bytes = T.bitstream_words > 0 ? (uint64_t)T.bitstream_words * 8u : 0u;
    const uint64_t base_byte = bucket_bit >> 3;
    const uint32_t win_bytes = base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
    const __amdgpu_buffer_rsrc_t r_bs = awq_rsrc(
        reinterpret_cast<const uint8_t *>(T.bitstream) + (base_byte < bs_bytes ? base_byte : 0), win_bytes);
    const uint32_t off0 = ((pos >> 5) & ~1u) * 4u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto x = __builtin_amdgcn_raw_buffer_load_b128(r_bs, off0 + 16u * (uint32_t)i, 0, 0);
      first[2 * i] = make_uint2(x[0], x[1]);
      first[2 * i + 1] = make_uint2(x[2], x[3]);
    }
  }
  const uint32_t m = (uint32_t)T.m;
  auto gbase = [&](uint32_t gi, int32_t row, int32_t col, bool &bad) -> uint32_t {
    if (gi >= (uint32_t)groups) return 0u;
    bad |= row < 0 || (int64_t)row >= T.n || col < 0 || (int64_t)col + 128 > T.m;
    return (uint32_t)row * m + (uint32_t)col + ((w & 1u) << 6);
  };
  bool bad_row = false;
  const uint32_t base_lo = gbase(gi0, row0, col0, bad_row);
  const uint32_t base_hi = gbase(gi1, row1, col1, bad_row);
  if (__builtin_amdgcn_ballot_w64(bad_row)) {
    if (wl == 0) flag(status, MPS_STATUS_BAD_ROW);
    return;
  }
  const uint32_t count = (uint32_t)groups / 8u + ((w >> 1) < ((uint32_t)groups & 7u) ? 1u : 0u);
  if (run_flags & 2u)
    awq_slab_decode<true, kLayGroups>(T, lut, region, (uint32_t)tid, (uint32_t)tid, 10u, count, base_lo, base_hi,
                                      (uint32_t)groups, 0u, bucket_bit, first, pos, pos_end, status);
  else
    awq_slab_decode<false, kLayGroups>(T, lut, region, (uint32_t)tid, (uint32_t)tid, 10u, count, base_lo, base_hi,
                                       (uint32_t)groups, 0u, bucket_bit, first, pos, pos_end, status);
}

// Plan launch: workgroup i decodes buckets work[i].y .. work[i].y + work[i].z - 1
// of tensor work[i].x; work[i].w = 1 marks one slab-path bucket (above). A
// record's buckets have identical table ids (one scale),
// so they share the tables in LDS; each gets kAwqBlock / nsub work-items (its k
// lanes) and a kRowSlots / nsub slice of the row offsets. With k = 256 four
// buckets run in one workgroup instead of one (the tables allow one
// workgroup per CU).
// out_delta: elements every tensor's output moves by (a plan decoding into a
// buffer laid out like, but other than, the one it was created with).
// kRanges: bit 0, the plan has row ranges (kind 2 records); bit 1, row ranges
// side by side (kind 3); bit 2, tiny buckets (awq_tiny_lane); bit 3, flat ranges
// (kind 4); bit 4, by-scale groups of other sizes than 128 columns, flat or not. Plans without
// them launch the instantiation that leaves that path out: the range path's
// code in the same kernel measured 4.6% slower on a by-scale layer, the tiny
// path's 4.4% slower on a row-bucket layer.
// A bucket with no more elements than substreams codes one element a lane
// (k_eff = its element count), so staging its 16 tables in LDS (128 KiB) costs
// far more than its decode: each lane looks its one code up in the global
// tables instead (decode_huffman.cu:417-468 for one element: the peek, the
// length nibble, ESC with its 16 raw bits), and checks that the code ends
// where the next lane's begins.
__device__ __forceinline__ void awq_tiny_lane(const mps_awq_tensor &T, int64_t b, int32_t ra, int32_t c0, int32_t cl,
                                              int32_t k, int lane, uint32_t *status) {
  const uint32_t *__restrict__ sb = T.bucket_thread_startbit + b * ((int64_t)k + 1);
  const uint64_t pos0 = (uint64_t)T.bucket_bit_base[b] + gload(sb + lane);
  const uint64_t pos_end = (uint64_t)T.bucket_bit_base[b] + gload(sb + lane + 1);
  const bool empty = T.bitstream_words <= 0;
  const uint32_t *__restrict__ bs32 = empty ? g_awq_zero_chunks : reinterpret_cast<const uint32_t *>(T.bitstream);
  const uint64_t nchunks = empty ? 2u : (uint64_t)T.bitstream_words * 2u;
  const uint64_t cb = pos0 >> 5;
  // 64 bits from the code's first chunk: the code and an ESC payload (27 bits) fit after any skip < 32
  const uint64_t buf = (((uint64_t)chunk_at(bs32, nchunks, cb) << 32) | chunk_at(bs32, nchunks, cb + 1))
                       << (pos0 & 31u);
  const int32_t rr = lane / cl, cc = lane - rr * cl;
  const int64_t row = gload(T.row_indices + ra + rr);
  const int64_t col = T.group_col_start ? (int64_t)gload(T.group_col_start + ra + rr) : (int64_t)c0;
  const bool ok = row >= 0 && row < T.n && col >= 0 && col + cl <= T.m;
  if (!ok) flag(status, MPS_STATUS_BAD_ROW);
  const uint32_t idx = ok ? (uint32_t)(row * T.m + col) + (uint32_t)cc : 0u;
  const uint32_t q = ok ? (uint32_t)gload(T.int4 + idx) & 15u : 0u;
  const int32_t gid = gload(T.bucket_table + b * 16 + q);
  const uint32_t peek = (uint32_t)(buf >> (64 - kAwqL));
  uint32_t nib = 15u, sym = 0u;
  if (gid >= 0 && gid < T.num_tables) {  // a missing table decodes as ESC, as the reference's kernel does
    const uint32_t ln = gload(T.decode_lens + (size_t)gid * kAwqPacked + (peek >> 1));
    nib = (peek & 1u) ? (ln >> 4) & 15u : ln & 15u;
    sym = gload(T.decode_syms + (size_t)gid * kAwqTable + peek);
  }
  uint32_t len = nib;
  if (nib == 15u) {  // ESC: the code is L bits, then 16 raw bits (decode_huffman.cu:454-460)
    sym = (uint32_t)((buf << kAwqL) >> 48);
    len = kAwqL + 16u;
  }
  if (ok) *(__attribute__((address_space(1))) uint16_t *)(T.out + idx) = (uint16_t)sym;
  if (pos0 + len != pos_end) flag(status, MPS_STATUS_DESYNC);
}

template <int kRanges>
__device__ __forceinline__ void awq_plan_record(const mps_awq_tensor *__restrict__ tensors, const AwqWork &wk,
                                                const uint32_t *__restrict__ ckpt, uint32_t *status,
                                                int64_t out_delta, uint32_t *__restrict__ lut,
                                                uint32_t *__restrict__ s_base) {
  constexpr bool kAny = (kRanges & 16) != 0;
  const int4 w = make_int4(wk.tensor, wk.bucket, wk.nsub, wk.kind);
  mps_awq_tensor T = tensors[w.x];
  T.out += out_delta;
  uint32_t run_flags = 0;
  if (wk.kind == 1) {
    // a run of nsub buckets with identical table ids: the first bucket that
    // passes its checks loads the tables (the whole workgroup); the buckets
    // after it run wave by wave. Until the tables are in, every bucket takes
    // the workgroup path, whose checks are uniform, so all waves meet at its
    // barriers.
    for (int r = 0; r < wk.nsub; ++r) {
      const int64_t b = (int64_t)wk.bucket + r;
      if ((run_flags & kRunTables) == 0u) {
        awq_slab_bucket<0, kAny>(T, wk, b, true, run_flags, ckpt, lut, s_base, status);
      } else if constexpr (kAny) {
        __syncthreads();  // the waves' queues are free for the next bucket's flag words
        awq_slab_bucket<0, kAny>(T, wk, b, false, run_flags, ckpt, lut, s_base, status);
      } else {
        awq_slab_bucket_wave(T, b, run_flags, lut, s_base, status);
      }
    }
    return;
  }
  if constexpr ((kRanges & 1) != 0) {
    if (wk.kind == 2) {
      awq_slab_bucket<1, kAny>(T, wk, wk.bucket, true, run_flags, ckpt, lut, s_base, status);
      return;
    }
  }
  if constexpr ((kRanges & 8) != 0) {
    if (wk.kind == 4) {
      awq_slab_bucket<3, kAny>(T, wk, wk.bucket, true, run_flags, ckpt, lut, s_base, status);
      return;
    }
  }
  if constexpr ((kRanges & 2) != 0) {
    if (wk.kind == 3) {
      awq_slab_bucket<2, kAny>(T, wk, wk.bucket, true, run_flags, ckpt, lut, s_base, status);
      return;
    }
  }
  const int nsub = w.z;
  const int per = kAwqBlock / nsub;
  const int slots = kRowSlots / nsub;
  const int tid = threadIdx.x;
  const int sub = tid / per, lane = tid - sub * per;
  const int64_t b = (int64_t)w.y + (sub < nsub ? sub : 0);
  if ((kRanges & 4) != 0 && wk.tiny) {
    // Tiny buckets (the plan checked that each has no more elements than k):
    // no tables in LDS, no barrier. Compiled only into the plans that have
    // such records: the path costs the others registers.
    if (tid == 0) {
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int32_t g = gload(T.bucket_table + (int64_t)w.y * 16 + q);
        if (g < -1 || g >= T.num_tables) flag(status, MPS_STATUS_BAD_TABLE);
      }
    }
    if (sub >= nsub) return;
    const int32_t ra = T.bucket_row_offsets[b], rb = T.bucket_row_offsets[b + 1];
    const bool by_scale = T.group_col_start != nullptr;
    const int32_t c0 = by_scale ? 0 : T.bucket_col_start[b];
    const int32_t cl = by_scale ? (int32_t)T.group_size : T.bucket_col_len[b];
    if (rb <= ra) return;
    if (cl <= 0 || ra < 0 || (int64_t)rb > T.num_row_indices || (!by_scale && (c0 < 0 || (int64_t)c0 + cl > T.m))) {
      if (lane == 0) flag(status, MPS_STATUS_BAD_BUCKET);
      return;
    }
    const int64_t total = (int64_t)(rb - ra) * cl;
    if (lane < total && lane < (int)T.k) awq_tiny_lane(T, b, ra, c0, cl, (int32_t)T.k, lane, status);
    return;
  }

  // Tables of the record's first bucket, filled by all work-items (as awq_bucket<1>).
  {
    const int64_t b0 = w.y;
    int32_t gid[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) gid[q] = T.bucket_table[b0 * 16 + q];
    if (tid == 0) {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        if (gid[q] < -1 || gid[q] >= T.num_tables) flag(status, MPS_STATUS_BAD_TABLE);
    }
    const int64_t G = T.num_tables;
    if (G <= 0) {
      for (int i = tid; i < kLutEntries; i += kAwqBlock) lut[i] = 15u;
    } else {
      uint32_t sy[32], ln[32];
#pragma unroll
      for (int it = 0; it < 32; ++it) {
        const int i = it * kAwqBlock + tid;
        const int q = i >> kAwqL, p = i & (kAwqTable - 1);
        const uint32_t g = (gid[q] >= 0 && gid[q] < G) ? (uint32_t)gid[q] : 0u;
        sy[it] = T.decode_syms[(size_t)g * kAwqTable + p];
        ln[it] = T.decode_lens[(size_t)g * kAwqPacked + (p >> 1)];
      }
#pragma unroll
      for (int it = 0; it < 32; ++it) {
        const int i = it * kAwqBlock + tid;
        const int q = i >> kAwqL, p = i & (kAwqTable - 1);
        const bool ok = gid[q] >= 0 && gid[q] < G;
        lut[i] = ok ? (sy[it] << 16) | ((p & 1) ? (ln[it] >> 4) : (ln[it] & 15u)) : 15u;
      }
    }
  }
  // This work-item's bucket (decode_huffman.cu:417-444, :528-545).
  const int32_t ra = T.bucket_row_offsets[b], rb = T.bucket_row_offsets[b + 1];
  const int32_t rows = rb - ra;
  const bool by_scale = T.group_col_start != nullptr;
  const int32_t c0 = by_scale ? 0 : T.bucket_col_start[b];
  const int32_t cl = by_scale ? (int32_t)T.group_size : T.bucket_col_len[b];
  bool ok = sub < nsub && rows > 0;
  if (ok && (cl <= 0 || ra < 0 || (int64_t)rb > T.num_row_indices ||
             (!by_scale && (c0 < 0 || (int64_t)c0 + cl > T.m)))) {
    if (lane == 0) flag(status, MPS_STATUS_BAD_BUCKET);
    ok = false;
  }
  uint32_t *__restrict__ my_base = s_base + sub * slots;
  if (ok) {
    const int32_t staged = rows < slots ? rows : slots;
    for (int r = lane; r < staged; r += per) {
      const int64_t row = T.row_indices[ra + r];
      const int64_t col = by_scale ? (int64_t)T.group_col_start[ra + r] : (int64_t)c0;
      uint32_t base = kBadBase;
      if (row >= 0 && row < T.n && col >= 0 && col + cl <= T.m) base = (uint32_t)(row * T.m + col);
      else flag(status, MPS_STATUS_BAD_ROW);
      my_base[r] = base;
    }
  }
  __syncthreads();
  if (!ok) return;
  const int64_t total = (int64_t)rows * cl;
  const int32_t k = (int32_t)T.k;
  const int32_t k_eff = total < k ? (int32_t)total : k;
  if (lane >= k_eff) return;
  // nsub > 1 only for buckets whose rows all fit their slice (the plan checks)
  if (rows <= slots) awq_lane<true>(T, lut, my_base, b, ra, c0, cl, total, k, k_eff, lane, status);
  else awq_lane<false>(T, lut, my_base, b, ra, c0, cl, total, k, k_eff, lane, status);
}

// Record trace, in instrumented builds only (python -m mpserve_amd.build
// --define MPS_TRACE_ITEMS=1 --out LIB; mpserve_amd.item_trace reads it):
// record r < kAwqTraceRecs stores the real-time clock (100 MHz) at its start
// and after a closing barrier, kind << 32 | nsub, and its ordering key.
#ifndef MPS_TRACE_ITEMS
#define MPS_TRACE_ITEMS 0
#endif
#if MPS_TRACE_ITEMS
constexpr int kAwqTraceRecs = 8192;
__device__ uint64_t g_awq_trace[kAwqTraceRecs * 4];
#endif

// The plan kernel is persistent (one workgroup per CU) and takes its records
// from a queue, as the FP8 plan kernel does: workgroup g starts with record g;
// thread 0 takes a ticket t from queue[0] as its wave finishes a record, and
// the workgroup's next record is gridDim.x + t. The records are sorted largest
// first, so the CUs that drew small records take more of them, and no record
// pays a workgroup launch. The last workgroup to leave (queue[1] counts them)
// puts both words back to zero: launches of one queue must not overlap.
__device__ __forceinline__ uint32_t queue_add(uint32_t *q, uint32_t v) {
  return __hip_atomic_fetch_add((__attribute__((address_space(1))) uint32_t *)(q), v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
}

template <int kRanges>
__global__ __launch_bounds__(kAwqBlock) void awq_decode_plan(const mps_awq_tensor *__restrict__ tensors,
                                                             const AwqWork *__restrict__ work, int64_t nwork,
                                                             const uint32_t *__restrict__ ckpt, uint32_t *status,
                                                             int64_t out_delta, uint32_t *queue) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[kRowSlots + kLutEntries];  // as in awq_decode_kernel
  uint32_t *s_base = lds, *lut = lds + kRowSlots;
  if ((int64_t)blockIdx.x < nwork) {
    int64_t r = blockIdx.x;
    for (;;) {
#if MPS_TRACE_ITEMS
      const uint64_t tr0 = __builtin_amdgcn_s_memrealtime();
#endif
      const AwqWork wk = work[r];
      awq_plan_record<kRanges>(tensors, wk, ckpt, status, out_delta, lut, s_base);
      // The ticket is taken once wave 0 is through with the record, so the
      // next record goes to a workgroup that is about to be free (taken at the
      // record's start, a long record's successor would wait behind it); its
      // round trip overlaps the other waves' last steps. Every wave is then
      // done with the LDS (the record's queue, where the ticket goes), thread 0
      // hands out the ticket, and every wave has read it before the next
      // record's set-up writes the LDS.
      uint32_t t = 0;
      if (threadIdx.x == 0) t = queue_add(queue, 1u);
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (threadIdx.x == 0) lds[0] = t;
      __syncthreads();
      const int64_t next = (int64_t)gridDim.x + (int64_t)lds[0];
      __syncthreads();
#if MPS_TRACE_ITEMS
      if (threadIdx.x == 0 && r < kAwqTraceRecs) {
        uint64_t *tp = g_awq_trace + (size_t)r * 4;
        tp[0] = tr0;
        tp[1] = __builtin_amdgcn_s_memrealtime();
        tp[2] = ((uint64_t)(uint32_t)wk.kind << 32) | (uint32_t)wk.nsub;
        tp[3] = (uint64_t)wk.elems;
      }
#endif
      if (next >= nwork) break;
      r = next;
    }
  }
  if (threadIdx.x == 0) {
    if (queue_add(queue + 1, 1u) == gridDim.x - 1) {
      __hip_atomic_exchange((__attribute__((address_space(1))) uint32_t *)(queue), 0u, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_exchange((__attribute__((address_space(1))) uint32_t *)(queue + 1), 0u, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

}  // namespace
}  // namespace mps
