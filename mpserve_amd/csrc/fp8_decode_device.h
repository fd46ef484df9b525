// FP8 + Huffman-sidecar -> BF16 decode for MI355X (gfx950).
//
// Format (reference kernel/build_huffman.cu:786-925): bucket b owns rows
// row_indices[row_offsets[b] .. row_offsets[b+1]) x columns [col_start, col_start+col_len).
// Its elements, flattened row-major, are dealt round-robin to k_eff = min(k, total)
// lanes: lane t codes e = t, t+k_eff, ...; each lane's codes form one MSB-first
// substream starting at bit bucket_bit_base[b] + bucket_thread_startbit[b][t].
// A code is looked up with the next 7 bits in the table of the key
// (bucket scale, fp8 byte of the element); a length nibble with bit 3 set marks
// ESC: 16 raw BF16 bits follow the code.
//
// Mapping to CDNA4: one workgroup of 1024 work-items per bucket (one lane per
// work-item, 16 wave64s). The bucket's 256 code tables are expanded once into
// LDS as 32-bit entries {sym:16 | len:3 | esc:1} (128 KiB), so one ds_read_b32
// per element resolves symbol, length and ESC. The bitstream is read as 32-bit
// chunks into a 64-bit MSB-aligned register buffer that is topped up whenever
// fewer than 32 bits remain, which keeps 7 + 16 bits available for any code
// plus its ESC payload.
//
// Included by fp8_decode.hip (the host side and the kernels of k = 1024, 256 and
// 512 slab buckets) and fp8_decode_flat.hip (the kernels that also decode flat
// buckets): each instantiates the kernels it launches.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mps_common.h"

namespace mps {

namespace {

constexpr int kL = 7;
constexpr int kTable = 1 << kL;           // 128 entries per code table
constexpr int kPacked = kTable / 2;       // 64 bytes of packed 4-bit lengths
constexpr int kBlock = 1024;              // work-items per bucket workgroup (>= k)
constexpr int kRowsLds = 256;             // row indices staged in LDS
// LDS code table entry: sym << 16 | esc << 4 | len. A shift by the whole entry
// shifts by len (its low 5 bits), and a 16-bit store of the high half stores sym.
constexpr uint32_t kEscBit = 1u << 4;
constexpr int kMaxDevices = 64;

// A load through a global (not generic) pointer: generic (flat) loads count in
// two counters, and an outstanding one makes the compiler turn every later
// memory wait into a full one.
template <typename V>
__device__ __forceinline__ V gload(const V *p) {
  return *(const __attribute__((address_space(1))) V *)(p);
}
// The same, not merged with its neighbours (which would make an unaligned wide
// load, and a generic one).
template <typename V>
__device__ __forceinline__ V gload_single(const V *p) {
  return *(const volatile __attribute__((address_space(1))) V *)(p);
}

// A store through a global pointer, for the same reason.
template <typename V>
__device__ __forceinline__ void gstore(V *p, V v) {
  *(__attribute__((address_space(1))) V *)(p) = v;
}

// Integrity flags go to a per-device status word passed to every launch. The
// atomic addresses global memory, not a generic pointer: an outstanding
// generic (flat) access makes the compiler turn every later memory wait into a
// full one.
__device__ __forceinline__ void flag(uint32_t *status, unsigned int f) {
  __hip_atomic_fetch_or((__attribute__((address_space(1))) uint32_t *)(status), f, __ATOMIC_RELAXED,
                        __HIP_MEMORY_SCOPE_AGENT);
}

// Stream chunk c (32 bits, stream order) of a bitstream of u64 words stored
// little-endian: word w's high half (its first 32 stream bits) is u32 2w+1.
// Past the end the last chunk is re-read instead of zeros, so the load needs no
// branch: a well-formed stream never consumes those bits, and a 7-bit peek that
// runs past its last code selects a table entry whose low bits do not matter.
__device__ __forceinline__ uint32_t chunk_at(const uint32_t *__restrict__ bs32, uint64_t nchunks, uint64_t c) {
  const uint64_t cc = c < nchunks ? c : nchunks - 1;
  return gload(bs32 + (cc ^ 1u));
}

__device__ uint32_t g_zero_chunks[2];

// Decode path of a bucket.
enum : int32_t { kPathBad = 0, kPathGeneric = 1, kPathFast = 2, kPathK1024 = 3, kPathFlat = 4 };
// A plan's fast-path item whose 1024 / k_eff row ranges of one bucket run side
// by side, one per k_eff work-items (WorkItem::path bit 4; bits 8..15: rows a range).
constexpr int32_t kMultiRange = 0x10;
// A flat item (a whole bucket, a range of its slabs, or several ranges side by
// side): `rows` holds its elements, bits 8.. of `path` the column its first
// element has in its first row, and bits 12.. of `k_eff` the slabs a range
// (kMultiRange). A run (kFlatRun) is several small whole buckets with the same
// tables, which are staged once: the item is the first of them, bits 8.. of
// `path` hold how many there are, and bits 12.. of `k_eff` where the others'
// records start among the plan's followers. The work-items' groups of k_eff
// take the run's buckets in turn.
constexpr int32_t kFlatRun = 0x20;
constexpr int kFlatColBits = 24, kFlatSlabShift = 12;

struct BucketShape {
  int32_t rows;   // 0 for a bad bucket
  int32_t k_eff;  // lanes with elements
  int32_t path;
};

// Shape and decode path of the bucket with row range [ra, rb) and column
// range [c0, c0 + cl) of tensor T. A range outside the tensor (or more rows
// than the LDS stages) makes the bucket bad. Shared by the plan builder (host)
// and the single-tensor kernel (device).
// flat_ok: the kernels to be launched decode flat buckets: those whose column
// range is no multiple of their k = 256, 512 or 1024 substreams, and at least 4
// (else the general path).
__host__ __device__ inline BucketShape bucket_shape(int32_t ra, int32_t rb, int32_t c0, int32_t cl,
                                                    const mps_fp8_tensor &T, bool flat_ok) {
  const bool ok = ra >= 0 && rb >= ra && (int64_t)rb <= T.num_row_indices && rb - ra <= kRowsLds && cl > 0 &&
                  c0 >= 0 && (int64_t)c0 + cl <= T.m;
  BucketShape s;
  s.rows = ok ? rb - ra : 0;
  const int64_t total = (int64_t)s.rows * cl;
  s.k_eff = (int32_t)(T.k < total ? T.k : (total > 0 ? total : 1));
  const uint64_t nm = (uint64_t)T.n * (uint64_t)T.m;
  const bool small_stream = (uint64_t)T.bitstream_words < 0x10000000ull;
  // k = 1024 path (any tensor below 2^31 elements) and the general fast path.
  const bool k1024 = ok && s.rows <= 128 && s.k_eff == 1024 && cl % 1024 == 0 && nm <= (1ull << 31) - 16u &&
                     small_stream;
  const bool fast = !k1024 && ok && s.rows <= 128 && cl % s.k_eff == 0 && nm <= (1ull << 29) && small_stream;
  const bool flat = flat_ok && ok && !k1024 && !fast && (T.k == 256 || T.k == 512 || T.k == 1024) &&
                    s.k_eff == T.k && s.rows <= 128 && cl >= 4 && cl < (1 << kFlatColBits) &&
                    nm <= (1ull << 31) - 16u && small_stream;
  s.path = !ok ? kPathBad : k1024 ? kPathK1024 : fast ? kPathFast : flat ? kPathFlat : kPathGeneric;
  return s;
}

// One unit of decode work: a bucket, or a range of its rows. Its tensor,
// column range, shape and the addresses of its per-bucket arrays. Substream
// (lane) t starts at bit bit_base + startbits[t] and ends at bit_base +
// endbits[t]: for a whole bucket, its start bits and the next lane's
// (endbits = startbits + 1); for a row range, the lane checkpoints the plan
// computed at the range's first and next range's first row. A plan builds
// these once (64 bytes: one scalar load per item, which leaves the table ids,
// row indices and start bits one dependent load away); the single-tensor
// kernel builds them on the fly.
struct WorkItem {
  int32_t tensor;       // index into the plan's descriptors
  int32_t c0, cl;       // col_start[b], col_len[b]
  int32_t rows, k_eff;
  int32_t path;                // decode path (bits 0..3); kMultiRange (bit 4): ranges side by side, bits 8..15 their rows
  int64_t bit_base;            // bucket_bit_base[b]
  const int32_t *table_ids;    // bucket_table + 256 b
  const uint32_t *startbits;   // per substream: start bit, relative to bit_base
  const uint32_t *endbits;     // per substream: end bit, relative to bit_base
  const int32_t *row_idx;      // row_indices + row_offsets[b] (+ the range's first row)
};
static_assert(sizeof(WorkItem) == 64, "one scalar load per work item");

// One lane: decode its substream.
//
// Memory discipline (gfx9 counts loads and stores in one in-order vmcnt): all
// global loads of a block of kDepth elements - the block's FP8 bytes and the
// next two bitstream chunks - are issued together one block ahead, and no load
// is issued inside the element loop. The wait at the top of a block is then a
// static vmcnt(kDepth) (the previous block's stores may stay in flight) on
// loads issued a whole block earlier.
//
// Bit supply: a 64-bit MSB-aligned buffer `buf` holding `cnt` bits, topped up
// by 32 bits from a 4-chunk register queue whenever cnt < 32. Without ESC a
// block consumes <= 7*kDepth = 56 bits, i.e. at most two chunks; the two
// chunks staged per block keep the queue at >= 2 chunks at every block start.
// ESC payloads can drain the queue; then a chunk is read directly (slow path).
constexpr int kDepth = 8;

template <typename Idx>
__device__ __forceinline__ void decode_lane(const mps_fp8_tensor &T, uint16_t *__restrict__ out,
                                            const uint32_t *__restrict__ lut,
                                            const int32_t *__restrict__ s_rows, int32_t lane, int32_t k_eff,
                                            int64_t total, int32_t c0, int32_t cl, uint64_t pos0, uint64_t pos_end,
                                            uint32_t *status) {
  const bool empty = T.bitstream_words <= 0;
  const uint32_t *__restrict__ bs32 = empty ? g_zero_chunks : reinterpret_cast<const uint32_t *>(T.bitstream);
  const uint64_t nchunks = empty ? 2u : (uint64_t)T.bitstream_words * 2u;

  // Initial fill: buffer from chunks c0, c0+1; queue = c0+2 .. c0+5; tail = c0+6.
  const uint64_t cb = pos0 >> 5;
  const int skip = (int)(pos0 & 31u);
  uint64_t buf = (((uint64_t)chunk_at(bs32, nchunks, cb) << 32) | chunk_at(bs32, nchunks, cb + 1)) << skip;
  int cnt = 64 - skip;
  uint32_t q0 = chunk_at(bs32, nchunks, cb + 2), q1 = chunk_at(bs32, nchunks, cb + 3);
  uint32_t q2 = chunk_at(bs32, nchunks, cb + 4), q3 = chunk_at(bs32, nchunks, cb + 5);
  int qn = 4;
  uint64_t tail = cb + 6;  // index of the first chunk not yet in buf/queue

  // Element walk e = lane + i*k_eff -> (rr, cc) = (e / cl, e % cl), incrementally.
  int32_t rr = lane / cl;
  int32_t cc = lane - rr * cl;
  const int32_t dr = k_eff / cl;
  const int32_t dc = k_eff - dr * cl;
  const int32_t count = (int32_t)((total - lane + k_eff - 1) / k_eff);
  const int32_t last_row = (int32_t)((total - 1) / cl);
  const Idx m = (Idx)T.m;
  const uint8_t *__restrict__ fp8 = T.fp8;

  // Addresses of the next kDepth elements (elements past `count` repeat the
  // lane's first element, whose address is always valid).
  const Idx first = (Idx)s_rows[rr] * m + (Idx)c0 + (Idx)cc;
  int32_t walked = 0;
  auto next_block = [&](Idx (&idx)[kDepth]) {
    int32_t rrs[kDepth], ccs[kDepth];
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      rrs[j] = rr < last_row ? rr : last_row;
      ccs[j] = cc;
      cc += dc;
      rr += dr;
      if (cc >= cl) {
        cc -= cl;
        rr += 1;
      }
    }
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      const Idx v = (Idx)s_rows[rrs[j]] * m + (Idx)c0 + (Idx)ccs[j];
      idx[j] = (walked + j < count) ? v : first;
    }
    walked += kDepth;
  };

  Idx ia[kDepth], ib[kDepth];
  uint32_t qa[kDepth], qb[kDepth];
  next_block(ia);
#pragma unroll
  for (int j = 0; j < kDepth; ++j) qa[j] = gload(fp8 + ia[j]);
  uint32_t s0 = chunk_at(bs32, nchunks, tail), s1 = chunk_at(bs32, nchunks, tail + 1);
  bool stale = false;  // the staged pair no longer starts at `tail`

  // Each branch merges its own chunk into buf: a loaded value that both
  // branches shared would force a full vmcnt wait on every element.
  auto refill = [&]() {
    if (cnt < 32) {
      if (qn > 0) {
        buf |= (uint64_t)q0 << (32 - cnt);
        q0 = q1;
        q1 = q2;
        q2 = q3;
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
  auto decode_one = [&](uint32_t q, Idx idx) {
    const uint32_t peek = (uint32_t)(buf >> (64 - kL));
    const uint32_t ent = lut[(q << kL) | peek];
    const int len = (int)(ent & 7u);
    buf <<= len;
    cnt -= len;
    uint32_t sym = ent >> 16;
    if (ent & kEscBit) {
      sym = (uint32_t)(buf >> 48);
      buf <<= 16;
      cnt -= 16;
    }
    gstore(out + idx, (uint16_t)sym);
    refill();
  };
  // One block: decode (qc, ic) while (qn_, in_) receive the next block's loads.
  auto block = [&](int32_t i0, uint32_t (&qc)[kDepth], Idx (&ic)[kDepth], uint32_t (&qnx)[kDepth],
                   Idx (&inx)[kDepth]) {
    // Append the pair staged one block ago if it is current and fits.
    if (!stale && qn <= 2) {
      q0 = (qn == 0) ? s0 : q0;
      q1 = (qn == 0) ? s1 : (qn == 1) ? s0 : q1;
      q2 = (qn == 1) ? s1 : (qn == 2) ? s0 : q2;
      q3 = (qn == 2) ? s1 : q3;
      qn += 2;
      tail += 2;
    }
    stale = false;
    next_block(inx);
#pragma unroll
    for (int j = 0; j < kDepth; ++j) qnx[j] = gload(fp8 + inx[j]);
    s0 = chunk_at(bs32, nchunks, tail);
    s1 = chunk_at(bs32, nchunks, tail + 1);
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
  // The next unread bit must be where the next lane's substream begins:
  // buf holds cnt bits and the queue qn chunks, all before chunk `tail`.
  if (tail * 32u - (uint64_t)(cnt + 32 * qn) != pos_end) flag(status, MPS_STATUS_DESYNC);
}

// Buffer resource over [base, base + bytes): raw buffer loads past the end
// return 0 and stores past the end are dropped (gfx9 V# with stride 0).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

// ---------------------------------------------------------------------------
// Fast path: buckets whose column range is a multiple of k_eff and that hold
// at most 128 rows (every bucket of a Llama-shaped tensor with k = 1024).
// Then every lane owns exactly rows * P elements (P = col_len / k_eff), and
// lane t's i-th element sits at row i / P, column c0 + t + (i % P) * k_eff:
// the walk is the same for every lane. It runs in scalar registers and feeds
// the FP8 loads and BF16 stores as the buffer soffset; the per-lane voffset
// is the lane (x2 for BF16).
//
// Bit supply. Each lane keeps the next chunks (32 stream bits) of its
// substream in an 8-deep LDS queue (slot-major: chunk c of lane t at
// [(c % 8) * 1024 + t], so a wave's accesses hit 64 distinct banks). Chunks
// arrive in aligned pairs (one u64 bitstream word): every block of kDepth
// elements each lane requests the next pair if it holds fewer than kAhead
// chunks ahead of its read position, and writes the pair requested kRing
// blocks earlier into the queue. The request is one unconditional
// buffer_load_dwordx2 per block (lanes that do not need a pair read out of
// range and ignore the zeros), so every block issues the same memory
// instructions - 1 bitstream load, kDepth FP8 loads, kDepth stores - and the
// compiler's in-order vmcnt waits stay kRing - 1 blocks deep. A group of kG = 4
// elements decodes from a 32-bit window cut out of two queued chunks (4 codes
// of <= 7 bits). An ESC code (16 raw bits follow) re-reads the window; a
// lane whose queue has run dry reads its two chunks from memory directly.
// ---------------------------------------------------------------------------
constexpr int kG = 4;
#ifndef MPS_DECODE_RING
#define MPS_DECODE_RING 4
#endif
constexpr int kRing = MPS_DECODE_RING;     // blocks in flight: FP8 ring slots and bitstream request slots
constexpr uint32_t kAhead = 7;             // request while fewer chunks than this are queued ahead
constexpr int kQSlots = 8;                 // LDS queue depth (chunks per lane)
constexpr uint32_t kPast = 0x40000000u;    // offset beyond every fast-path buffer (2*n*m <= 2^30)
constexpr uint32_t kBsPast = 0x80000000u;  // bitstream offset beyond every bucket's range
constexpr uint32_t kSlabPast = 0xFFFFFFF0u;  // BF16 byte offset beyond every k = 1024 output (2*n*m < 2^32 - 16)
constexpr int kCacheNT = 2;                  // buffer cache-policy bits: non-temporal (gfx950 NT)
// Cache-policy bits of the slab path's streams (tuning builds only; gfx950
// encodes sc0 = 1, nt = 2, sc1 = 16): the BF16 stores, the FP8 loads and the
// bitstream reserve loads.
#ifndef MPS_SLAB_OUT_CPOL
#define MPS_SLAB_OUT_CPOL kCacheNT
#endif
#ifndef MPS_SLAB_FP8_CPOL
#define MPS_SLAB_FP8_CPOL 0
#endif
#ifndef MPS_SLAB_BS_CPOL
#define MPS_SLAB_BS_CPOL 0
#endif

// LDS: the queue (kQSlots x kBlock u32) at offset 0, then 256 tables x 128 u32
// entries. During set-up the queue region also holds the fp8 -> table map; the
// generic path keeps the bucket's row indices there.
constexpr int kQWords = kQSlots * kBlock;
constexpr int kLutWords = 256 * kTable;
constexpr int kLdsWords = kQWords + kLutWords;

__device__ __forceinline__ uint32_t uni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ __forceinline__ void decode_rows_fast(const mps_fp8_tensor &T, uint16_t *out,
                                                 const uint32_t *__restrict__ lut,
                                                 uint32_t *__restrict__ queue, uint32_t qlane, uint32_t lane,
                                                 uint32_t k_eff, uint32_t rows, uint32_t P, uint32_t rowoff_lo,
                                                 uint32_t rowoff_hi, uint64_t bucket_bit,
                                                 uint2 first[3], uint32_t pos, uint32_t pos_end,
                                                 uint32_t *status) {
  // Uniform values computed on the VALU (the division above, selects) would
  // otherwise stay in VGPRs and drag the whole walk, and the buffer offsets it
  // feeds, into vector registers.
  k_eff = uni(k_eff);
  rows = uni(rows);
  P = uni(P);
  bucket_bit = ((uint64_t)uni((uint32_t)(bucket_bit >> 32)) << 32) | uni((uint32_t)bucket_bit);
  const uint32_t nm = (uint32_t)(T.n * T.m);
  const __amdgpu_buffer_rsrc_t r_fp8 = make_rsrc(T.fp8, nm);
  const __amdgpu_buffer_rsrc_t r_out = make_rsrc(out, 2u * nm);
  // Bitstream window of this bucket: from its 64-bit aligned base to the end.
  const uint64_t bs_bytes = T.bitstream_words > 0 ? (uint64_t)T.bitstream_words * 8u : 0u;
  const uint64_t base_byte = bucket_bit >> 3;
  const uint32_t win_bytes = base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
  const __amdgpu_buffer_rsrc_t r_bs =
      make_rsrc(reinterpret_cast<const uint8_t *>(T.bitstream) + (base_byte < bs_bytes ? base_byte : 0), win_bytes);
  // Stream chunk c (relative to the bucket base): u32 at byte (c ^ 1) * 4.
  auto chunk_mem = [&](uint32_t c) -> uint32_t {
    return __builtin_amdgcn_raw_buffer_load_b32(r_bs, (c ^ 1u) << 2, 0, 0);
  };
  auto qidx = [&](uint32_t c) -> uint32_t { return ((c & (kQSlots - 1)) * kBlock) + qlane; };

  // Initial queue: the three pairs loaded during set-up.
  const uint32_t rq0 = (pos >> 5) & ~1u;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    queue[qidx(rq0 + 2 * i)] = first[i].y;      // high half = first chunk of the pair
    queue[qidx(rq0 + 2 * i + 1)] = first[i].x;
  }
  uint32_t rq = rq0 + 6;  // next pair to request
  uint32_t wq = rq0 + 6;  // chunks below wq are (or were) in the queue

  // Uniform element walker: offset (elements) of the next element, then advance.
  const uint32_t count = rows * P;
  auto row_offset = [&](uint32_t r) -> uint32_t {
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)rowoff_lo, (int)(r & 63u));
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)rowoff_hi, (int)(r & 63u));
    return r < 64u ? a : b;
  };
  struct Walker {
    uint32_t r, p, off;
  };
  auto walk = [&](Walker &w) -> uint32_t {
    const uint32_t so = w.r < rows ? w.off : kPast;
    w.off += k_eff;
    if (++w.p == P) {
      w.p = 0;
      ++w.r;
      w.off = row_offset(w.r < rows ? w.r : rows - 1u);
    }
    return so;
  };
  Walker wl{0u, 0u, row_offset(0)}, ws{0u, 0u, row_offset(0)};

  uint32_t qr[kRing][kDepth];  // FP8 bytes, one ring slot per block
  uint2 inflight[kRing];       // requested pairs, one slot per block of the ring
  bool valid[kRing];
#pragma unroll
  for (int s = 0; s < kRing; ++s) valid[s] = false;
#pragma unroll
  for (int b = 0; b < kRing - 1; ++b)
#pragma unroll
    for (int j = 0; j < kDepth; ++j) qr[b][j] = __builtin_amdgcn_raw_buffer_load_b8(r_fp8, lane, walk(wl), 0);
#pragma unroll
  for (int s = 0; s < kRing; ++s) inflight[s] = make_uint2(0u, 0u);

  // Window of the next 32 stream bits at `pos`, from the queue or (if the
  // queue has not got them yet) from memory.
  auto window_at = [&](uint32_t p) -> uint32_t {
    const uint32_t c = p >> 5;
    uint32_t c0 = queue[qidx(c)];
    uint32_t c1 = queue[qidx(c + 1)];
    const bool dry = c + 1u >= wq;
    if (__builtin_amdgcn_ballot_w64(dry)) {
      if (dry) {
        c0 = chunk_mem(c);
        c1 = chunk_mem(c + 1);
        __asm__ volatile("" ::"v"(c0), "v"(c1));  // wait for the loads here, not at a later join
      }
    }
    const uint64_t w = ((uint64_t)c0 << 32) | c1;
    return (uint32_t)(w >> (32u - (p & 31u)));
  };

  auto decode_block = [&](uint32_t (&q)[kDepth], uint32_t nvalid) {
#pragma unroll
    for (int g = 0; g < kDepth; g += kG) {
      uint32_t win = window_at(pos);
#pragma unroll
      for (int j = g; j < g + kG; ++j) {
        if ((uint32_t)j < nvalid) {
          const uint32_t so = walk(ws);
          const uint32_t idx = (q[j] << kL) | (win >> (32 - kL));
          uint32_t ent = lut[idx];
          const uint32_t len = ent & 7u;
          win <<= len;
          pos += len;
          uint32_t sym = ent >> 16;
          if (ent & kEscBit) {
            // ESC: the symbol is the next 16 raw bits.
            sym = window_at(pos) >> 16;
            pos += 16;
            win = window_at(pos);
          }
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)sym, r_out, 2u * lane, 2u * so, 0);
        }
      }
    }
  };

  auto block = [&](int slot, uint32_t nvalid) {
    const int ps = slot;
    // 1. the pair requested kRing blocks ago joins the queue
    if (valid[ps]) {
      queue[qidx(wq)] = inflight[ps].y;
      queue[qidx(wq + 1)] = inflight[ps].x;
      wq += 2;
    }
    // 2. request the next pair if fewer than kAhead chunks are queued ahead
    const bool need = (int32_t)(rq - (pos >> 5)) < (int32_t)kAhead;
    {
      const uint32_t off = need ? rq * 4u : kBsPast;
      const auto v = __builtin_amdgcn_raw_buffer_load_b64(r_bs, off, 0, 0);
      inflight[ps] = make_uint2(v[0], v[1]);
    }
    valid[ps] = need;
    rq += need ? 2u : 0u;
    // 3. FP8 bytes kRing - 1 blocks ahead
#pragma unroll
    for (int j = 0; j < kDepth; ++j)
      qr[(slot + kRing - 1) % kRing][j] = __builtin_amdgcn_raw_buffer_load_b8(r_fp8, lane, walk(wl), 0);
    // 4. decode this block
    decode_block(qr[slot], nvalid);
  };

  const uint32_t nfull = count / kDepth;
  const uint32_t rem = count % kDepth;
  uint32_t b0 = 0;
  for (; b0 + kRing <= nfull; b0 += kRing) {
#pragma unroll
    for (int slot = 0; slot < kRing; ++slot) block(slot, kDepth);
  }
  // last round: remaining full blocks, then the partial block
#pragma unroll
  for (int slot = 0; slot < kRing; ++slot) {
    const uint32_t bi = b0 + (uint32_t)slot;
    if (bi < nfull) block(slot, kDepth);
    else if (bi == nfull && rem) block(slot, rem);
  }
  if (pos != pos_end) flag(status, MPS_STATUS_DESYNC);
}

// ---------------------------------------------------------------------------
// k = 1024, col_len = P * 1024 (every bucket of a checkpoint written with the
// compress CLI's default of 1024 substreams whose column range is a multiple
// of 1024: every Llama linear has P >= 4).
//
// Element i of a substream lives in slab i: the 1024 columns
// [c0 + 1024 (i % P), +1024) of the bucket's row i / P. Lane l of wave w,
// in 16-lane row R = l / 16 at position v = l % 16, decodes substream
// (column) t = 64w + 4v + R, four elements (one "group", slabs 4g..4g+3) at a
// time. Per group and wave:
//  - FP8: lane (R, v) loads the dword of slab 4g+R at columns 64w+4v..+3, so
//    each 16-lane row reads one contiguous 64-byte segment. A 4x4 byte
//    transpose between the lanes (0, v), (1, v), (2, v), (3, v) (one
//    permlane32 swap, one permlane16 swap and two byte permutes) leaves each
//    lane the four bytes of its own column.
//  - decode: one 32-bit window cut from the lane's LDS bitstream queue covers
//    the group's four codes (<= 7 bits each). The window is never shifted: the
//    7-bit peek of the code that starts o bits in is rotr(window, 23 - o)
//    bits 8..2, which with the FP8 byte << 9 is the code table entry's byte
//    address. The running shift s = 23 - o is decremented by whole entries
//    (their low bits are the length) and only its low 16 bits are kept.
//  - BF16: the inverse transpose (two permlane32 swaps, one permlane16 swap,
//    four byte permutes) gives lane (R, v) slab 4g+R's symbols for columns
//    64w+4v..+3, written with one 8-byte store; each 16-lane row again writes
//    one contiguous 128-byte segment.
// Bitstream: a lane requests up to 64 bytes at a time into a register reserve
// (aligned so that each request touches one half of a 128-byte line) and,
// once per four groups, moves 16 bytes from the reserve into its LDS queue;
// a window whose chunks are not queued is read from memory. FP8 dwords are
// loaded DF groups ahead. Every group issues the same vector-memory
// instructions, so the in-order vmcnt waits stay static.
//
// The queue here stores chunk h in slot (~h) & 7 (slot-major, 4 KiB per
// slot), and positions are kept negated (np = -p, with p biased by two
// chunks: queue chunk h holds stream chunk h - 2 and bit position p is kept
// as p + 64), so the window's slot addresses and its funnel shift come
// straight from np.
//
// ESC (kEsc: the bucket's tables hold ESC entries). An ESC entry's low half is
// 16 + len, so the running shift already steps over the 16 raw bits that
// follow the code; but four codes with ESC payloads can need more than one
// 32-bit window. A lane whose group holds an ESC code (one ballot per group)
// decodes that group again one code at a time, a window per code, taking the
// symbol from the 16 raw bits. ESC codes are rare (the symbols a key's
// 127 most frequent leave out), so the wave almost never takes that branch.
// ---------------------------------------------------------------------------
// kWrap: 0 when P % 4 == 0 (a group's four slabs lie in one row); 1 when P > 4
// and P % 4 != 0 (they may straddle two rows); 2 when P < 4 (they span two to
// four rows: slab i is row i / P, block i % P, taken per lane).
//
// 3 and 4: flat buckets, whose column range (any width cl >= 4) is no multiple
// of the k substreams. Slab i is then the k elements from i * k on in the
// bucket's row-major order, wherever its rows end: `rows` is the number of
// elements, `P` is cl, `fcol` the column of the first one. Each lane walks the
// row and column of its own four elements (a step of 4k elements is the same
// rows and columns for every lane, plus a carry) and takes the row's offset
// from the wave's row registers with a lane permute. The last slab may be short:
// a lane decodes as many elements of the last group as its substream has.
// With cl % 4 == 0 (kWrap 3) a lane's four elements share a row. Otherwise
// (kWrap 4) they may continue in the next one, after the first a of them: every
// group then loads two dwords, the one that ends with the row (lanes whose
// elements do not reach the row's end: their own four bytes) and the next
// row's first, joined by one funnel shift; and a group in which some lane's
// elements are split stores those with 2-byte stores.
// Measured, as plans, against the general path's byte loads and 2-byte stores
// over whole buckets: 3001 x 5000, k = 1024: 200 -> 25.6 us; 4096 x 4096 in 128 x
// 128 blocks (four groups a bucket, so mostly set-ups): 46 -> 35 us.
template <int kWrap, bool kEsc, int kShift>
__device__ __forceinline__ void decode_slab4(const mps_fp8_tensor &T, uint16_t *out, const uint32_t *__restrict__ lut,
                                             uint32_t *__restrict__ queue, uint32_t qlane, uint32_t lane,
                                             uint32_t kshift, uint32_t rows, uint32_t P,
                                             uint32_t rowoff_lo, uint32_t rowoff_hi, uint64_t bucket_bit,
                                             const uint2 (&first)[4], uint32_t pos, uint32_t pos_end,
                                             uint32_t *status, uint32_t fcol = 0) {
#ifndef MPS_SLAB_PREFETCH
#define MPS_SLAB_PREFETCH 8
#endif
  constexpr bool kFlat = kWrap >= 3;
  constexpr int DF = kWrap == 4 ? 4 : MPS_SLAB_PREFETCH;  // FP8 prefetch distance (groups)
  static_assert(DF >= 4 && DF % 4 == 0, "the bitstream is served once per four groups");
  rows = uni(rows);
  P = uni(P);
  kshift = kShift ? (uint32_t)kShift : uni(kshift);
  bucket_bit = ((uint64_t)uni((uint32_t)(bucket_bit >> 32)) << 32) | uni((uint32_t)bucket_bit);
  const uint32_t count = kFlat ? rows >> kshift : rows * P;  // elements per lane (flat: whole slabs)
  const uint32_t nfull = count >> 2;
  // Elements of the last, partial group (only when P % 4 != 0; flat: by lane).
  uint32_t tail = count & 3u;
  uint32_t gall = nfull + (tail ? 1u : 0u);
  if constexpr (kFlat) {
    const uint32_t rest = rows - (nfull << (kshift + 2u));
    const uint32_t t = (lane & ~63u) | ((lane & 15u) << 2) | ((lane >> 4) & 3u);  // the lane's substream
    tail = rest > t ? (rest - t + (1u << kshift) - 1u) >> kshift : 0u;
    gall = nfull + (rest ? 1u : 0u);
  }
  const uint32_t nm = (uint32_t)(T.n * T.m);
  const __amdgpu_buffer_rsrc_t r_fp8 = make_rsrc(T.fp8, nm);
  const __amdgpu_buffer_rsrc_t r_out = make_rsrc(out, 2u * nm);
  const uint64_t bs_bytes = T.bitstream_words > 0 ? (uint64_t)T.bitstream_words * 8u : 0u;
  const uint64_t base_byte = bucket_bit >> 3;
  const uint32_t win_bytes = base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
  const __amdgpu_buffer_rsrc_t r_bs =
      make_rsrc(reinterpret_cast<const uint8_t *>(T.bitstream) + (base_byte < bs_bytes ? base_byte : 0), win_bytes);

  const uint32_t lane4 = qlane << 2;  // the work-item's queue column
  const uint32_t R = (lane >> 4) & 3u;
  const uint32_t colw = (lane & ~63u) | ((lane & 15u) << 2);  // 64w + 4v
  const char *qbytes = reinterpret_cast<const char *>(queue);
  const char *lbytes = reinterpret_cast<const char *>(lut);
  // byte selectors of the FP8 transpose (v_perm: 0-3 pick the second operand's bytes, 4-7 the first's)
  const uint32_t selA = (R & 2u) ? 0x07060302u : 0x05040100u;
  const uint32_t selB = (R & 1u) ? 0x07030501u : 0x06020400u;

  // --- bitstream queue -----------------------------------------------------
  auto chunk_mem = [&](uint32_t h) -> uint32_t {  // biased chunk h from memory (h < 2: out of range, zeros)
    return __builtin_amdgcn_raw_buffer_load_b32(r_bs, ((h - 2u) ^ 1u) << 2, 0, 0);
  };
  // Chunks h (even) and h + 1: slots (~h) & 7 and the one below it.
  auto put_pair = [&](uint32_t h, uint32_t hi, uint32_t lo) {
    uint32_t *slot = queue + (((~h << 10) & 0x1800u) | qlane);
    slot[0] = lo;     // chunk h + 1
    slot[1024] = hi;  // chunk h: the high half of a bitstream word is its first chunk
  };
#ifndef MPS_SLAB_ALIGN
#define MPS_SLAB_ALIGN 1
#endif
#ifndef MPS_SLAB_RESERVE_BLOCKS
#define MPS_SLAB_RESERVE_BLOCKS 4
#endif
  constexpr int RB = MPS_SLAB_RESERVE_BLOCKS;  // 16-byte blocks per bitstream request
  // Byte address of the bucket's bitstream modulo one request (16 * RB bytes):
  // requests after the first start on that boundary, so each one touches a
  // single cache-line half (RB = 4) or line (RB = 8).
  const uint32_t line_phase = (uint32_t)reinterpret_cast<uintptr_t>(T.bitstream) + (uint32_t)(bucket_bit >> 3);
  const uint32_t phase = line_phase & (16u * RB - 1u);
  // The initial queue (written below): the four words read during set-up, or
  // three when the fourth would leave the next request off a 16-byte boundary.
  const uint32_t rq0 = ((pos >> 5) & ~1u) + 2u;
  const uint32_t nfirst = (MPS_SLAB_ALIGN && ((phase + 4u * (rq0 - 2u)) & 15u)) ? 6u : 8u;
  uint32_t wqb = (rq0 + nfirst) << 5;  // 32 x (first chunk not yet written)
  uint32_t rqb = wqb;                  // 32 x (first chunk not yet requested)
  uint32_t np = 0u - (pos + 64u);      // negated biased position

  // 32 stream bits at -npv; from memory for lanes whose queue lacks the two
  // chunks. (Checking once per four groups instead, with an unchecked copy of
  // the groups, measured slower: the extra branch splits the scheduling region.)
  auto window = [&](uint32_t npv) -> uint32_t {
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

  // Register reserve: up to RB 16-byte blocks that follow the queue's last
  // chunk. Every eighth group (MPS_SLAB_REQ_EVERY below), a lane whose reserve
  // is down to one block requests the next RB * 16 bytes (loads from the same
  // lines, so a 128-byte line is fetched about twice instead of once per 16
  // bytes); they land in the reserve four or more groups later, once it is
  // empty. Every fourth group the reserve's front block moves into the queue
  // if four slots are free.
  uint4 rv[RB], inb[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) rv[i] = inb[i] = make_uint4(0u, 0u, 0u, 0u);
  uint32_t rcnt = 0;  // blocks in rv
  bool ifl = false;   // a request is in flight (into inb)
  auto feed = [&]() {
    const bool f = rcnt != 0u && (int32_t)(wqb + np) < 128;
    if (f) {
      const uint32_t h = wqb >> 5;
      put_pair(h, rv[0].y, rv[0].x);
      put_pair(h + 2u, rv[0].w, rv[0].z);
#pragma unroll
      for (int i = 0; i + 1 < RB; ++i) rv[i] = rv[i + 1];
    }
    wqb += f ? 128u : 0u;
    rcnt -= f ? 1u : 0u;
  };
  uint32_t ninb = 0;  // blocks of the request in flight
#ifndef MPS_SLAB_REQ_EVERY
#define MPS_SLAB_REQ_EVERY 2
#endif
#ifndef MPS_SLAB_REQ_AT
#define MPS_SLAB_REQ_AT 1
#endif
  // Requests are considered every MPS_SLAB_REQ_EVERY-th bitstream step, by
  // lanes whose reserve is down to MPS_SLAB_REQ_AT blocks; landing and feeding
  // run every step. Lanes reach the request point on different steps, so a
  // request's four loads carry few active lanes; asking every other step
  // gathers about twice as many into each load and halves their number.
  static_assert(MPS_SLAB_REQ_EVERY >= 1 && (MPS_SLAB_REQ_EVERY & (MPS_SLAB_REQ_EVERY - 1)) == 0,
                "a power of two");
  uint32_t bstep = 0;  // bitstream steps taken (uniform)
  auto land = [&]() {
    const bool l = ifl && rcnt == 0u;
    if (l) {
#pragma unroll
      for (int i = 0; i < RB; ++i) rv[i] = inb[i];
    }
    rcnt = l ? ninb : rcnt;
    ifl = ifl && !l;
  };
  auto reserve = [&]() {
    const uint32_t off = (rqb >> 3) - 8u;
    // no requests past the substream's end (biased end + the window's reach)
    const bool req = !ifl && rcnt <= (uint32_t)MPS_SLAB_REQ_AT && (int32_t)(rqb - (pos_end + 192u)) < 0;
    // blocks up to the next request boundary (the first request may be short)
    const uint32_t nreq = MPS_SLAB_ALIGN ? (16u * RB - ((phase + off) & (16u * RB - 1u))) >> 4 : (uint32_t)RB;
    if (req) {
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r_bs, (uint32_t)i < nreq ? off + 16u * (uint32_t)i : kBsPast,
                                                             0, MPS_SLAB_BS_CPOL);
        inb[i] = make_uint4(v[0], v[1], v[2], v[3]);
      }
      ninb = nreq;
    }
    ifl = ifl || req;
    rqb += req ? nreq << 7 : 0u;
  };
  // Once per four groups: one 16-byte feed covers the 4 x 28 bits they can consume.
  auto bitstream_step = [&]() {
    land();
    if ((bstep & (MPS_SLAB_REQ_EVERY - 1)) == 0u) reserve();
    bstep = uni(bstep + 1u);
    feed();
  };

  // --- group walker ----------------------------------------------------------
  auto row_offset = [&](uint32_t r) -> uint32_t {
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)rowoff_lo, (int)(r & 63u));
    const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)rowoff_hi, (int)(r & 63u));
    return r < 64u ? a : b;
  };
  uint32_t w_g = 0, w_row = 0, w_blk = 0;
  uint32_t w_off = row_offset(0);
  uint32_t w_next = row_offset(rows > 1u ? 1u : 0u);  // offset of row w_row + 1 (kWrap)
  const uint32_t vf_al = (R << kshift) + colw;       // lane's FP8 byte offset within an aligned group
  // FP8 load of the walker's group; returns the group's BF16 store offset
  // (aligned: the uniform element offset of slab 4g; kWrap: the lane's byte offset).
  auto load_group = [&](uint32_t &F) -> uint32_t {
    uint32_t ret;
    if constexpr (!kWrap) {
      const uint32_t so = uni(w_off + (w_blk << kshift));
      F = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, vf_al, so, MPS_SLAB_FP8_CPOL);
      ret = so;
    } else if constexpr (kWrap == 1) {
      const uint32_t b = w_blk + R;
      const bool wrap = b >= P;
      const bool ok = !wrap || w_row + 1u < rows;
      const uint32_t off = (wrap ? w_next : w_off) + ((wrap ? b - P : b) << kshift) + colw;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, ok ? off : 0u, 0, MPS_SLAB_FP8_CPOL);
      ret = ok ? off << 1 : kSlabPast;
    } else {
      // P < 4: lane R's slab 4g + R is row w_row + d, block b - d P, where
      // b = w_blk + R < 6 and d = b / P < 4. Slabs past the bucket's last row
      // (a partial last group) load in bounds and store out of range.
      const uint32_t b = w_blk + R;
      const uint32_t d = P == 1u ? b : P == 2u ? (b >> 1) : (b >= 3u ? 1u : 0u);
      const uint32_t o0 = row_offset(w_row), o1 = row_offset(w_row + 1u);
      const uint32_t o2 = row_offset(w_row + 2u), o3 = row_offset(w_row + 3u);
      const bool ok = w_row + d < rows;
      const uint32_t off = (d == 0u ? o0 : d == 1u ? o1 : d == 2u ? o2 : o3) + ((b - d * P) << kshift) + colw;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, ok ? off : 0u, 0, MPS_SLAB_FP8_CPOL);
      ret = ok ? off << 1 : kSlabPast;
    }
    // advance (branch-free; past the last group the walk stays on it)
    const bool more = w_g + 1u < gall;
    const uint32_t nb = w_blk + 4u;
    if constexpr (kWrap == 2) {
      // four slabs on: P = 1 and 2 move whole rows, P = 3 one or two rows
      const uint32_t dr = P == 1u ? 4u : P == 2u ? 2u : (nb >= 6u ? 2u : 1u);
      w_blk = uni(more ? nb - dr * P : w_blk);
      w_row = uni(w_row + (more ? dr : 0u));
      w_g = uni(w_g + (more ? 1u : 0u));
      return ret;
    }
    const bool wr = nb >= P;
    const uint32_t nrow = w_row + ((more && wr) ? 1u : 0u);
    const uint32_t noff = row_offset(nrow);
    const uint32_t nnext = row_offset(nrow + 1u < rows ? nrow + 1u : nrow);
    // uni(): selects of uniform values may be computed on the VALU, which would
    // pull the walk (and the loads' soffset) into vector registers.
    w_blk = uni(more ? (wr ? nb - P : nb) : w_blk);
    w_off = uni(nrow != w_row ? noff : w_off);
    w_next = uni(nrow != w_row ? nnext : w_next);
    w_row = uni(nrow);
    w_g = uni(w_g + (more ? 1u : 0u));
    return ret;
  };

  // Flat: the lane's four elements of the walker's group, then 4k elements on.
  // (The values are the walker's where kWrap < 3, whose lanes share one.)
  uint32_t f_at = 0, f_row = 0, f_col = 0;  // element within the item; row and column
  const uint32_t f_dr = kFlat ? uni((4u << kshift) / P) : 0u, f_dc = kFlat ? uni((4u << kshift) - f_dr * P) : 0u;
  const bool f_hi = kFlat && uni((fcol + rows + P - 1u) / P) > 64u;
  if constexpr (kFlat) {
    f_at = (R << kshift) + colw;
    const uint32_t x = fcol + f_at;
    f_row = x / P;
    f_col = x - f_row * P;
  }
  auto lane_row_offset = [&](uint32_t r) -> uint32_t {  // every lane of the wave takes part
    uint32_t o = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(r << 2), (int)rowoff_lo);
    if (f_hi) {
      const uint32_t h = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(r << 2), (int)rowoff_hi);
      o = r < 64u ? o : h;
    }
    return o;
  };
  // Loads the group's bytes into F (and F2); returns the store's byte offset.
  // sh (kWrap 4): 4 - the elements of the lane that lie in its row.
  auto load_flat = [&](uint32_t &F, uint32_t &F2, uint32_t &sh) -> uint32_t {
    const bool ok = f_at < rows;
    const uint32_t off = lane_row_offset(f_row) + f_col;
    uint32_t so = ok ? off << 1 : kSlabPast;
    if constexpr (kWrap == 3) {
      F = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, ok ? off : kSlabPast, 0, MPS_SLAB_FP8_CPOL);
    } else {
      const uint32_t left = P - f_col;  // columns to the row's end
      sh = ok && left < 4u ? 4u - left : 0u;
      const bool more = sh != 0u && f_at + left < rows;
      const uint32_t next = __builtin_amdgcn_ballot_w64(more) ? lane_row_offset(f_row + 1u) : 0u;
      F = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, ok ? off - sh : kSlabPast, 0, MPS_SLAB_FP8_CPOL);
      F2 = __builtin_amdgcn_raw_buffer_load_b32(r_fp8, more ? next : kSlabPast, 0, MPS_SLAB_FP8_CPOL);
      so = sh ? kSlabPast : so;
    }
    f_at += 4u << kshift;
    f_row += f_dr;
    f_col += f_dc;
    const bool carry = f_col >= P;
    f_row += carry ? 1u : 0u;
    f_col -= carry ? P : 0u;
    return so;
  };

  // --- one group ---------------------------------------------------------------
  // sh, gi (kWrap 4): the group's sh as load_flat gave it, and its number.
  auto group = [&](auto is_tail, uint32_t F, uint32_t so, uint32_t sh = 0, uint32_t gi = 0) {
    constexpr bool kTail = decltype(is_tail)::value;
    const auto p1 = __builtin_amdgcn_permlane32_swap(F, F, false, false);
    const uint32_t gq = __builtin_amdgcn_perm(p1[1], p1[0], selA);
    const auto p2 = __builtin_amdgcn_permlane16_swap(gq, gq, false, false);
    const uint32_t fq = __builtin_amdgcn_perm(p2[1], p2[0], selB);  // byte j = element j's FP8 byte
    const uint32_t np0 = np;
    const uint32_t win = window(np);
    uint32_t e[4];
    uint32_t s = 23u;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (kFlat || !kTail || (uint32_t)j < tail) {
        const uint32_t qb = (fq >> (8 * j)) & 0xFFu;
        const uint32_t q9 = qb << 9;
        const uint32_t x = __builtin_amdgcn_alignbit(win, win, s);
        e[j] = *reinterpret_cast<const uint32_t *>(lbytes + ((x & 0x1FCu) ^ q9));
        if (kFlat && kTail) e[j] = (uint32_t)j < tail ? e[j] : 0u;  // by lane
        s -= e[j];
      } else {
        e[j] = 0u;
      }
    }
    np += (uint32_t)((int32_t)(s << 16) >> 16) - 23u;  // minus the bits consumed
    if constexpr (kEsc) {
      // The first ESC code of the group is read from the right place, so its
      // flag is seen even when the window does not reach the codes after it.
      const bool esc = ((e[0] | e[1] | e[2] | e[3]) & kEscBit) != 0u;
      if (__builtin_amdgcn_ballot_w64(esc)) {
        if (esc) {
          uint32_t p = np0;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (!kTail || (uint32_t)j < tail) {
              const uint32_t qb = (fq >> (8 * j)) & 0xFFu;
              const uint32_t q9 = qb << 9;
              const uint32_t w = window(p);
              uint32_t ent = *reinterpret_cast<const uint32_t *>(lbytes + (((w >> 23) & 0x1FCu) ^ q9));
              p -= ent & 7u;
              if (ent & kEscBit) {
                ent = window(p) & 0xFFFF0000u;  // the symbol: the 16 raw bits after the code
                p -= 16u;
              }
              e[j] = ent;
            }
          }
          np = p;
        }
      }
    }
    const auto t0 = __builtin_amdgcn_permlane32_swap(e[0], e[2], false, false);
    const auto t1 = __builtin_amdgcn_permlane32_swap(e[1], e[3], false, false);
    const uint32_t a = __builtin_amdgcn_perm(t0[1], t0[0], 0x07060302u);
    const uint32_t b = __builtin_amdgcn_perm(t1[1], t1[0], 0x07060302u);
    const auto t2 = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    const v2u o = {__builtin_amdgcn_perm(t2[1], t2[0], 0x05040100u), __builtin_amdgcn_perm(t2[1], t2[0], 0x07060302u)};
    // Non-temporal: the output is written once, and L2 is better spent on the
    // lanes' bitstream lines and the FP8 lines that wave pairs share.
    if constexpr (!kWrap) __builtin_amdgcn_raw_buffer_store_b64(o, r_out, vf_al << 1, uni(so) << 1, MPS_SLAB_OUT_CPOL);
    else __builtin_amdgcn_raw_buffer_store_b64(o, r_out, so, 0, MPS_SLAB_OUT_CPOL);
    if constexpr (kWrap == 4) {
      if (__builtin_amdgcn_ballot_w64(sh != 0u)) {
        const uint32_t f = (((gi << 2) + R) << kshift) + colw, x = fcol + f;
        const uint32_t row = x / P, a = 4u - sh;
        const uint32_t o0 = lane_row_offset(row) + (x - row * P), o1 = lane_row_offset(row + 1u) - a;
#pragma unroll
        for (uint32_t j = 0; j < 4u; ++j) {
          const bool ok = sh != 0u && f + j < rows;
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o[j / 2u] >> (16u * (j & 1u))), r_out,
                                                ok ? ((j < a ? o0 : o1) + j) << 1 : kSlabPast, 0, 0);
        }
      }
    }
  };

  uint32_t Fr[DF], SOr[DF];
  uint32_t F2r[kWrap == 4 ? DF : 1], SHr[kWrap == 4 ? DF : 1];
  // Group u of the ring: its bytes (joined) and offsets, and the load of the group DF ahead.
  auto load_ring = [&](int u) {
    if constexpr (kFlat) SOr[u] = load_flat(Fr[u], F2r[kWrap == 4 ? u : 0], SHr[kWrap == 4 ? u : 0]);
    else SOr[u] = load_group(Fr[u]);
  };
  auto ring_bytes = [&](int u) -> uint32_t {
    if constexpr (kWrap == 4) return __builtin_amdgcn_alignbit(F2r[u], Fr[u], SHr[u] << 3);
    return Fr[u];
  };
#pragma unroll
  for (int u = 0; u < DF; ++u) load_ring(u);
  // The initial queue, written once the first FP8 loads are in flight: the
  // wait for the set-up's bitstream words overlaps them.
#pragma unroll
  for (int i = 0; i < 3; ++i) put_pair(rq0 + 2 * i, first[i].y, first[i].x);
  if (nfirst == 8u) put_pair(rq0 + 6u, first[3].y, first[3].x);
  // Every wave of the workgroup decodes the same number of groups, but the
  // issue arbiter favours the oldest ready wave (waves 4r..4r+3 are the r-th
  // oldest on their SIMDs): left alone, the oldest waves finish first and the
  // bucket ends with a few young waves and little latency hiding. So a wave
  // lowers its priority by one level per quarter of its groups, counted from
  // a head start that grows with its age: older waves yield issue slots to
  // younger ones, and a wave that is ahead to the ones behind.
#ifndef MPS_PRIO_LEAD
#define MPS_PRIO_LEAD 8
#endif
  const uint32_t quarter = uni(nfull / 4u > 0u ? nfull / 4u : 1u);
  const uint32_t lead = (3u - (uni(qlane) >> 8)) * (quarter * MPS_PRIO_LEAD / 16u);  // head start (groups)
  uint32_t prio = 3u - (lead / quarter < 3u ? lead / quarter : 3u);
  uint32_t prio_at = (lead / quarter + 1u) * quarter - lead;  // groups done when the priority next drops
  if (prio == 3u) __builtin_amdgcn_s_setprio(3);
  else if (prio == 2u) __builtin_amdgcn_s_setprio(2);
  else if (prio == 1u) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
  uint32_t g = 0;
  for (; g + (uint32_t)DF <= nfull; g += (uint32_t)DF) {
    if (g >= prio_at) {
      prio_at += quarter;
      --prio;
      if (prio == 2u) __builtin_amdgcn_s_setprio(2);
      else if (prio == 1u) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
    }
#pragma unroll
    for (int u = 0; u < DF; ++u) {
      if (u % 4 == 0) bitstream_step();
      if constexpr (kWrap == 4) {
        const uint32_t F = ring_bytes(u), so = SOr[u], sh = SHr[u];
        load_ring(u);
        group(std::false_type{}, F, so, sh, g + (uint32_t)u);
      } else {
        const uint32_t F = Fr[u], so = SOr[u];
        load_ring(u);  // the group DF ahead
        group(std::false_type{}, F, so);
      }
    }
  }
  __builtin_amdgcn_s_setprio(0);
  // the last (fewer than DF) full groups and the partial one; their FP8 is already loaded
#pragma unroll
  for (int u = 0; u < DF; ++u) {
    if (g + (uint32_t)u < gall) {
      if (u % 4 == 0) bitstream_step();
      if constexpr (kWrap == 4) {
        if (g + (uint32_t)u < nfull) group(std::false_type{}, ring_bytes(u), SOr[u], SHr[u], g + (uint32_t)u);
        else group(std::true_type{}, ring_bytes(u), SOr[u], SHr[u], g + (uint32_t)u);
      } else {
        if (g + (uint32_t)u < nfull) group(std::false_type{}, Fr[u], SOr[u]);
        else group(std::true_type{}, Fr[u], SOr[u]);
      }
    }
  }
  if (0u - np - 64u != pos_end) flag(status, MPS_STATUS_DESYNC);
}

// The work item of bucket b of tensor T (the single-tensor kernel).
__device__ __forceinline__ WorkItem bucket_item(const mps_fp8_tensor &T, int64_t b, bool flat_ok) {
  WorkItem w;
  w.tensor = 0;
  const int32_t ra = T.bucket_row_offsets[b];
  const int32_t rb = T.bucket_row_offsets[b + 1];
  w.c0 = T.bucket_col_start[b];
  w.cl = T.bucket_col_len[b];
  const BucketShape s = bucket_shape(ra, rb, w.c0, w.cl, T, flat_ok);
  w.rows = s.path == kPathFlat ? s.rows * w.cl : s.rows;
  w.k_eff = s.k_eff;
  w.path = s.path;
  w.bit_base = T.bucket_bit_base[b];
  w.table_ids = T.bucket_table + b * 256;
  w.startbits = T.bucket_thread_startbit + b * (T.k + 1);
  w.endbits = w.startbits + 1;
  w.row_idx = T.row_indices + (s.path != kPathBad ? ra : 0);
  return w;
}

// Item trace, in instrumented builds only (python -m mpserve_amd.build --define
// MPS_TRACE_ITEMS=1 --out LIB; mpserve_amd.item_trace reads it). decode_bucket
// then also notes the real-time clock after its set-up's last barrier.
#ifndef MPS_TRACE_ITEMS
#define MPS_TRACE_ITEMS 0
#endif
#if MPS_TRACE_ITEMS
#define MPS_TR_PARAM , uint64_t (&tr)[4]
#define MPS_TR_ARG , tr
#else
#define MPS_TR_PARAM
#define MPS_TR_ARG
#endif

// kQueue: the work item also takes the ticket of the workgroup's next one
// from the launch's work counter (queue[0]), at the start of its set-up, so
// that the atomic's round trip overlaps the set-up's loads; every thread
// gets it in `ticket` (zero without kQueue).
// kSlabK: fast-path buckets with k_eff 256 or 512 take the slab path (else the
// scalar element walk). Only launches whose tensors have such
// k compile it in: the extra slab instances cost the k = 1024 launches 1.5%
// (registers), though their own code is unchanged.
// kFlat: flat items (their paths' registers and code stay out of the kernels of
// launches that have none).
template <bool kQueue, bool kSlabK, bool kFlat>
__device__ __forceinline__ void decode_bucket(const mps_fp8_tensor &T, uint16_t *out, const WorkItem &item,
                                              uint32_t *lds, uint32_t *status, uint32_t *queue,
                                              uint32_t &ticket, int32_t wg_part, int32_t wg_parts,
                                              const WorkItem *__restrict__ followers MPS_TR_PARAM) {
  uint32_t *qregion = lds;
  uint32_t *lut = lds + kQWords;
  int32_t *s_rows = reinterpret_cast<int32_t *>(qregion) + 6 * kBlock;    // queue slot 6 (generic path)
  uint32_t *s_wflag = qregion + 5 * kBlock;                             // queue slot 5: the waves' flag words
  // The work-item id through an opaque move: the per-lane constants of every
  // decode path derive from it, and hoisted out of the bucket loop they would
  // all stay live across the set-up, which then runs out of VGPRs.
  int tid;
  __asm__ volatile("v_mov_b32 %0, %1" : "=v"(tid) : "v"((int)threadIdx.x));

  const int32_t path = item.path & 0xF;
  // A run: this work-item's group of k_eff starts with the run's bucket `r_at`, whose
  // record takes the item's place here (the tables are the same).
  const bool run = kFlat && (item.path & kFlatRun) != 0;
  const uint32_t run_k = kFlat ? (uint32_t)item.k_eff & ((1u << kFlatSlabShift) - 1u) : 0u;
  const uint32_t run_n = run ? (uint32_t)item.path >> 8 : 1u, run_from = (uint32_t)item.k_eff >> kFlatSlabShift;
  uint32_t r_at = run ? uni((uint32_t)tid / run_k) : 0u;
  const bool spare = r_at >= run_n;
  auto own_item = [&]() -> decltype(auto) {
    if constexpr (kFlat) {
      WorkItem x = item;
      if (run && r_at > 0 && !spare) x = followers[run_from + r_at - 1u];
      return x;
    } else {
      return (item);
    }
  };
  decltype(auto) w = own_item();
  const int32_t c0 = w.c0, cl = w.cl, k_eff = kFlat ? (int32_t)run_k : w.k_eff;
  const bool bucket_ok = path != kPathBad;
  const bool k1024 = path == kPathK1024;
  const bool fast = path == kPathFast;
  const bool flat = kFlat && path == kPathFlat;
  // A multi-range item (fast path, k_eff 256 or 512): work-items
  // [sub * k_eff, (sub + 1) * k_eff) decode its sub-th range, whose rows,
  // start bits and end bits follow the previous range's (uniform per wave).
  const bool multi = (item.path & kMultiRange) != 0;
  const int32_t mrr = (w.path >> 8) & 0xFF;
  const int32_t sub = multi ? (int32_t)uni((uint32_t)(tid >> (k_eff == 256 ? 8 : 9))) : 0;
  int32_t rows = multi ? max(0, min(mrr, w.rows - sub * mrr)) : w.rows;
  // A flat item: its (or, side by side, its sub-th range's) elements, the column
  // of the first in its row, and the item's rows before that row.
  uint32_t f_elems = 0, f_col = 0, f_row0 = 0;
  if (flat) {
    const uint32_t step = multi ? ((uint32_t)w.k_eff >> kFlatSlabShift) * (uint32_t)k_eff : 0u;  // elements a range
    const uint32_t at = (uint32_t)sub * step, all = spare ? 0u : (uint32_t)w.rows;
    f_elems = uni(at < all ? (multi ? min(step, all - at) : all) : 0u);
    const uint32_t x = (run ? 0u : (uint32_t)w.path >> 8) + at;
    f_row0 = uni(x / (uint32_t)cl);
    f_col = uni(x - f_row0 * (uint32_t)cl);
    rows = (int32_t)uni((f_col + f_elems + (uint32_t)cl - 1u) / (uint32_t)cl);
    rows = f_elems ? rows : 0;
  }
  const int64_t total = (int64_t)rows * cl;
  const uint64_t nm = (uint64_t)T.n * (uint64_t)T.m;
  // the lane's substream (work-item within its range, or its bucket of a run)
  const int lane = multi || run ? (tid & (k_eff - 1)) : tid;
  // Substream of this work-item: the k = 1024 paths give wave w's 16-lane row
  // R, position v the column 64w + 4v + R (see decode_slab4); the others, the lane.
  // A fast-path bucket with k_eff 256 or 512 takes the slab path too (kSlabK).
  const bool slab = kSlabK && fast && (k_eff == 256 || k_eff == 512);
  const int col = k1024 ? ((tid & ~63) | ((tid & 15) << 2) | ((tid >> 4) & 3))
                  : (slab || flat) ? ((lane & ~63) | ((lane & 15) << 2) | ((lane >> 4) & 3)) : lane;
  const bool active = bucket_ok && rows > 0 && lane < k_eff;
  const uint32_t *sb = w.startbits + (int64_t)sub * k_eff;
  const uint32_t *eb = w.endbits + (int64_t)sub * k_eff;
  const int32_t *row_idx = w.row_idx + (flat ? (int64_t)f_row0 : (int64_t)sub * mrr);
  const uint64_t base = (uint64_t)w.bit_base;

  // Set-up: two levels of loads, each issued in full before any of its
  // results is used. (1) From the work record alone: the table ids, the row
  // indices (fast paths) and the lane's start bits. (2) From those: the
  // tables' contents and the lane's first bitstream words. They are buffer
  // loads, whose lanes out of range read zeros, so that none sits behind a
  // branch: a load under a branch is waited for where the branch joins.
  //
  // Thread tid expands the 16-byte slice tid % 16 of the tables of FP8 bytes
  // tid / 16 + 64 i (i < 4); 16 threads read each id.
  constexpr int kSlices = 256 * (kTable / 8) / kBlock;  // 4
  const bool rows_fast = k1024 || fast || flat;
  const int wl = lane & 63;
  // The ticket: a buffer atomic that only thread 0 addresses in range (the
  // others' are dropped), so no branch holds the set-up's loads behind it.
  uint32_t tk = 0;
  if (kQueue) {
    const __amdgpu_buffer_rsrc_t r_q = make_rsrc(queue, 4u);
    tk = (uint32_t)__builtin_amdgcn_raw_ptr_buffer_atomic_add_i32(1, r_q, tid == 0 ? 0u : kBsPast, 0, 0);
    tk = tid == 0 ? tk : 0u;
  }
  const __amdgpu_buffer_rsrc_t r_ids = make_rsrc(w.table_ids, 256u * 4u);
  const __amdgpu_buffer_rsrc_t r_rows = make_rsrc(row_idx, rows_fast ? (uint32_t)rows * 4u : 0u);
  const __amdgpu_buffer_rsrc_t r_sb = make_rsrc(sb, rows_fast ? (uint32_t)k_eff * 4u : 0u);
  const __amdgpu_buffer_rsrc_t r_eb = make_rsrc(eb, rows_fast ? (uint32_t)k_eff * 4u : 0u);
  int32_t gids[kSlices];
#pragma unroll
  for (int i = 0; i < kSlices; ++i)
    gids[i] = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_ids, (uint32_t)((tid >> 4) + 64 * i) * 4u, 0, 0);
  const int32_t r_lo = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_rows, (uint32_t)wl * 4u, 0, 0);
  const int32_t r_hi = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_rows, (uint32_t)(wl + 64) * 4u, 0, 0);
  const uint32_t sb_off = active ? (uint32_t)col * 4u : kBsPast;
  uint32_t pos = __builtin_amdgcn_raw_buffer_load_b32(r_sb, sb_off, 0, 0);
  uint32_t pos_end = __builtin_amdgcn_raw_buffer_load_b32(r_eb, sb_off, 0, 0);

#if MPS_TRACE_ITEMS
  const uint64_t tr_start = __builtin_amdgcn_s_memrealtime();
  __asm__ volatile("" ::"v"(gids[0]), "v"(gids[3]), "v"(r_lo), "v"(r_hi), "v"(pos), "v"(pos_end));
  const uint64_t tr_l1 = __builtin_amdgcn_s_memrealtime();
#endif
  bool bad_table = false;
#pragma unroll
  for (int i = 0; i < kSlices; ++i) {
    if (gids[i] < -1 || gids[i] >= T.num_tables) {
      bad_table = true;
      gids[i] = -1;
    }
  }
  // Row offsets: the fast paths keep rows 0..63 / 64..127 one per lane in
  // VGPRs (selects, not a branch, so the loads above are not sunk into one).
  const bool has_lo = rows_fast && wl < rows, has_hi = rows_fast && wl + 64 < rows;
  bool bad_row = (has_lo && (r_lo < 0 || r_lo >= T.n)) | (has_hi && (r_hi < 0 || r_hi >= T.n));
  const uint32_t rowoff_lo = has_lo ? (uint32_t)r_lo * (uint32_t)T.m + (uint32_t)c0 : 0u;
  const uint32_t rowoff_hi = has_hi ? (uint32_t)r_hi * (uint32_t)T.m + (uint32_t)c0 : 0u;
  // Offset of the lane's first bitstream words (loaded after the table
  // expansion), computed here: the wait for `pos` then falls before the table
  // loads are issued, not at the join of their two paths.
  uint32_t off0 = active ? ((pos >> 5) & ~1u) * 4u : kBsPast;
  __asm__ volatile("" : "+v"(off0));
  // Likewise the descriptor's bitstream fields (scalar loads).
  const uint8_t *bs_ptr = reinterpret_cast<const uint8_t *>(T.bitstream);
  int64_t bs_words = T.bitstream_words;
  __asm__ volatile("" : "+s"(bs_ptr), "+s"(bs_words));
  // The tables' contents (buffer loads when their byte offsets fit 31 bits).
  uint4 sv[kSlices];
  uint32_t nibs[kSlices];
  const int part = tid & 15;
  const bool vec_ok = ((reinterpret_cast<uintptr_t>(T.decode_syms) & 15u) == 0) &&
                      ((reinterpret_cast<uintptr_t>(T.decode_lens) & 3u) == 0);
  const bool tab_buffer = vec_ok && T.num_tables <= (1 << 22);
  if (tab_buffer) {
    const uint32_t ntab = (uint32_t)T.num_tables;
    const __amdgpu_buffer_rsrc_t r_syms = make_rsrc(T.decode_syms, ntab * (uint32_t)(kTable * 2));
    const __amdgpu_buffer_rsrc_t r_lens = make_rsrc(T.decode_lens, ntab * (uint32_t)kPacked);
#pragma unroll
    for (int i = 0; i < kSlices; ++i) {
      const bool has = gids[i] >= 0;
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(
          r_syms, has ? (uint32_t)gids[i] * (uint32_t)(kTable * 2) + (uint32_t)part * 16u : 0x80000000u, 0, 0);
      sv[i] = make_uint4(v[0], v[1], v[2], v[3]);
      nibs[i] = __builtin_amdgcn_raw_buffer_load_b32(
          r_lens, has ? (uint32_t)gids[i] * (uint32_t)kPacked + (uint32_t)part * 4u : 0x80000000u, 0, 0);
    }
  }
  if (bad_table) flag(status, MPS_STATUS_BAD_TABLE);
  // The two fallbacks below load through global pointers (gload), so that the
  // waits after their join stay partial and the first bitstream words' loads
  // below can still be in flight during the expansion.
  if (!rows_fast) {
    for (int i = tid; i < rows; i += kBlock) {
      const int32_t r = gload(w.row_idx + i);
      bad_row |= r < 0 || r >= T.n;
      s_rows[i] = r;
    }
  }
#pragma unroll
  for (int i = 0; i < kSlices && !tab_buffer; ++i) {
    const int32_t g = gids[i];
    sv[i] = make_uint4(0u, 0u, 0u, 0u);
    nibs[i] = 0;
    if (g >= 0) {
      const uint16_t *sp = T.decode_syms + (int64_t)g * kTable + part * 8;
      const uint8_t *lp = T.decode_lens + (int64_t)g * kPacked + part * 4;
      if (vec_ok) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 v = gload(reinterpret_cast<const u32x4 *>(sp));
        sv[i] = make_uint4(v[0], v[1], v[2], v[3]);
        nibs[i] = gload(reinterpret_cast<const uint32_t *>(lp));
      } else {
        uint32_t h[8], b[4];
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = gload_single(sp + j);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[j] = gload_single(lp + j);
        sv[i] = make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
        nibs[i] = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
      }
    }
  }

#if MPS_TRACE_ITEMS
  __asm__ volatile("" ::"v"(sv[0].x), "v"(sv[3].w), "v"(nibs[0]), "v"(nibs[3]));
  const uint64_t tr_l2 = __builtin_amdgcn_s_memrealtime();
  tr[1] = ((tr_l1 - tr_start) & 0xFFFFFFFFull) | ((tr_l2 - tr_start) << 32);
  if ((tid & 63) == 0) s_wflag[32 + (tid >> 6)] = (uint32_t)(tr_l2 - tr_start);
#endif
  uint32_t esc_seen = 0;
#pragma unroll
  for (int i = 0; i < kSlices; ++i) {
    esc_seen |= nibs[i] & 0x88888888u;
    // Entry j = sym_j << 16 | (nib_j & 7) | (nib_j & 8 ? 16 : 0). The nibbles go
    // to bytes (even entries in `fl`, odd ones in `fh`), where nib + (nib & 8)
    // is the entry's low byte; one byte permute per entry then joins it with
    // the symbol (the high or low half of sv: entries 2c and 2c + 1 share word c).
    const uint32_t lo = nibs[i] & 0x0F0F0F0Fu, hi = (nibs[i] >> 4) & 0x0F0F0F0Fu;
    const uint32_t fl = lo + (lo & 0x08080808u), fh = hi + (hi & 0x08080808u);
    const uint32_t w4[4] = {sv[i].x, sv[i].y, sv[i].z, sv[i].w};
    uint32_t e[8];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      e[2 * c] = __builtin_amdgcn_perm(w4[c], fl, 0x05040C00u | (uint32_t)c);      // [fl byte c, 0, sym lo]
      e[2 * c + 1] = __builtin_amdgcn_perm(w4[c], fh, 0x07060C00u | (uint32_t)c);  // [fh byte c, 0, sym hi]
    }
    const uint32_t qt = (uint32_t)((tid >> 4) + 64 * i);  // the table's FP8 byte
    uint32_t *tab = lut + qt * kTable;
    *reinterpret_cast<uint4 *>(tab + (uint32_t)part * 8u) = make_uint4(e[0], e[1], e[2], e[3]);
    *reinterpret_cast<uint4 *>(tab + (uint32_t)part * 8u + 4u) = make_uint4(e[4], e[5], e[6], e[7]);
  }
#if MPS_TRACE_ITEMS
  const uint64_t tr_exp = __builtin_amdgcn_s_memrealtime();
#endif
  // First four bitstream words of this lane (two 16-byte loads); the slab
  // path queues all four, the others three. A lane's words are scattered (64
  // lines a wave), and the CU's memory path takes its waves' loads in order:
  // issued with the table loads they held back the later waves' tables (and so
  // the barrier below); issued at the decode's start, their round trip added
  // to it. Issued here, once the wave's own tables are in LDS, they overlap
  // the other waves' expansion and the two barriers; the decode waits for them
  // after issuing its first FP8 loads.
  __builtin_amdgcn_sched_barrier(0);
  uint2 first[4];
  {
    const uint64_t bs_bytes = bs_words > 0 ? (uint64_t)bs_words * 8u : 0u;
    const uint64_t base_byte = base >> 3;
    const uint32_t win_bytes = rows_fast && base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u;
    const __amdgpu_buffer_rsrc_t r_bs = make_rsrc(bs_ptr + (base_byte < bs_bytes ? base_byte : 0), win_bytes);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(r_bs, off0 + 16u * (uint32_t)i, 0, 0);
      first[2 * i] = make_uint2(v[0], v[1]);
      first[2 * i + 1] = make_uint2(v[2], v[3]);
    }
  }
  // Block-wide ORs of "a row index is out of range" (bit 0) and "a table has an
  // ESC entry" (bit 1): one word per wave; wave 0's also carries the ticket
  // (bits 2..31). Every wave gets its own copy of the 16 words, in its own
  // queue columns: wave w's lane i writes the word to column 64 i + w, and wave
  // i reads columns 64 i .. 64 i + 15. Only wave i writes those columns later
  // (its queue), after reading them, so no second barrier has to keep a fast
  // wave's queue from overwriting words a slower wave has not read yet.
  {
    const uint32_t wf = (__builtin_amdgcn_ballot_w64(bad_row) ? 1u : 0u) |
                        (__builtin_amdgcn_ballot_w64(esc_seen != 0) ? 2u : 0u) | (uni(tk) << 2);
    if ((tid & 63) < kBlock / 64) s_wflag[((tid & 63) << 6) | (tid >> 6)] = wf;
  }
  __syncthreads();
#if MPS_TRACE_ITEMS
  const uint64_t tr_b1 = __builtin_amdgcn_s_memrealtime();
  uint32_t tr_l2max = 0;
  for (int w = 0; w < kBlock / 64; ++w) tr_l2max = max(tr_l2max, s_wflag[32 + w]);
  tr[2] = ((tr_exp - tr_start) & 0xFFFFFFFFull) | ((tr_b1 - tr_start) << 32);
  tr[3] = tr_l2max;
#endif
  uint32_t bflags = 0;
  {
    const uint32_t *mine = s_wflag + (uni((uint32_t)tid) & ~63u);  // this wave's copy
#pragma unroll
    for (int w = 0; w < kBlock / 64; w += 4) {
      const uint4 f = *reinterpret_cast<const uint4 *>(mine + w);
      bflags |= f.x | f.y | f.z | f.w;
    }
  }
  bflags = uni(bflags);
  ticket = bflags >> 2;
  const bool has_esc = (bflags & 2u) != 0;
  const bool any_bad_row = (bflags & 1u) != 0;
#if MPS_TRACE_ITEMS
  tr[0] = __builtin_amdgcn_s_memrealtime();
#endif

  // (In a run, a bad row skips its bucket only: below, wave by wave.)
  if (!bucket_ok || (any_bad_row && !run)) {
    if (tid == 0) flag(status, !bucket_ok ? MPS_STATUS_BAD_BUCKET : MPS_STATUS_BAD_ROW);
    return;
  }
  if (!active) return;
  // A bucket shared by `wg_parts` workgroups (the single-tensor kernel, few
  // buckets for the CUs): every one expands the tables; on the k = 1024 paths
  // workgroup `wg_part` then decodes the substreams of waves
  // [16 wg_part / wg_parts, 16 (wg_part + 1) / wg_parts), on the others part 0 decodes all.
  if (wg_parts > 1) {
    const int32_t wv = (int32_t)(uni((uint32_t)tid) >> 6);
    if (k1024 || (flat && k_eff == kBlock) ? (wv * wg_parts / (kBlock / 64) != wg_part) : (wg_part != 0)) return;
  }
  if (k1024) {
    const uint32_t P = (uint32_t)cl / 1024u;
    if (P >= 4) {
#define MPS_SLAB(WRAP, ESC)                                                                               \
  decode_slab4<WRAP, ESC, 10>(T, out, lut, qregion, (uint32_t)lane, (uint32_t)lane, 10u, (uint32_t)rows, P, \
                              rowoff_lo, rowoff_hi, base, first, pos, pos_end, status)
      if (P % 4 == 0) {
        if (has_esc) MPS_SLAB(0, true);
        else MPS_SLAB(0, false);
      } else {
        if (has_esc) MPS_SLAB(1, true);
        else MPS_SLAB(1, false);
      }
      return;
    }
    // P < 4: the same path, with groups that span two to four rows
    if (has_esc) MPS_SLAB(2, true);
    else MPS_SLAB(2, false);
#undef MPS_SLAB
  } else if (kFlat && flat) {
    const uint32_t ks = k_eff == 1024 ? 10u : k_eff == 512 ? 9u : 8u;
    uint32_t cl_at = (uint32_t)cl, lo_at = rowoff_lo, hi_at = rowoff_hi;
    uint64_t base_at = base;
    bool bad = run && __builtin_amdgcn_ballot_w64(bad_row) != 0;
    if (bad && wl == 0) flag(status, MPS_STATUS_BAD_ROW);
    for (;;) {
#define MPS_FLAT(WRAP, ESC)                                                                                          \
  decode_slab4<WRAP, ESC, 0>(T, out, lut, qregion, (uint32_t)tid, (uint32_t)lane, ks, f_elems, cl_at, lo_at, hi_at,   \
                             base_at, first, pos, pos_end, status, f_col)
      if (bad) {
      } else if (cl_at % 4u == 0u) {
        if (has_esc) MPS_FLAT(3, true);
        else MPS_FLAT(3, false);
      } else {
        if (has_esc) MPS_FLAT(4, true);
        else MPS_FLAT(4, false);
      }
#undef MPS_FLAT
      if (!run) return;
      // The run's next bucket of this group, wave by wave: a lane's queue column is
      // its own and the tables stay, so nothing here meets the other waves.
      do {
        r_at += (uint32_t)kBlock >> ks;
        if (r_at >= run_n) return;
        const WorkItem x = followers[run_from + r_at - 1u];
        cl_at = (uint32_t)x.cl;
        f_elems = (uint32_t)x.rows;
        base_at = (uint64_t)x.bit_base;
        const uint32_t nr = f_elems / cl_at;  // whole rows
        const __amdgpu_buffer_rsrc_t r_rw = make_rsrc(x.row_idx, nr * 4u);
        const int32_t lo = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_rw, (uint32_t)wl * 4u, 0, 0);
        const int32_t hi = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(r_rw, (uint32_t)(wl + 64) * 4u, 0, 0);
        const __amdgpu_buffer_rsrc_t r_bits = make_rsrc(x.startbits, ((uint32_t)k_eff + 1u) * 4u);
        pos = __builtin_amdgcn_raw_buffer_load_b32(r_bits, (uint32_t)col * 4u, 0, 0);
        pos_end = __builtin_amdgcn_raw_buffer_load_b32(r_bits, (uint32_t)col * 4u + 4u, 0, 0);
        const uint64_t bs_bytes = bs_words > 0 ? (uint64_t)bs_words * 8u : 0u, base_byte = base_at >> 3;
        const __amdgpu_buffer_rsrc_t r_bs =
            make_rsrc(bs_ptr + (base_byte < bs_bytes ? base_byte : 0), base_byte < bs_bytes ? (uint32_t)(bs_bytes - base_byte) : 0u);
        const uint32_t o = ((pos >> 5) & ~1u) * 4u;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto v = __builtin_amdgcn_raw_buffer_load_b128(r_bs, o + 16u * (uint32_t)i, 0, 0);
          first[2 * i] = make_uint2(v[0], v[1]);
          first[2 * i + 1] = make_uint2(v[2], v[3]);
        }
        const bool in_lo = (uint32_t)wl < nr, in_hi = (uint32_t)wl + 64u < nr;
        bad = __builtin_amdgcn_ballot_w64((in_lo && (lo < 0 || lo >= T.n)) || (in_hi && (hi < 0 || hi >= T.n))) != 0;
        lo_at = in_lo ? (uint32_t)lo * (uint32_t)T.m + (uint32_t)x.c0 : 0u;
        hi_at = in_hi ? (uint32_t)hi * (uint32_t)T.m + (uint32_t)x.c0 : 0u;
        if (bad && wl == 0) flag(status, MPS_STATUS_BAD_ROW);
      } while (bad);
    }
  } else if (kSlabK && slab) {
    // k_eff 256 / 512 (col_len % k_eff == 0 on the fast path): work-item tid
    // decodes substream `col` of its range, over slabs of k_eff columns
    const uint32_t ks = k_eff == 512 ? 9u : 8u;
    const uint32_t P = (uint32_t)cl >> ks;
#define MPS_SLABK(WRAP, ESC)                                                                                   \
  decode_slab4<WRAP, ESC, 0>(T, out, lut, qregion, (uint32_t)tid, (uint32_t)lane, ks, (uint32_t)rows, P, rowoff_lo, \
                             rowoff_hi, base, first, pos, pos_end, status)
    if (P % 4 == 0) {
      if (has_esc) MPS_SLABK(0, true);
      else MPS_SLABK(0, false);
    } else if (P > 4) {
      if (has_esc) MPS_SLABK(1, true);
      else MPS_SLABK(1, false);
    } else {
      if (has_esc) MPS_SLABK(2, true);
      else MPS_SLABK(2, false);
    }
#undef MPS_SLABK
  } else if (fast) {
    decode_rows_fast(T, out, lut, qregion, (uint32_t)tid, (uint32_t)lane, (uint32_t)k_eff, (uint32_t)rows,
                     (uint32_t)(cl / k_eff), rowoff_lo, rowoff_hi, base, first, pos, pos_end, status);
  } else {
    const uint64_t pos0 = base + gload(sb + lane);
    const uint64_t pend = base + gload(w.endbits + lane);
    if (nm <= 0xFFFFFFFFull)
      decode_lane<uint32_t>(T, out, lut, s_rows, lane, k_eff, total, c0, cl, pos0, pend, status);
    else
      decode_lane<uint64_t>(T, out, lut, s_rows, lane, k_eff, total, c0, cl, pos0, pend, status);
  }
}

// End of a bucket: drain the wave's memory counters (its last stores and the
// FP8 and bitstream prefetches past its substream's end) before the barrier,
// where the wait overlaps the other waves' last groups. The next set-up then
// starts with nothing outstanding, and none of its loads waits behind these.
__device__ __forceinline__ void end_bucket() {
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();  // the next bucket's set-up overwrites the LDS
}

// Both kernels are persistent: one workgroup per CU (the LDS holds one
// bucket's tables) walks its share of the buckets, so a bucket's set-up does
// not also pay a workgroup launch. fp8_decode_one deals the buckets
// round-robin; every workgroup runs the same uniform loop to its end.
//
// parts > 1 (k = 1024 tensors with fewer buckets than CUs): the grid is
// buckets x parts, and workgroup g decodes part g % parts of bucket g / parts
// (decode_bucket), so that a tensor of 8 buckets runs on 128 CUs instead of 8.
// A bucket's substreams are sequential chains, which only lane checkpoints (a
// plan's) cut into row ranges; fewer waves a CU run each chain faster.
template <bool kSlabK, bool kFlat>
__global__ __launch_bounds__(kBlock) void fp8_decode_one(mps_fp8_tensor T, uint32_t *status, int32_t parts) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[kLdsWords];
  uint32_t ticket;
#if MPS_TRACE_ITEMS
  uint64_t tr[4];
#endif
  if (parts > 1) {
    const int64_t b = (int64_t)blockIdx.x / parts;
    if (b < T.num_buckets)
      decode_bucket<false, kSlabK, kFlat>(T, T.out, bucket_item(T, b, kFlat), lds, status, nullptr, ticket,
                                          (int32_t)(blockIdx.x % parts), parts, nullptr MPS_TR_ARG);
    return;
  }
  for (int64_t b = blockIdx.x; b < T.num_buckets; b += gridDim.x) {
    decode_bucket<false, kSlabK, kFlat>(T, T.out, bucket_item(T, b, kFlat), lds, status, nullptr, ticket, 0, 1,
                                        nullptr MPS_TR_ARG);
    end_bucket();
  }
}

// fp8_decode_plan takes its work items from a queue: workgroup g starts with
// item g; each item takes a ticket t from queue[0] (in its set-up, or with
// kEndTicket as it ends), and the workgroup's next item is gridDim.x + t. The items are sorted largest first,
// so the CUs that drew small items or ran fast take more of them, and all
// finish close together (a fixed deal would leave the CUs with the larger
// shares running alone at the end). The last workgroup to leave (queue[1]
// counts them) puts both words back to zero for the next launch: launches of
// one queue must not overlap.
//
// out_delta: elements every tensor's output moves by (a plan decoding into a
// buffer laid out like, but other than, the one it was created with).
//
// Tickets travel in 30 bits of the set-up's flag words: a launch holds fewer
// than kMaxQueueItems work items.
constexpr int64_t kMaxQueueItems = (int64_t(1) << 30) - 65536;

// The item trace (instrumented builds): workgroup g < kTraceWgs records its
// first kTraceItems items, kTraceWords words each: the real-time clock (100 MHz) at the
// item's start and after its end barrier, the item's path << 40 | rows << 20 |
// k_eff, its col_len, the clock after the set-up's last barrier, the clock
// when waves 0 and 15 finished their decode (before the end drain), and wave
// 0's ticks from its set-up start: to its level-1 loads' return (word 7 low
// half), its tables' return (word 7 high half), the end of its table expansion
// (word 8 low half), the set-up's first barrier (word 8 high half) and the
// last wave's tables (word 9). Threads 0 and 960 write them with ordinary
// stores after the barrier; words 10 and 11 are spare. (Each translation unit has its
// own; the host reads fp8_decode.hip's, whose kernels see no flat items.)
#if MPS_TRACE_ITEMS
constexpr int kTraceWgs = 256, kTraceItems = 128, kTraceWords = 12;
__device__ uint64_t g_item_trace[kTraceWgs * kTraceItems * kTraceWords];
#endif

template <bool kSlabK, bool kEndTicket, bool kFlat>
__global__ __launch_bounds__(kBlock) void fp8_decode_plan(const mps_fp8_tensor *__restrict__ tensors,
                                                          const WorkItem *__restrict__ work, int64_t nwork,
                                                          uint32_t *status, int64_t out_delta, uint32_t *queue) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[kLdsWords];
  if ((int64_t)blockIdx.x < nwork) {
    WorkItem w = work[blockIdx.x];
#if MPS_TRACE_ITEMS
    int tr_it = 0;
#endif
    for (;;) {
      uint32_t ticket;
#if MPS_TRACE_ITEMS
      const uint64_t tr0 = __builtin_amdgcn_s_memrealtime();
      uint64_t tr[4] = {0, 0, 0, 0};
#endif
      const mps_fp8_tensor &T = tensors[w.tensor];
      decode_bucket<!kEndTicket, kSlabK, kFlat>(T, T.out + out_delta, w, lds, status, queue, ticket, 0, 1, work + nwork MPS_TR_ARG);
#if MPS_TRACE_ITEMS
      const uint64_t tr_wave = __builtin_amdgcn_s_memrealtime();
#endif
      if constexpr (kEndTicket) {
        // The ticket is taken once wave 0 is through with the item, so the
        // next item goes to a workgroup that is about to be free; thread 0
        // hands it out through the LDS once every wave is done with the
        // item's queue, and every wave reads it before the next set-up.
        uint32_t tq = 0;
        if (threadIdx.x == 0)
          tq = __hip_atomic_fetch_add((__attribute__((address_space(1))) uint32_t *)(queue), 1u, __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        end_bucket();
        if (threadIdx.x == 0) lds[0] = tq;
        __syncthreads();
        ticket = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds[0]);
        __syncthreads();
      }
      const int64_t next = (int64_t)gridDim.x + ticket;
      // The next record (scalar registers); with the set-up's ticket it is
      // loaded before the drain of this item's stores, which covers its round trip.
      const WorkItem wn = work[next < nwork ? next : 0];
      if constexpr (!kEndTicket) end_bucket();
#if MPS_TRACE_ITEMS
      if (blockIdx.x < kTraceWgs && tr_it < kTraceItems) {
        uint64_t *tp = g_item_trace + ((size_t)blockIdx.x * kTraceItems + tr_it) * kTraceWords;
        if (threadIdx.x == 0) {
          tp[0] = tr0;
          tp[1] = __builtin_amdgcn_s_memrealtime();
          tp[2] = ((uint64_t)(uint32_t)w.path << 40) | ((uint64_t)(uint32_t)w.rows << 20) | (uint64_t)(uint32_t)w.k_eff;
          tp[3] = (uint64_t)(uint32_t)w.cl;
          tp[4] = tr[0];
          tp[5] = tr_wave;
          tp[7] = tr[1];
          tp[8] = tr[2];
          tp[9] = tr[3];
        } else if (threadIdx.x == 960) {
          tp[6] = tr_wave;
        }
      }
      ++tr_it;
#endif
      if (next >= nwork) break;
      w = wn;
    }
  }
  if (threadIdx.x == 0) {
    if (atomicAdd(queue + 1, 1u) == gridDim.x - 1) {
      atomicExch(queue, 0u);
      atomicExch(queue + 1, 0u);
    }
  }
}

}  // namespace
}  // namespace mps
