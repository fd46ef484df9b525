// The sidecar builder's passes over the elements, one *unit* of one bucket a
// workgroup (included by fp8_encode.hip, inside its namespace).
//
// A bucket's elements share one scale, so inside a bucket a (key, symbol) pair
// is 24 bits, and a scale has a few thousand distinct pairs: they fit one LDS
// hash table. A unit is a run of whole steps (k_eff elements, one a substream)
// of one bucket, so the same units serve every pass:
//   unit_hist    counts a unit's pairs in LDS and writes them as a list;
//   merge_lists  adds up the lists of one scale (one q range of it) in LDS and
//                sorts them by (q, count, symbol): the builder's item order;
//   number_keys  table ids of the keys, in (scale, q) order;
//   (the codebooks, from the sorted entries, fp8_encode.hip)
//   unit_codes   maps a unit's elements to code words through an LDS table of
//                the scale's pairs, stores them (16 bits an element, in bucket
//                order) and sums each substream's bits within the unit;
//   bucket_starts   start bits of the substreams and buckets;
//   unit_pack    writes each substream's piece of the unit into the bitstream.
// Every pass has as many workgroups as units, so a tensor of few buckets, or
// of few substreams a bucket, fills the chip too: a piece of a substream
// starts at its substream's start bit plus the bits of its earlier pieces.
//
// Measured against one work-item a substream over a hash table in global
// memory (the general path of fp8_encode.hip, for the calls this one does not
// take), one 14336 x 4096 FP8 weight, k = 1024: counting 1.89 ms -> 69 us,
// grouping and sorting 1.38 ms -> 43 us, code words and bits 1.60 ms -> 92 us,
// packing 0.57 ms -> 85 us.
#pragma once

constexpr int kUnitThreads = 1024;
constexpr uint32_t kPairSlots = 8192;   // LDS slots of a unit's, or a part's, pairs
constexpr uint32_t kUnitRows = 1024;    // a unit spans at most this many rows (groups), + 2 partial ones
constexpr uint32_t kNoPair = 0xFFFFFFFFu;
constexpr uint32_t kMaxProbes = 256;

// The scales' ranks among their sorted distinct values: res[0] the number of
// values, ranks[i] of scale i, values[] ascending. One workgroup over a set of
// 65536 bits in LDS: a few microseconds, where the host took some 80 for its
// tables of 65536 alone (of a 1024 x 4096 weight's 360 us a build). What bounds
// it is the latency of one CU's loads, so they are 16 bytes wide where the array
// is aligned, four in flight: 131,072 scales of a 4096 x 4096 weight 70 -> 20 us.
__global__ __launch_bounds__(kUnitThreads) void scale_ranks(const uint16_t *__restrict__ scales, uint64_t n,
                                                            uint32_t *__restrict__ res, uint16_t *__restrict__ ranks,
                                                            uint16_t *__restrict__ values) {
  constexpr uint32_t kWords = 65536 / 32, kPer = kWords / kUnitThreads, kLoads = 4;
  __shared__ uint32_t s_set[kWords], s_tmp[16];
  __shared__ uint2 s_rank[kWords];  // a word of the set, and the values before it
  const uint32_t tid = threadIdx.x;
  const uint64_t n8 = reinterpret_cast<uintptr_t>(scales) % 16 == 0 ? n / 8 : 0;  // 16-byte loads; the rest one by one
  const uint4 *scales8 = reinterpret_cast<const uint4 *>(scales);
  for (uint32_t i = tid; i < kWords; i += kUnitThreads) s_set[i] = 0u;
  __syncthreads();
  auto mark = [&](uint32_t v) {
    const uint32_t bit = 1u << (v & 31u);
    if (!(s_set[v >> 5] & bit)) atomicOr(&s_set[v >> 5], bit);
  };
  for (uint64_t i = tid; i < n8; i += kLoads * kUnitThreads) {
    uint4 v[kLoads];
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
      const uint64_t at = i + j * kUnitThreads;
      v[j] = scales8[at < n8 ? at : i];
    }
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
      const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (uint32_t h = 0; h < 4u; ++h) {
        mark(w[h] & 0xFFFFu);
        mark(w[h] >> 16);
      }
    }
  }
  for (uint64_t i = 8 * n8 + tid; i < n; i += kUnitThreads) mark(scales[i]);
  __syncthreads();
  uint32_t mine = 0;
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j) mine += (uint32_t)__popc(s_set[tid * kPer + j]);
  uint32_t total = 0, at = block_exclusive_scan(mine, s_tmp, &total);
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j) {
    const uint32_t w = tid * kPer + j;
    uint32_t bits = s_set[w];
    s_rank[w] = make_uint2(bits, at);
    while (bits) {
      values[at++] = (uint16_t)(32u * w + (uint32_t)__builtin_ctz(bits));
      bits &= bits - 1u;
    }
  }
  __syncthreads();
  auto rank = [&](uint32_t v) {
    const uint2 r = s_rank[v >> 5];
    return r.y + (uint32_t)__popc(r.x & ((1u << (v & 31u)) - 1u));
  };
  for (uint64_t i = tid; i < n8; i += kLoads * kUnitThreads) {
    uint4 v[kLoads];
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
      const uint64_t at = i + j * kUnitThreads;
      v[j] = scales8[at < n8 ? at : i];
    }
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
      const uint64_t at = i + j * kUnitThreads;
      uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (uint32_t h = 0; h < 4u; ++h) w[h] = rank(w[h] & 0xFFFFu) | (rank(w[h] >> 16) << 16);
      if (at < n8) reinterpret_cast<uint4 *>(ranks)[at] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  for (uint64_t i = 8 * n8 + tid; i < n; i += kUnitThreads) ranks[i] = (uint16_t)rank(scales[i]);
  if (tid == 0) res[0] = total;
}

// A bucket's rows (groups, by scale) are those of one scale, in order: a stable
// counting sort of the scales by rank, for up to kSortRanks distinct ones. A
// tile's ranks are counted in LDS (rank_hist, hist[tile][rank]); rank_sort adds
// up the counts before its tile's, gives each wave a run of the tile and places
// an item after the run's earlier ones of its rank: lanes of equal rank find
// each other by a ballot a rank bit.
// Bound by latency, a few loads and LDS steps a work-item (a tile is 2048 items
// while that gives no more than 256): 131,072 groups of a 4096 x 4096 AWQ weight
// 4 + 11 us, where the host's loop and the copies of its result took 0.22 ms of
// the build's 0.72; 917,504 groups of a 4096 x 14336 one 1.7 of 2.6 ms.
constexpr uint32_t kSortRanks = 4096;
__global__ __launch_bounds__(kUnitThreads) void rank_hist(const uint16_t *__restrict__ ranks, uint32_t n, uint32_t tile,
                                                          const uint32_t *__restrict__ res, uint32_t *__restrict__ hist) {
  __shared__ uint32_t s_n[kSortRanks];
  const uint32_t tid = threadIdx.x, S = res[0], S4 = (S + 3u) & ~3u;
  if (S > kSortRanks) return;
  for (uint32_t r = tid; r < S4; r += kUnitThreads) s_n[r] = 0u;
  __syncthreads();
  const uint32_t i0 = blockIdx.x * tile, i1 = i0 + tile < n ? i0 + tile : n;
  for (uint32_t i = i0 + tid; i < i1; i += kUnitThreads) atomicAdd(&s_n[ranks[i]], 1u);
  __syncthreads();
  for (uint32_t r = tid; r < S4; r += kUnitThreads) hist[(uint64_t)blockIdx.x * kSortRanks + r] = s_n[r];
}

// counts[]: items of each rank. An item is (row, column range) i / per_row and (i % per_row) * width.
__global__ __launch_bounds__(kUnitThreads) void rank_sort(const uint16_t *__restrict__ ranks, uint32_t n, uint32_t tile,
                                                          const uint32_t *__restrict__ res,
                                                          const uint32_t *__restrict__ hist,
                                                          uint32_t *__restrict__ counts, uint32_t per_row, uint32_t width,
                                                          int32_t *__restrict__ rows, int32_t *__restrict__ cols) {
  constexpr uint32_t kWaves = kUnitThreads / 64;
  __shared__ uint32_t s_base[kSortRanks], s_tmp[16];
  __shared__ uint32_t s_wave[kWaves][kSortRanks / 2];  // 16 bits a rank: a tile has fewer than 2^16 items
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, S = res[0];
  if (S > kSortRanks) return;
  uint4 all = make_uint4(0, 0, 0, 0), before = all;
  if (4u * tid < S) {
    const uint4 *h4 = reinterpret_cast<const uint4 *>(hist) + tid;
#pragma unroll 8
    for (uint32_t t = 0; t < gridDim.x; ++t) {
      const uint4 h = h4[(uint64_t)t * (kSortRanks / 4u)];
      const uint32_t mine = t < blockIdx.x ? ~0u : 0u;
      all = make_uint4(all.x + h.x, all.y + h.y, all.z + h.z, all.w + h.w);
      before = make_uint4(before.x + (h.x & mine), before.y + (h.y & mine), before.z + (h.z & mine),
                          before.w + (h.w & mine));
    }
    if (blockIdx.x == 0) reinterpret_cast<uint4 *>(counts)[tid] = all;
  }
  uint32_t total = 0;
  const uint32_t at = block_exclusive_scan(all.x + all.y + all.z + all.w, s_tmp, &total);
  if (4u * tid < S) {
    s_base[4u * tid] = at + before.x;
    s_base[4u * tid + 1u] = at + all.x + before.y;
    s_base[4u * tid + 2u] = at + all.x + all.y + before.z;
    s_base[4u * tid + 3u] = at + all.x + all.y + all.z + before.w;
  }
  uint16_t *mine = reinterpret_cast<uint16_t *>(s_wave[wave]);
  for (uint32_t r = lane; r < (S + 1u) / 2u; r += 64u) s_wave[wave][r] = 0u;
  const int bits = S > 1u ? 32 - __builtin_clz(S - 1u) : 0;
  const uint64_t below = lane == 0u ? 0ull : (~0ull >> (64u - lane));
  auto lds_sync = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  auto same = [&](uint32_t r, bool in) {  // the lanes that hold rank r
    uint64_t m = __ballot(in);
    for (int b = 0; b < bits; ++b) {
      const bool one = (r >> b) & 1u;
      const uint64_t v = __ballot(one);
      m &= one ? v : ~v;
    }
    return m;
  };
  const uint32_t run = tile / kWaves, i0 = blockIdx.x * tile + wave * run;
  lds_sync();
  for (uint32_t c = 0; c < run; c += 64u) {
    const uint32_t i = i0 + c + lane;
    const bool in = i < n;
    const uint32_t r = in ? ranks[i] : 0u;
    const uint64_t m = same(r, in);
    if (in && !(m & below)) mine[r] += (uint16_t)__popcll(m);
    lds_sync();
  }
  __syncthreads();
  for (uint32_t r = tid; r < S; r += kUnitThreads) {
    uint32_t o = 0;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
      uint16_t *p = reinterpret_cast<uint16_t *>(s_wave[w]) + r;
      const uint32_t c = *p;
      *p = (uint16_t)o;
      o += c;
    }
  }
  __syncthreads();
  for (uint32_t c = 0; c < run; c += 64u) {
    const uint32_t i = i0 + c + lane;
    const bool in = i < n;
    const uint32_t r = in ? ranks[i] : 0u;
    const uint64_t m = same(r, in);
    if (in) {
      const uint32_t to = s_base[r] + mine[r] + (uint32_t)__popcll(m & below);
      const uint32_t row = i / per_row;
      rows[to] = (int32_t)row;
      if (cols) cols[to] = (int32_t)((i - row * per_row) * width);
    }
    lds_sync();
    if (in && !(m & below)) mine[r] += (uint16_t)__popcll(m);
    lds_sync();
  }
}

struct Unit {
  uint32_t bucket;
  uint32_t i0, i1;  // steps: elements [i0 * k_eff, min(i1 * k_eff, total)) of the bucket
  uint32_t sidx;    // the bucket's scale
};

struct UnitArgs {
  const Unit *units;
  const uint16_t *bf16;
  const uint8_t *q;
  uint32_t m;
  uint32_t qmask;
  const int32_t *row_offsets;
  const int32_t *row_indices;
  const int32_t *col_start;  // by bucket (null with row_col)
  const int32_t *col_len;
  const int32_t *row_col;    // by row: column start of each group (by-scale layout), or null
  uint32_t k;
  int32_t vec8;  // 8 elements of a row can be loaded at once (widths, starts and pointers are multiples)
};

struct UnitGeom {
  uint32_t cl, k_eff, total;  // the bucket
  uint32_t e0, e1, r0;        // the unit's elements and its first row
};

// Where a pair's probes start: the symbol's sign and low bits. The symbols of
// one scale span some 20 of the 32 octaves these bits tell apart, so pairs of
// different symbols start at different slots; a symbol's second q value (at a
// rounding boundary) steps away.
template <uint32_t kSlots>
__device__ __forceinline__ uint32_t pair_slot(uint32_t pair) {
  static_assert(kSlots == 8192 || kSlots == 16384, "sign + 12 or 13 low bits");
  return kSlots == 8192 ? (pair & 0xFFFu) | ((pair >> 3) & 0x1000u) : (pair & 0x1FFFu) | ((pair >> 2) & 0x2000u);
}
__device__ __forceinline__ uint32_t pair_step(uint32_t pair) { return ((pair >> 16) * 0x2F2u + 0x4D7u) | 1u; }

// Elements of bucket `b` are counted in 32 bits: a tensor has fewer than 2^32.
// Stages the unit's row offsets (first element of each row's column range) in LDS.
__device__ __forceinline__ UnitGeom unit_geom(const UnitArgs &a, const Unit &u, uint32_t *s_base) {
  UnitGeom g;
  const int32_t ra = a.row_offsets[u.bucket];
  const uint32_t rows = (uint32_t)(a.row_offsets[u.bucket + 1] - ra);
  g.cl = (uint32_t)a.col_len[u.bucket];
  g.total = rows * g.cl;
  g.k_eff = a.k < g.total ? a.k : (g.total > 0 ? g.total : 1u);
  g.e0 = u.i0 * g.k_eff;
  const uint64_t end = (uint64_t)u.i1 * g.k_eff;
  g.e1 = end < g.total ? (uint32_t)end : g.total;
  g.r0 = g.e0 / g.cl;
  const uint32_t nrows = g.e1 > g.e0 ? (g.e1 - 1u) / g.cl - g.r0 + 1u : 0u;
  const uint32_t c0 = a.row_col ? 0u : (uint32_t)a.col_start[u.bucket];
  for (uint32_t r = threadIdx.x; r < nrows; r += kUnitThreads) {
    const int32_t at = ra + (int32_t)(g.r0 + r);
    s_base[r] = (uint32_t)a.row_indices[at] * a.m + (a.row_col ? (uint32_t)a.row_col[at] : c0);
  }
  return g;
}

// Adds `add` to a pair's count; false when no slot was found.
__device__ __forceinline__ bool pair_add(uint32_t *s_key, uint32_t *s_cnt, uint32_t pair, uint32_t add) {
  uint32_t h = pair_slot<kPairSlots>(pair);
  for (uint32_t i = 0; i < kMaxProbes; ++i) {
    uint32_t cur = s_key[h];
    if (cur == kNoPair) {
      cur = atomicCAS(&s_key[h], kNoPair, pair);
      if (cur == kNoPair) cur = pair;
    }
    if (cur == pair) {
      atomicAdd(&s_cnt[h], add);
      return true;
    }
    h = (h + pair_step(pair)) & (kPairSlots - 1u);
  }
  return false;
}

// One unit's pairs and counts -> lists[list_off[u] ..] (list_n[u] of them, any
// order). Bound by the LDS: a read and an add an element, at random banks.
__global__ __launch_bounds__(kUnitThreads) void unit_hist(UnitArgs a, const uint32_t *__restrict__ list_off,
                                                          uint2 *__restrict__ lists, uint32_t *__restrict__ list_n,
                                                          uint32_t *overflow) {
  __shared__ uint32_t s_key[kPairSlots], s_cnt[kPairSlots], s_base[kUnitRows + 2], s_n;
  const uint32_t tid = threadIdx.x;
  const Unit u = a.units[blockIdx.x];
  const UnitGeom g = unit_geom(a, u, s_base);
  for (uint32_t i = tid; i < kPairSlots; i += kUnitThreads) {
    s_key[i] = kNoPair;
    s_cnt[i] = 0u;
  }
  if (tid == 0) s_n = 0u;
  __syncthreads();
  bool ok = true;
  uint32_t done = g.e0;
  if (a.vec8 && g.e0 % 8u == 0u) {
    done = g.e1 & ~7u;
    for (uint32_t e = g.e0 + 8u * tid; e < done; e += 8u * kUnitThreads) {
      const uint32_t r = e / g.cl;
      const uint32_t idx = s_base[r - g.r0] + (e - r * g.cl);
      const uint4 b = *reinterpret_cast<const uint4 *>(a.bf16 + idx);
      const uint2 q = *reinterpret_cast<const uint2 *>(a.q + idx);
      const uint32_t bw[4] = {b.x, b.y, b.z, b.w}, qw[2] = {q.x, q.y};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t sym = (bw[j / 2] >> (16 * (j & 1))) & 0xFFFFu;
        const uint32_t qv = (qw[j / 4] >> (8 * (j & 3))) & a.qmask;
        ok &= pair_add(s_key, s_cnt, (qv << 16) | sym, 1u);
      }
    }
    if (done < g.e0) done = g.e0;
  }
  for (uint32_t e = done + tid; e < g.e1; e += kUnitThreads) {
    const uint32_t r = e / g.cl;
    const uint32_t idx = s_base[r - g.r0] + (e - r * g.cl);
    ok &= pair_add(s_key, s_cnt, ((uint32_t)(a.q[idx] & a.qmask) << 16) | a.bf16[idx], 1u);
  }
  if (!ok) atomicOr(overflow, 1u);
  __syncthreads();
  uint2 *out = lists + list_off[blockIdx.x];
  const int lane = (int)(tid & 63u);
  for (uint32_t i = tid; i < kPairSlots; i += kUnitThreads) {
    const uint32_t key = s_key[i];
    const uint64_t live = __ballot(key != kNoPair);
    uint32_t base = 0;
    if (lane == 0 && live) base = atomicAdd(&s_n, (uint32_t)__popcll(live));
    base = (uint32_t)__shfl((int)base, 0);
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (key != kNoPair) out[base + (uint32_t)__popcll(live & below)] = make_uint2(key, s_cnt[i]);
  }
  __syncthreads();
  if (tid == 0) list_n[blockIdx.x] = s_n;
}

// Part p of scale s (blockIdx.x = s * parts + p): the pairs with q in
// [p * qvals / parts, (p + 1) * qvals / parts), added up over the scale's unit
// lists and sorted by (q, count as int, symbol) into skeys[part_off ..]; the
// keys' entry counts and first entries (tcount, toff, indexed s * 256 + q).
// The parts keep the sorts short and the workgroups many when the scales are
// few. Measured on 14336 x 4096: 66 us with a list a wave, a load at a time, and
// a barrier a sorting step; 43 us as below (1024 x 4096: 34 -> 26 us).
__global__ __launch_bounds__(kUnitThreads) void merge_lists(const uint32_t *__restrict__ scale_unit_off,
                                                            const uint32_t *__restrict__ unit_of_scale,
                                                            const uint32_t *__restrict__ list_off,
                                                            const uint32_t *__restrict__ list_n,
                                                            const uint2 *__restrict__ lists, uint32_t parts,
                                                            uint32_t qvals, const uint32_t *__restrict__ part_off,
                                                            uint64_t *__restrict__ skeys, uint32_t *__restrict__ tcount,
                                                            uint32_t *__restrict__ toff, uint32_t *__restrict__ part_n,
                                                            uint32_t *__restrict__ part_keys, uint32_t *overflow) {
  __shared__ __attribute__((aligned(16))) uint32_t s_pairs[2 * kPairSlots];
  __shared__ uint32_t s_len[kUnitThreads], s_off[kUnitThreads], s_n, s_keys;
  uint32_t *s_key = s_pairs, *s_cnt = s_pairs + kPairSlots;
  uint64_t *s_sort = reinterpret_cast<uint64_t *>(s_pairs);
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t s = blockIdx.x / parts, p = blockIdx.x % parts;
  const uint32_t q0 = p * qvals / parts, q1 = (p + 1u) * qvals / parts;
  for (uint32_t i = tid; i < kPairSlots; i += kUnitThreads) {
    s_key[i] = kNoPair;
    s_cnt[i] = 0u;
  }
  if (tid == 0) s_n = s_keys = 0u;
  __syncthreads();
  // The lists in chunks of 512 entries dealt to the waves, eight loads a lane in
  // flight; 1024 lists' lengths at a time in LDS.
  bool ok = true;
  const uint32_t first_list = scale_unit_off[s], num_lists = scale_unit_off[s + 1] - first_list;
  for (uint32_t l0 = 0; l0 < num_lists; l0 += kUnitThreads) {
    const uint32_t nl = num_lists - l0 < kUnitThreads ? num_lists - l0 : kUnitThreads;
    if (l0) __syncthreads();
    if (tid < nl) {
      const uint32_t u = unit_of_scale[first_list + l0 + tid];
      s_len[tid] = list_n[u];
      s_off[tid] = list_off[u];
    }
    __syncthreads();
    uint32_t l = 0, chunk = wave;  // the wave's chunk: chunk `chunk` of list l
    for (;;) {
      uint32_t chunks = 0;
      while (l < nl && chunk >= (chunks = (s_len[l] + 511u) >> 9)) {
        chunk -= chunks;
        ++l;
      }
      if (l >= nl) break;
      const uint2 *from = lists + s_off[l];
      const uint32_t n = s_len[l];
      uint2 e[8];
#pragma unroll
      for (uint32_t j = 0; j < 8u; ++j) {
        const uint32_t at = (chunk << 9) + (j << 6) + lane;
        e[j] = from[at < n ? at : 0u];
        if (at >= n) e[j].x = kNoPair;  // (no q range holds it)
      }
#pragma unroll
      for (uint32_t j = 0; j < 8u; ++j) {
        const uint32_t q = e[j].x >> 16;
        if (q >= q0 && q < q1) ok &= pair_add(s_key, s_cnt, e[j].x, e[j].y);
      }
      chunk += kUnitThreads / 64;
    }
  }
  if (!ok) atomicOr(overflow, 1u);
  __syncthreads();
  // The pairs as sort keys, in place: read into registers, then written back dense.
  constexpr int kPer = kPairSlots / kUnitThreads;
  uint64_t v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint32_t key = s_key[tid + i * kUnitThreads], cnt = s_cnt[tid + i * kUnitThreads];
    v[i] = key == kNoPair ? ~0ull : ((uint64_t)(key >> 16) << 48) | item_key(cnt, key & 0xFFFFu);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const uint64_t live = __ballot(v[i] != ~0ull);
    uint32_t base = 0;
    if (lane == 0 && live) base = atomicAdd(&s_n, (uint32_t)__popcll(live));
    base = (uint32_t)__shfl((int)base, 0);
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64u - lane));
    if (v[i] != ~0ull) s_sort[base + (uint32_t)__popcll(live & below)] = v[i];
  }
  __syncthreads();
  const uint32_t n = s_n;
  uint32_t np = 64;
  while (np < n) np <<= 1;
  for (uint32_t i = n + tid; i < np; i += kUnitThreads) s_sort[i] = ~0ull;
  __syncthreads();
  // Bitonic: the steps of distance below 64 in a wave's registers, 64 entries at
  // a time, the others in LDS with a barrier each.
  auto in_wave = [&](uint32_t size_from, uint32_t size_to) {
    for (uint32_t b = wave * 64u; b < np; b += kUnitThreads) {
      uint64_t x = s_sort[b + lane];
      for (uint32_t size = size_from; size <= size_to; size <<= 1) {
        const bool up = ((b + lane) & size) == 0u;
        for (uint32_t d = size < 64u ? size >> 1 : 32u; d > 0; d >>= 1) {
          const uint64_t y = (uint64_t)__shfl_xor((unsigned long long)x, (int)d);
          const bool low = (lane & d) == 0u;
          if ((y < x) == (low == up)) x = y;  // the low lane keeps the smaller (going up)
        }
      }
      s_sort[b + lane] = x;
    }
    __syncthreads();
  };
  in_wave(2u, 64u);
  for (uint32_t size = 128; size <= np; size <<= 1) {
    for (uint32_t d = size >> 1; d >= 64u; d >>= 1) {
      for (uint32_t i = tid; i < np / 2; i += kUnitThreads) {
        const uint32_t x = ((i & ~(d - 1u)) << 1) | (i & (d - 1u)), y = x + d;
        const uint64_t vx = s_sort[x], vy = s_sort[y];
        if ((vx > vy) == ((x & size) == 0u)) {
          s_sort[x] = vy;
          s_sort[y] = vx;
        }
      }
      __syncthreads();
    }
    in_wave(size, size);
  }
  const uint32_t off = part_off[blockIdx.x];
  for (uint32_t i = tid; i < n; i += kUnitThreads) skeys[off + i] = s_sort[i];
  if (tid < q1 - q0) {
    auto first = [&](uint32_t q) {  // first entry with a q of at least this one
      uint32_t lo = 0, hi = n;
      while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if ((uint32_t)(s_sort[mid] >> 48) < q) lo = mid + 1u;
        else hi = mid;
      }
      return lo;
    };
    const uint32_t a = first(q0 + tid), b = first(q0 + tid + 1u);
    tcount[s * 256u + q0 + tid] = b - a;
    toff[s * 256u + q0 + tid] = off + a;
    if (b > a) atomicAdd(&s_keys, 1u);
  }
  __syncthreads();
  if (tid == 0) {
    part_n[blockIdx.x] = n;
    part_keys[blockIdx.x] = s_keys;
  }
}

// Table ids of scale blockIdx.x's keys (after the keys of the parts before its
// own), and their size classes' lists. Workgroup 0 also sums up, in res: [0]
// keys in all, [1] entries in all, [2] most entries of one scale.
__global__ __launch_bounds__(256) void number_keys(const uint32_t *__restrict__ tcount,
                                                   const uint32_t *__restrict__ part_keys,
                                                   const uint32_t *__restrict__ part_n, uint32_t scales, uint32_t parts,
                                                   uint32_t T, uint32_t qvals, uint32_t *__restrict__ tgid,
                                                   uint32_t *__restrict__ gid_tkey, uint32_t *lists, uint32_t cap,
                                                   uint32_t *n3, uint32_t *res) {
  __shared__ uint32_t s_tmp[16], s_before, s_all[3];
  const uint32_t tid = threadIdx.x;
  if (tid == 0) s_before = s_all[0] = s_all[1] = s_all[2] = 0u;
  __syncthreads();
  uint32_t before = 0;
  for (uint32_t i = tid; i < blockIdx.x * parts; i += 256u) before += part_keys[i];
  if (before) atomicAdd(&s_before, before);
  __syncthreads();
  const uint32_t tk = blockIdx.x * 256u + tid;
  const uint32_t ni = tid < qvals ? tcount[tk] : 0u;
  const uint32_t gid = s_before + block_exclusive_scan(ni ? 1u : 0u, s_tmp, nullptr);
  if (ni) {
    tgid[tk] = gid;
    gid_tkey[gid] = tk;
  }
  cb_append(gid, ni ? cb_class(ni, T) : -1, lists, cap, n3);
  if (blockIdx.x != 0) return;
  uint32_t keys = 0, entries = 0, most = 0;
  for (uint32_t s = tid; s < scales; s += 256u) {
    uint32_t d = 0;
    for (uint32_t p = 0; p < parts; ++p) {
      keys += part_keys[s * parts + p];
      d += part_n[s * parts + p];
    }
    entries += d;
    most = most > d ? most : d;
  }
  atomicAdd(&s_all[0], keys);
  atomicAdd(&s_all[1], entries);
  atomicMax(&s_all[2], most);
  __syncthreads();
  if (tid < 3u) res[tid] = s_all[tid];
}

// Code word of an element, 16 bits (L <= 11): code | length << 11 | raw16 << 15.
__device__ __forceinline__ uint32_t cw16(uint32_t cw) {
  return (cw & 0x7FFu) | (cw_len(cw) << 11) | ((cw & kRaw) ? 0x8000u : 0u);
}
__device__ __forceinline__ uint32_t cw16_len(uint32_t c) { return (c >> 11) & 0xFu; }

// Pieces of a unit: piece j of substream t is steps [i0 + j * per, + per) of the
// unit, up to 1024 / k_eff pieces side by side; thread j * k_eff + t has it.
__device__ __forceinline__ uint32_t piece_steps(const Unit &u, uint32_t k_eff) {
  const uint32_t nsub = kUnitThreads / k_eff;
  return (u.i1 - u.i0 + nsub - 1u) / nsub;
}
struct UnitPiece {
  uint32_t lane, i, iend;  // substream, first step and end (none: i >= iend)
};
__device__ __forceinline__ UnitPiece unit_piece(const Unit &u, uint32_t k_eff) {
  const uint32_t sub = threadIdx.x / k_eff, per = piece_steps(u, k_eff);
  UnitPiece p;
  p.lane = threadIdx.x - sub * k_eff;
  p.i = u.i0 + sub * per;
  p.iend = sub >= kUnitThreads / k_eff ? 0u : p.i + per < u.i1 ? p.i + per : u.i1;
  return p;
}

// The unit's elements as code words (codes[bucket_elem[b] + e], e in bucket
// order) and each piece's bits (piece_bits[unit * 1024 + thread]).
template <uint32_t kSlots>
__global__ __launch_bounds__(kUnitThreads) void unit_codes(UnitArgs a, uint32_t parts,
                                                           const uint32_t *__restrict__ part_off,
                                                           const uint32_t *__restrict__ part_n,
                                                           const uint64_t *__restrict__ skeys,
                                                           const uint32_t *__restrict__ entry_cw,
                                                           const uint32_t *__restrict__ bucket_elem,
                                                           uint16_t *__restrict__ codes,
                                                           uint32_t *__restrict__ piece_bits, uint32_t *err) {
  __shared__ uint2 s_map[kSlots];  // pair, code word
  __shared__ uint32_t s_base[kUnitRows + 2];
  const uint32_t tid = threadIdx.x;
  const Unit u = a.units[blockIdx.x];
  const UnitGeom g = unit_geom(a, u, s_base);
  for (uint32_t i = tid; i < kSlots; i += kUnitThreads) s_map[i] = make_uint2(kNoPair, 0u);
  __syncthreads();
  for (uint32_t p = 0; p < parts; ++p) {
    const uint32_t off = part_off[u.sidx * parts + p], n = part_n[u.sidx * parts + p];
    for (uint32_t i = tid; i < n; i += kUnitThreads) {
      const uint64_t key = skeys[off + i];
      const uint32_t pair = ((uint32_t)(key >> 48) << 16) | cb_sym(key);
      const uint32_t cw = cw16(entry_cw[off + i]);
      uint32_t h = pair_slot<kSlots>(pair);
      while (atomicCAS(&s_map[h].x, kNoPair, pair) != kNoPair) h = (h + pair_step(pair)) & (kSlots - 1u);
      s_map[h].y = cw;
    }
  }
  __syncthreads();
  const UnitPiece pc = unit_piece(u, g.k_eff);
  uint32_t bits = 0;
  bool found = true;
  uint16_t *out = codes + bucket_elem[u.bucket];
  // The piece's element, its row (from the unit's first) and column: a step is the
  // same for every work-item, plus a carry. (A division an element bounded the pass.)
  const uint32_t dr = g.k_eff / g.cl, dc = g.k_eff - dr * g.cl;
  uint32_t at = pc.lane + pc.i * g.k_eff;
  uint32_t row = at / g.cl, col = at - row * g.cl;
  row -= g.r0;
  constexpr int kB = 8;  // elements in flight a work-item
  for (uint32_t i = pc.i; i < pc.iend; i += kB) {
    uint32_t pair[kB], e[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      const bool in = i + j < pc.iend && at < g.e1;
      e[j] = in ? at : kNoPair;
      // past the end: the unit's first row, not stored
      const uint32_t idx = s_base[in ? row : 0u] + (in ? col : 0u);
      at += g.k_eff;
      row += dr;
      col += dc;
      const bool carry = col >= g.cl;
      row += carry ? 1u : 0u;
      col -= carry ? g.cl : 0u;
      pair[j] = ((uint32_t)(a.q[idx] & a.qmask) << 16) | a.bf16[idx];
    }
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      uint32_t h = pair_slot<kSlots>(pair[j]);
      uint2 s = s_map[h];
      while (s.x != pair[j] && s.x != kNoPair) {
        h = (h + pair_step(pair[j])) & (kSlots - 1u);
        s = s_map[h];
      }
      found &= s.x == pair[j];
      if (e[j] != kNoPair) {
        out[e[j]] = (uint16_t)s.y;
        bits += cw16_len(s.y) + ((s.y >> 15) << 4);
      }
    }
  }
  piece_bits[(uint64_t)blockIdx.x * kUnitThreads + tid] = bits;
  if (!found) atomicOr(err, 4u);
}

// Bucket blockIdx.x's substreams: start bits (k + 1 of them) from the pieces'
// bits, each piece's offset from its substream's start (in place), and the
// bucket's bits. The workgroup that finishes last (`done` counts them, from
// zero) then lays out the buckets: 64-bit aligned bases, and the end of the last
// bucket unaligned (build_huffman.cu:813-818).
__global__ __launch_bounds__(kUnitThreads) void bucket_starts(const Unit *__restrict__ units,
                                                              const uint32_t *__restrict__ bucket_unit,
                                                              const uint32_t *__restrict__ lane_base, uint32_t k,
                                                              uint32_t *__restrict__ piece_bits,
                                                              uint32_t *__restrict__ startbit,
                                                              uint32_t *bucket_bits, int64_t *__restrict__ bit_base,
                                                              uint32_t *done, int64_t *__restrict__ end) {
  __shared__ uint32_t s_tmp[16];
  __shared__ bool s_last;
  const uint32_t b = blockIdx.x, t = threadIdx.x;
  const uint32_t k_eff = lane_base[b + 1] - lane_base[b];
  uint32_t acc = 0;
  if (t < k_eff) {
    for (uint32_t i = bucket_unit[b]; i < bucket_unit[b + 1]; ++i) {
      const Unit u = units[i];
      const uint32_t per = piece_steps(u, k_eff), np = (u.i1 - u.i0 + per - 1u) / per;
      uint32_t *pb = piece_bits + (uint64_t)i * kUnitThreads + t;
      for (uint32_t j0 = 0; j0 < np; j0 += 4) {  // four loads at a time
        uint32_t v[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) v[j] = j0 + j < np ? pb[(j0 + j) * k_eff] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
          if (j0 + j < np) pb[(j0 + j) * k_eff] = acc;
          acc += v[j];
        }
      }
    }
  }
  uint32_t total = 0;
  const uint32_t ex = block_exclusive_scan(acc, s_tmp, &total);
  uint32_t *sb = startbit + (uint64_t)b * (k + 1u);
  if (t < k) sb[t + 1] = t < k_eff ? ex + acc : total;
  if (t == 0) {
    sb[0] = 0u;
    __hip_atomic_store(bucket_bits + b, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u;
  }
  __syncthreads();
  if (!s_last) return;
  const uint32_t B = gridDim.x;
  uint64_t run = 0;  // 64-bit words
  for (uint32_t b0 = 0; b0 < B; b0 += kUnitThreads) {
    const bool in = b0 + t < B;
    const uint32_t bits = in ? __hip_atomic_load(bucket_bits + b0 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    const uint32_t words = (uint32_t)(((uint64_t)bits + 63u) >> 6);
    uint32_t sum = 0;
    const uint32_t first = block_exclusive_scan(words, s_tmp, &sum);
    if (in) bit_base[b0 + t] = (int64_t)((run + first) << 6);
    if (b0 + t + 1u == B) bit_base[B] = *end = (int64_t)(((run + first) << 6) + bits);
    run += sum;
  }
}

// The unit's pieces into the bitstream, MSB-first in 32-bit chunks (chunk c of
// the stream is u32 c ^ 1: a 64-bit word's first half is its high half).
//
// A chunk is written by the piece that holds its first bit, whole: the piece
// goes on with the codes that follow its own (the substream's next steps, then
// the next substream's) until its last chunk is full or the bucket ends, and
// leaves out a first chunk that began before it. Merging shared chunks with
// atomics instead (two a piece, and the stream zeroed first) bounded the pass:
// device-scope atomics passed at some 8 G/s.
// Measured on 14336 x 4096, k = 1024: 259 us with atomics, 137 us without, 91 us
// with neighbouring units on one XCD (below); 4096 x 4096 AWQ 157 -> 32 us.
// Staging the chunks in LDS to write a piece's run from eight lanes did not
// help (313 us against 259, both with the atomics).
// kJoin codes of at most 28 (7 x 4) or 22 (11 x 2) bits in all enter the bit
// buffer together (14336 x 4096: 91 -> 85 us); a raw symbol among them is taken
// up code by code. Loading a batch ahead did not help (83 us, but 4096 x 4096
// AWQ 31 -> 36 us).
template <int kJoin>
__global__ __launch_bounds__(kUnitThreads) void unit_pack(UnitArgs a, uint32_t num_units,
                                                          const uint32_t *__restrict__ bucket_elem,
                                                          const uint16_t *__restrict__ codes,
                                                          const uint32_t *__restrict__ piece_at,
                                                          const uint32_t *__restrict__ startbit,
                                                          const int64_t *__restrict__ bit_base,
                                                          uint32_t *__restrict__ chunks) {
  // consecutive units (one substream's neighbouring pieces) on one XCD, whose L2 then merges their lines
  const uint32_t per = gridDim.x / 8u, unit = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
  if (unit >= num_units) return;
  const Unit u = a.units[unit];
  const int32_t ra = a.row_offsets[u.bucket];
  const uint32_t cl = (uint32_t)a.col_len[u.bucket];
  const uint32_t total = (uint32_t)(a.row_offsets[u.bucket + 1] - ra) * cl;
  const uint32_t k_eff = a.k < total ? a.k : total;
  const UnitPiece pc = unit_piece(u, k_eff);
  if (pc.i >= pc.iend) return;
  const uint32_t *sb = startbit + (uint64_t)u.bucket * (a.k + 1u);
  const uint64_t base = (uint64_t)bit_base[u.bucket];
  const uint64_t p0 = base + sb[pc.lane] + piece_at[(uint64_t)unit * kUnitThreads + threadIdx.x];
  uint64_t c = p0 >> 5;
  uint64_t acc = 0;                      // bits from the top: `used` of them
  uint32_t used = (uint32_t)(p0 & 31u);  // < 32 between codes
  bool own = used == 0u;                 // the chunk being filled began here
  auto put = [&](uint32_t v, uint32_t len) {
    acc |= (uint64_t)v << (64u - used - len);
    used += len;
    if (used >= 32u) {
      if (own) chunks[c ^ 1u] = (uint32_t)(acc >> 32);
      own = true;
      ++c;
      acc <<= 32;
      used -= 32u;
    }
  };
  const uint16_t *in = codes + bucket_elem[u.bucket];
  auto put_code = [&](uint32_t w, uint32_t e) {
    const uint32_t len = cw16_len(w);
    if (len) put(w & 0x7FFu, len);
    if (w & 0x8000u) {
      const uint32_t r = e / cl;
      const int32_t at = ra + (int32_t)r;
      const uint32_t col = (uint32_t)(a.row_col ? a.row_col[at] : a.col_start[u.bucket]) + (e - r * cl);
      put(a.bf16[(uint64_t)(uint32_t)a.row_indices[at] * a.m + col], 16u);
    }
  };
  constexpr int kB = 8;  // codes loaded at a time
  for (uint32_t i = pc.i; i < pc.iend; i += kB) {
    uint32_t w[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      const uint32_t e = pc.lane + (i + j) * k_eff;
      w[j] = i + j < pc.iend && e < total ? in[e] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kB; j += kJoin) {
      uint32_t raw = 0, v = 0, len = 0;
#pragma unroll
      for (int x = j; x < j + kJoin; ++x) {
        const uint32_t l = cw16_len(w[x]);
        raw |= w[x] & 0x8000u;
        v = (v << l) | (w[x] & 0x7FFu);
        len += l;
      }
      if (raw) {
#pragma unroll
        for (int x = j; x < j + kJoin; ++x) put_code(w[x], pc.lane + (i + x) * k_eff);
      } else if (len) {
        put(v, len);
      }
    }
  }
  // The rest of the last chunk.
  uint32_t lane = pc.lane, i = pc.iend;
  const uint64_t last = c;
  while (own && used && c == last) {
    uint32_t w[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      const uint32_t e = lane + (i + j) * k_eff;
      w[j] = e < total ? in[e] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kB; ++j)
      if (c == last) put_code(w[j], lane + (i + j) * k_eff);
    i += kB;
    if (c == last && lane + i * k_eff >= total) {  // the next substream
      i = 0;
      if (++lane == k_eff) {
        chunks[c ^ 1u] = (uint32_t)(acc >> 32);
        break;
      }
    }
  }
  // A bucket of an odd number of chunks ends with half a word of padding.
  if (pc.lane + 1u == k_eff && pc.iend * (uint64_t)k_eff >= total) {
    const uint64_t end = (base + sb[k_eff] + 31u) >> 5;
    if (end & 1u) chunks[end ^ 1u] = 0u;
  }
}
