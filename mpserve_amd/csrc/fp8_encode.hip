// GPU sidecar builder for the FP8 + Huffman weight path (MI355X, gfx950).
//
// Produces byte for byte what the reference's host builder
// huffman_build_fp8_decode_tables_entry (kernel/build_huffman.cu:292-969) produces:
//   1. histogram of (scale, fp8) keys x BF16 symbols    (:392-401)
//   2. keys in ascending order -> table id (gid)         (:403-412)
//   3. per key: ESC selection, package-merge lengths,    (:445-578)   -> a wave or a workgroup per key, in LDS
//      canonical codes in (count asc, sym asc) order,
//      decode LUT and packed 4-bit lengths
//   4. row buckets, bucket_table, U/uniq/uidx            (:582-783)   -> rows dealt to their scales by a counting
//                                                                        sort (few: on the host), tables by a kernel
//   5. per-lane bit counts, u32 lane starts, 64-bit      (:786-925)
//      aligned bucket bases, MSB-first packing
// Steps 1, 2 and 5 run on units of one bucket over tables in LDS
// (encode_units.h). The general path further down, over hash tables in global
// memory with a work-item a substream, takes the calls the units do not: codes
// longer than 11 bits, fewer than 32 substreams, tensors past 2^31 elements,
// very small buckets, and scales with more pairs than an LDS table holds.
// The reference is single-threaded; here every O(N) pass runs on the GPU.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_segmented_radix_sort.hpp>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <exception>
#include <memory>
#include <new>
#include <string>
#include <vector>

#include "mps_common.h"

namespace mps {
namespace {

constexpr uint64_t kEmpty = ~0ull;
constexpr uint32_t kRaw = 1u << 31;  // code word flag: 16 raw symbol bits follow the code

// Code word of one element: bits 0..15 code, 16..20 length, bit 31 raw16 follows.
__device__ __forceinline__ uint32_t cw_len(uint32_t cw) { return (cw >> 16) & 0x1Fu; }

__device__ __forceinline__ uint64_t hash64(uint64_t k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// ---------------------------------------------------------------------------
// Element addressing shared by the passes.
// ---------------------------------------------------------------------------
struct ScaleMap {
  // mode 0: scalar/per-row (row_sidx[row]); mode 1: block-2D (block_sidx[br*nb1+bc])
  int32_t mode;
  const uint16_t *row_sidx;
  const uint16_t *block_sidx;
  int64_t sb0, sb1, nb1;
};

__device__ __forceinline__ uint32_t sidx_of(const ScaleMap &S, int64_t row, int64_t col) {
  if (S.mode == 0) return S.row_sidx[row];
  return S.block_sidx[(row / S.sb0) * S.nb1 + col / S.sb1];
}

// key40 = sidx << 24 | fp8 << 16 | sym
__device__ __forceinline__ uint64_t key40(uint32_t sidx, uint32_t q, uint32_t sym) {
  return ((uint64_t)sidx << 24) | ((uint64_t)q << 16) | (uint64_t)sym;
}

// ---------------------------------------------------------------------------
// 1. Histogram
// ---------------------------------------------------------------------------
constexpr int kHistBlock = 256;
constexpr int kLdsSlots = 2048;

__device__ bool global_insert(uint64_t *keys, uint32_t *counts, uint64_t cap_mask, uint64_t k, uint32_t add) {
  uint64_t h = hash64(k) & cap_mask;
  for (uint64_t probe = 0; probe <= cap_mask; ++probe) {
    unsigned long long *slot = reinterpret_cast<unsigned long long *>(keys + h);
    unsigned long long cur = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (cur == kEmpty) {
      cur = atomicCAS(slot, (unsigned long long)kEmpty, (unsigned long long)k);
      if (cur == kEmpty) cur = k;
    }
    if (cur == k) {
      atomicAdd(counts + h, add);
      return true;
    }
    h = (h + 1) & cap_mask;
  }
  return false;
}

__global__ __launch_bounds__(kHistBlock) void hist_kernel(const uint16_t *__restrict__ bf16, const uint8_t *__restrict__ fp8,
                                                          int64_t n, int64_t m, ScaleMap S, uint32_t qmask,
                                                          int64_t elems_per_block, uint64_t *keys, uint32_t *counts,
                                                          uint64_t cap_mask, uint32_t *overflow) {
  __shared__ unsigned long long s_keys[kLdsSlots];
  __shared__ uint32_t s_cnt[kLdsSlots];
  for (int i = threadIdx.x; i < kLdsSlots; i += kHistBlock) {
    s_keys[i] = kEmpty;
    s_cnt[i] = 0;
  }
  __syncthreads();
  const int64_t numel = n * m;
  const int64_t e0 = (int64_t)blockIdx.x * elems_per_block;
  const int64_t e1 = e0 + elems_per_block < numel ? e0 + elems_per_block : numel;
  for (int64_t e = e0 + threadIdx.x; e < e1; e += kHistBlock) {
    const int64_t row = e / m, col = e - row * m;
    const uint64_t k = key40(sidx_of(S, row, col), fp8[e] & qmask, bf16[e]);
    // LDS first: a short probe, then the global table.
    uint32_t h = (uint32_t)(hash64(k) & (kLdsSlots - 1));
    bool done = false;
    for (int probe = 0; probe < 16 && !done; ++probe) {
      unsigned long long cur = s_keys[h];
      if (cur == kEmpty) {
        cur = atomicCAS(&s_keys[h], (unsigned long long)kEmpty, (unsigned long long)k);
        if (cur == kEmpty) cur = k;
      }
      if (cur == k) {
        atomicAdd(&s_cnt[h], 1u);
        done = true;
      }
      h = (h + 1) & (kLdsSlots - 1);
    }
    if (!done && !global_insert(keys, counts, cap_mask, k, 1)) atomicOr(overflow, 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kLdsSlots; i += kHistBlock) {
    if (s_keys[i] != kEmpty && !global_insert(keys, counts, cap_mask, s_keys[i], s_cnt[i])) atomicOr(overflow, 1u);
  }
}

// ---------------------------------------------------------------------------
// 2. Compaction (ballot + prefix within the wave, one atomic per wave)
// ---------------------------------------------------------------------------
__global__ void compact_kernel(const uint64_t *__restrict__ keys, const uint32_t *__restrict__ counts, uint64_t cap,
                               uint64_t *ckey, uint32_t *ccount, uint32_t *cslot, uint32_t *num) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = i < cap && keys[i] != kEmpty;
  const uint64_t mask = __ballot(live);
  const int lane = threadIdx.x & 63;
  const uint32_t below = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  uint32_t base = 0;
  if (lane == 0 && mask) base = atomicAdd(num, (uint32_t)__popcll(mask));
  base = __shfl(base, 0);
  if (live) {
    ckey[base + below] = keys[i];
    ccount[base + below] = counts[i];
    cslot[base + below] = (uint32_t)i;
  }
}

// ---------------------------------------------------------------------------
// Generic exclusive scan of u32 (two levels, up to 2^24 elements per level pair)
// ---------------------------------------------------------------------------
constexpr int kScanBlock = 1024;
constexpr int kScanItems = 4;  // per thread
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *s_tmp, uint32_t *total) {
  // wave-level inclusive scan, then across waves
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) s_tmp[wave] = x;
  __syncthreads();
  if (wave == 0) {
    const int nw = blockDim.x >> 6;
    uint32_t w = lane < nw ? s_tmp[lane] : 0u;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = __shfl_up(w, d);
      if (lane >= d) w += y;
    }
    if (lane < nw) s_tmp[lane] = w;
  }
  __syncthreads();
  const uint32_t before = wave > 0 ? s_tmp[wave - 1] : 0u;
  if (total) *total = s_tmp[(blockDim.x >> 6) - 1];
  __syncthreads();
  return before + x - v;
}

__global__ __launch_bounds__(kScanBlock) void scan_tiles(const uint32_t *in, uint32_t *out, uint64_t n,
                                                         uint32_t *tile_sums) {
  __shared__ uint32_t s_tmp[16];
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
  uint32_t v[kScanItems], s = 0;
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    v[j] = base + j < n ? in[base + j] : 0u;
    s += v[j];
  }
  uint32_t total = 0;
  uint32_t ex = block_exclusive_scan(s, s_tmp, &total);
#pragma unroll
  for (int j = 0; j < kScanItems; ++j) {
    if (base + j < n) out[base + j] = ex;
    ex += v[j];
  }
  if (threadIdx.x == 0 && tile_sums) tile_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanBlock) void scan_add(uint32_t *out, uint64_t n, const uint32_t *tile_offsets) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
  const uint32_t add = tile_offsets[blockIdx.x];
#pragma unroll
  for (int j = 0; j < kScanItems; ++j)
    if (base + j < n) out[base + j] += add;
}

// ---------------------------------------------------------------------------
// Table grouping
// ---------------------------------------------------------------------------
__global__ void table_count_kernel(const uint64_t *ckey, uint32_t num, uint32_t *tcount) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < num) atomicAdd(tcount + (ckey[i] >> 16), 1u);
}

__global__ void nonzero_kernel(const uint32_t *tcount, uint64_t T, uint32_t *nz) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < T) nz[i] = tcount[i] ? 1u : 0u;
}

__global__ void scatter_kernel(const uint64_t *ckey, const uint32_t *ccount, const uint32_t *cslot, uint32_t num,
                               const uint32_t *toff, uint32_t *tfill, uint16_t *seg_sym, uint32_t *seg_cnt,
                               uint32_t *seg_slot) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num) return;
  const uint64_t tk = ckey[i] >> 16;
  const uint32_t pos = toff[tk] + atomicAdd(tfill + tk, 1u);
  seg_sym[pos] = (uint16_t)(ckey[i] & 0xFFFF);
  seg_cnt[pos] = ccount[i];
  seg_slot[pos] = cslot[i];
}

// gid -> table key, for the non-empty table keys in ascending order
__global__ void table_list_kernel(const uint32_t *tcount, const uint32_t *tgid, uint64_t T, uint32_t *gid_tkey) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < T && tcount[i]) gid_tkey[tgid[i]] = (uint32_t)i;
}

// ---------------------------------------------------------------------------
// 3. Code book of one key, L >= 12 (one work-item per key; L <= 11 further down)
// ---------------------------------------------------------------------------
// Items (count, sym) compare as the reference's std::pair<int, uint16_t>.
// Items are ordered by (count, symbol) with counts compared as int, as the
// reference's item lists are: the sort key flips the count's sign bit so that
// an unsigned 64-bit compare orders it as a signed one.
__device__ __forceinline__ uint64_t item_key(uint32_t count, uint32_t sym) {
  return ((uint64_t)(count ^ 0x80000000u) << 16) | (sym & 0xFFFFu);
}
__device__ __forceinline__ uint32_t key_count(uint64_t k) { return (uint32_t)(k >> 16) ^ 0x80000000u; }

// Sorts n (key, value) pairs by key (distinct keys) with a bottom-up merge
// sort over runs of 16 made by insertion; tk/tv are scratch of n each. The
// result is in k/v.
__device__ void sort_pairs(uint64_t *k, uint32_t *v, uint64_t *tk, uint32_t *tv, uint32_t n) {
  constexpr uint32_t kRun = 16;
  for (uint32_t lo = 0; lo < n; lo += kRun) {
    const uint32_t hi = lo + kRun < n ? lo + kRun : n;
    for (uint32_t i = lo + 1; i < hi; ++i) {
      const uint64_t x = k[i];
      const uint32_t y = v[i];
      uint32_t j = i;
      for (; j > lo && k[j - 1] > x; --j) {
        k[j] = k[j - 1];
        v[j] = v[j - 1];
      }
      k[j] = x;
      v[j] = y;
    }
  }
  uint64_t *sk = k, *dk = tk;
  uint32_t *sv = v, *dv = tv;
  for (uint32_t width = kRun; width < n; width *= 2) {
    for (uint32_t lo = 0; lo < n; lo += 2 * width) {
      const uint32_t mid = lo + width < n ? lo + width : n;
      const uint32_t hi = lo + 2 * width < n ? lo + 2 * width : n;
      uint32_t i = lo, j = mid, o = lo;
      while (i < mid && j < hi) {
        const bool right = sk[j] < sk[i];
        dk[o] = right ? sk[j] : sk[i];
        dv[o] = right ? sv[j] : sv[i];
        i += right ? 0u : 1u;
        j += right ? 1u : 0u;
        ++o;
      }
      for (; i < mid; ++i, ++o) {
        dk[o] = sk[i];
        dv[o] = sv[i];
      }
      for (; j < hi; ++j, ++o) {
        dk[o] = sk[j];
        dv[o] = sv[j];
      }
    }
    uint64_t *t64 = sk;
    sk = dk;
    dk = t64;
    uint32_t *t32 = sv;
    sv = dv;
    dv = t32;
  }
  if (sk != k) {
    for (uint32_t i = 0; i < n; ++i) {
      k[i] = sk[i];
      v[i] = sv[i];
    }
  }
}

// Code lengths of n ascending weights by the package-merge (build_huffman.cu:46-118),
// in the level-count form: with cur_0 = the leaves and cur_j = merge(leaves,
// pairs of cur_{j-1}) (leaf first on equal weight, at most 4(n-1) items), the
// reference selects the first 2(n-1) items of cur_{L-1} and, recursively, the
// first 2p items of cur_{j-1} for the p packages selected in cur_j. Leaves keep
// their sorted order in every cur_j, so a level's selected prefix holds leaves
// 0..x_j-1, and a leaf's length is the number of levels with x_j above its
// index. The levels are built once, bottom-up (O(L n)); each keeps only a bit
// per item saying whether it is a leaf (masks: L words per 32 items of 4(n-1)),
// and the selection then walks them top-down. A and B hold 4(n-1) ints each.
__device__ void package_merge_lengths(const int32_t *w, int n, int L, int32_t *A, int32_t *B, uint32_t *masks,
                                      int32_t *lens) {
  for (int i = 0; i < n; ++i) lens[i] = 0;
  if (n == 1) {
    lens[0] = 1;
    return;
  }
  const int keep = 4 * (n - 1);
  const int words = (keep + 31) / 32;
  int na[16];
  int cur = n < keep ? n : keep;
  for (int i = 0; i < cur; ++i) A[i] = w[i];
  for (int i = 0; i < words; ++i) {
    const int b = cur - 32 * i;
    masks[i] = b >= 32 ? 0xFFFFFFFFu : (b > 0 ? (1u << b) - 1u : 0u);
  }
  na[0] = cur;
  for (int j = 1; j < L; ++j) {
    uint32_t *mk = masks + j * words;
    for (int i = 0; i < words; ++i) mk[i] = 0u;
    const int np = cur / 2;  // packages: pairs (0,1), (2,3), ... of the previous level
    int a = 0, b = 0, o = 0;
    while (o < keep && (a < n || b < np)) {
      const int32_t pw = b < np ? (int32_t)((uint32_t)A[2 * b] + (uint32_t)A[2 * b + 1]) : 0;
      if (a < n && (b >= np || w[a] <= pw)) {
        B[o] = w[a++];
        mk[o >> 5] |= 1u << (o & 31);
      } else {
        B[o] = pw;
        ++b;
      }
      ++o;
    }
    int32_t *t = A;
    A = B;
    B = t;
    cur = o;
    na[j] = o;
  }
  int c = 2 * (n - 1);  // selected prefix at the top level
  for (int level = L - 1; level >= 0 && c > 0; --level) {
    const int cc = c < na[level] ? c : na[level];
    const uint32_t *mk = masks + level * words;
    int x = 0;
    for (int i = 0; i < cc / 32; ++i) x += __popc(mk[i]);
    if (cc & 31) x += __popc(mk[cc / 32] & ((1u << (cc & 31)) - 1u));
    for (int i = 0; i < x; ++i) lens[i] += 1;
    c = 2 * (cc - x);
  }
}

// ESC rules of the three builders:
//  kEscFp8        build_huffman.cu:485-535 and :205-228: esc_sym = smallest u16 not kept, list re-sorted
//                 (count asc, sym asc), the ESC entries' nibble is len | 8.
//  kEscAwqBucket  build_huffman.cu:1775-1836: as kEscFp8 (ESC weight at least 1), but the ESC code
//                 has length L and its one LUT entry has nibble 15.
//  kEscAwqByScale build_huffman.cu:1251-1316: esc_sym = smallest u16 absent from all of the key's
//                 symbols (0xFFFF if none is); the list stays (count desc, sym asc) with ESC last, and
//                 the lengths package-merge returns for the sorted weights apply to it by position;
//                 ESC length L, nibble 15.
enum : int { kEscFp8 = 0, kEscAwqBucket = 1, kEscAwqByScale = 2 };

struct CodebookArgs {
  const uint32_t *gid_tkey;
  const uint32_t *toff;
  const uint32_t *tcount;
  uint16_t *seg_sym;  // sorted in place
  uint32_t *seg_cnt;
  uint32_t *seg_slot;  // hash slot of each entry; sorted along with seg_sym/seg_cnt
  int32_t *ws;        // per key: kWsSort ints per histogram entry + kWsPerItem per list item (ws_size_kernel)
  const uint32_t *ws_off;
  const uint16_t *scale_values;  // sidx -> scale u16
  uint32_t *cw_slot;             // hash slot -> code word
  uint16_t *decode_syms;         // [G, 2^L]
  uint8_t *decode_lens;          // [G, 2^(L-1)] (or [G,1] when L == 1)
  uint16_t *table_scale;
  uint16_t *table_fp8;
  uint32_t G;
  int L;
  int esc_mode;  // kEscFp8, kEscAwqBucket or kEscAwqByScale
  uint32_t *err;
  uint32_t *esc_stats;  // [0] keys with ESC, [1] collisions (elements)
};

// Workspace per key, in ints: sort scratch over the ni histogram entries
// (two 64-bit keys and two 32-bit values each, later the entry -> list
// position map), then per list item (nmax = min(ni, 2^L)): weights, symbols,
// lengths, histogram index, code, two package-merge lists of 4 items, the
// level masks (2, plus kWsFixed for the per-level rounding) and the sorted
// weights.
constexpr uint32_t kWsSort = 6;
constexpr uint32_t kWsPerItem = 16;
constexpr uint32_t kWsFixed = 20;

// One work-item per key: ESC selection, package-merge lengths, canonical codes
// in list order, the decode table and the code word of each histogram entry.
__global__ void codebook_kernel(CodebookArgs a) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= a.G) return;
  const int L = a.L;
  const uint32_t T = 1u << L;
  const uint32_t tk = a.gid_tkey[g];
  const uint32_t off = a.toff[tk];
  const uint32_t ni = a.tcount[tk];
  uint16_t *sym = a.seg_sym + off;
  uint32_t *cnt = a.seg_cnt + off;
  uint32_t *slot = a.seg_slot + off;
  a.table_scale[g] = a.scale_values[tk >> 8];
  a.table_fp8[g] = (uint16_t)(tk & 0xFF);
  uint16_t *dsyms = a.decode_syms + (uint64_t)g * T;
  uint8_t *dlens = a.decode_lens + (uint64_t)g * (T / 2 > 0 ? T / 2 : 1);

  if (ni == 1) {
    for (uint32_t j = 0; j < T; ++j) dsyms[j] = sym[0];
    for (uint32_t j = 0; j < T / 2; ++j) dlens[j] = 0x11;  // len 1 in both nibbles
    a.cw_slot[slot[0]] = (1u << 16) | 0u;
    return;
  }
  int32_t *ws = a.ws + a.ws_off[g];
  uint64_t *sk = reinterpret_cast<uint64_t *>(ws);  // 8-byte aligned: every key's size is even
  uint64_t *tk64 = sk + ni;
  uint32_t *sv = reinterpret_cast<uint32_t *>(tk64 + ni);
  uint32_t *tv = sv + ni;
  const uint32_t nmax = ni < T ? ni : T;
  int32_t *lw = ws + kWsSort * ni;  // weights of the coded list
  int32_t *ls = lw + nmax;          // its symbols
  int32_t *lens = ls + nmax;
  int32_t *hidx = lens + nmax;      // histogram entry of each list item (-1: the ESC item)
  uint32_t *code = reinterpret_cast<uint32_t *>(hidx + nmax);
  int32_t *A = reinterpret_cast<int32_t *>(code + nmax);
  int32_t *Bv = A + 4 * nmax;
  uint32_t *masks = reinterpret_cast<uint32_t *>(Bv + 4 * nmax);  // L * ceil(4(nmax-1)/32) <= 2 nmax + 16
  int32_t *sw = reinterpret_cast<int32_t *>(masks + 2 * nmax + 16);  // sorted weights (kEscAwqByScale)

  // (count asc, sym asc)
  for (uint32_t i = 0; i < ni; ++i) {
    sk[i] = item_key(cnt[i], sym[i]);
    sv[i] = slot[i];
  }
  sort_pairs(sk, sv, tk64, tv, ni);
  for (uint32_t i = 0; i < ni; ++i) {
    sym[i] = (uint16_t)(sk[i] & 0xFFFFu);
    cnt[i] = key_count(sk[i]);
    slot[i] = sv[i];
  }

  uint32_t nl = 0;
  bool use_esc = false;
  uint32_t esc_sym = 0;
  if (ni > T) {
    // ESC (build_huffman.cu:485-535): keep the 2^L-1 most frequent by (count
    // desc, sym asc); ESC weight = sum of the rest. In (count asc, sym asc)
    // order, count groups are taken from the top, each from its smallest symbol.
    use_esc = true;
    const uint32_t keep = T - 1;
    uint32_t taken = 0;
    int64_t i = (int64_t)ni - 1;
    while (taken < keep && i >= 0) {
      int64_t j = i;
      while (j > 0 && cnt[j - 1] == cnt[i]) --j;
      const uint32_t gsize = (uint32_t)(i - j + 1);
      const uint32_t take = gsize < keep - taken ? gsize : keep - taken;
      for (uint32_t t = 0; t < take; ++t) {
        lw[nl] = (int32_t)cnt[j + t];
        ls[nl] = sym[j + t];
        hidx[nl] = (int32_t)(j + t);
        ++nl;
      }
      taken += take;
      i = j - 1;
    }
    // ESC weight: total minus kept (int sums as in the reference)
    uint32_t total = 0;
    for (uint32_t t = 0; t < ni; ++t) total += cnt[t];
    uint32_t kept_sum = 0;
    for (uint32_t t = 0; t < nl; ++t) kept_sum += (uint32_t)lw[t];
    const uint32_t esc_w = total - kept_sum;
    if (a.esc_mode == kEscAwqByScale) {
      // Smallest u16 absent from all ni (distinct) symbols: the largest c with
      // #{sym < c} == c, found by bisection over c in [0, 65536].
      uint32_t lo = 0, hi = 65536;
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        uint32_t below = 0;
        for (uint32_t t = 0; t < ni; ++t) below += sym[t] < mid;
        if (below == mid) lo = mid;
        else hi = mid - 1;
      }
      esc_sym = lo > 0xFFFFu ? 0xFFFFu : lo;
      // The list keeps its (count desc, sym asc) order with ESC last; the
      // package-merge gets the same weights ascending: the kept ones reversed,
      // the ESC weight merged in.
      const int32_t ew = (int32_t)esc_w;
      uint32_t o = 0;
      bool placed = false;
      for (int64_t t = (int64_t)nl - 1; t >= 0; --t) {
        if (!placed && ew <= lw[t]) {
          sw[o++] = ew;
          placed = true;
        }
        sw[o++] = lw[t];
      }
      if (!placed) sw[o++] = ew;
      lw[nl] = ew;
      ls[nl] = (int32_t)esc_sym;
      hidx[nl] = -1;
      ++nl;
      atomicAdd(&a.esc_stats[0], 1u);
    } else {
      // smallest u16 not among the kept: their symbols sorted
      for (uint32_t t = 0; t < nl; ++t) {
        sk[t] = (uint64_t)(uint32_t)ls[t];
        sv[t] = 0u;
      }
      sort_pairs(sk, sv, tk64, tv, nl);
      uint32_t cand = 0;
      for (uint32_t p = 0; p < nl; ++p) {
        if ((uint32_t)sk[p] == cand) ++cand;
        else if ((uint32_t)sk[p] > cand) break;
      }
      esc_sym = cand & 0xFFFF;
      lw[nl] = (a.esc_mode == kEscAwqBucket && (int32_t)esc_w <= 0) ? 1 : (int32_t)esc_w;
      ls[nl] = (int32_t)esc_sym;
      hidx[nl] = -1;
      ++nl;
      // the list in (count asc, sym asc) order, with each item's histogram entry
      for (uint32_t t = 0; t < nl; ++t) {
        sk[t] = item_key((uint32_t)lw[t], (uint32_t)ls[t]);
        sv[t] = (uint32_t)hidx[t];
      }
      sort_pairs(sk, sv, tk64, tv, nl);
      for (uint32_t t = 0; t < nl; ++t) {
        lw[t] = (int32_t)key_count(sk[t]);
        ls[t] = (int32_t)(sk[t] & 0xFFFFu);
        hidx[t] = (int32_t)sv[t];
      }
      atomicAdd(&a.esc_stats[0], 1u);
    }
  } else {
    for (uint32_t t = 0; t < ni; ++t) {
      lw[t] = (int32_t)cnt[t];
      ls[t] = sym[t];
      hidx[t] = (int32_t)t;
    }
    nl = ni;
  }
  if (a.esc_mode == kEscAwqByScale && use_esc) {
    // package-merge sorts the weights and returns lengths by sorted position;
    // the reference applies them to its (unsorted) list position by position
    package_merge_lengths(sw, (int)nl, L, A, Bv, masks, lens);
  } else {
    // weights are ascending (as int); package-merge expects that order
    package_merge_lengths(lw, (int)nl, L, A, Bv, masks, lens);
  }
  // canonical codes (build_huffman.cu:171-203), handed out in list order
  uint32_t bl_count[16], next_code[16];
  for (int b = 0; b < 16; ++b) bl_count[b] = 0;
  for (uint32_t t = 0; t < nl; ++t) {
    if (lens[t] <= 0 || lens[t] > L) {
      atomicOr(a.err, 2u);
      return;
    }
    if (use_esc && a.esc_mode != kEscFp8 && (uint32_t)ls[t] == esc_sym) lens[t] = L;  // AWQ: ESC code has length L
    bl_count[lens[t]]++;
  }
  uint32_t cd = 0;
  next_code[0] = 0;
  for (int b = 1; b < 16; ++b) {
    cd = (cd + bl_count[b - 1]) << 1;
    next_code[b] = cd;
  }
  for (uint32_t j = 0; j < T; ++j) dsyms[j] = 0;
  for (uint32_t j = 0; j < T / 2; ++j) dlens[j] = 0;
  uint32_t esc_cw = 0;
  for (uint32_t t = 0; t < nl; ++t) {
    const int len = lens[t];
    const uint32_t c = next_code[len]++;
    code[t] = c;
    const uint32_t fill = 1u << (L - len);
    const uint32_t base = c << (L - len);
    const bool is_esc = use_esc && (uint32_t)ls[t] == esc_sym;
    const uint32_t nib = is_esc ? (a.esc_mode == kEscFp8 ? ((uint32_t)len | 0x8u) : 15u) : (uint32_t)len;
    for (uint32_t f = 0; f < fill; ++f) {
      const uint32_t e = base + f;
      dsyms[e] = (uint16_t)ls[t];
      if (T >= 2) dlens[e >> 1] |= (uint8_t)((nib & 0xF) << ((e & 1) * 4));
    }
    if (is_esc) esc_cw = ((uint32_t)len << 16) | (c & 0xFFFF);
  }
  // code word of every histogram entry: its list item's code; an entry outside
  // the list is coded as ESC + 16 raw bits, except one whose symbol is esc_sym
  // (the ESC code alone: a collision, as in the reference)
  int32_t *pos_of = ws;  // the sort scratch is free again
  for (uint32_t t = 0; t < ni; ++t) pos_of[t] = -1;
  for (uint32_t p = 0; p < nl; ++p)
    if (hidx[p] >= 0) pos_of[hidx[p]] = (int32_t)p;
  for (uint32_t t = 0; t < ni; ++t) {
    const int32_t p = pos_of[t];
    uint32_t cw;
    if (p >= 0) {
      cw = ((uint32_t)lens[p] << 16) | (code[p] & 0xFFFF);
    } else if (use_esc && sym[t] == esc_sym) {
      cw = esc_cw;
      atomicAdd(&a.esc_stats[1], cnt[t]);
    } else {
      cw = esc_cw | kRaw;  // outside the map: ESC code + raw16
    }
    a.cw_slot[slot[t]] = cw;
  }
}

// ---------------------------------------------------------------------------
// Codebooks, L <= 11. A key's histogram entries arrive sorted, in (count asc,
// sym asc) order; one workgroup builds its codebook in LDS (keys of at most 64
// entries: one wave, codebook_small_kernel):
//  - the ESC keep set from the sorted counts: the entry at ni - (2^L - 1) fixes
//    the boundary count c; every entry above c's run is kept, and the run's
//    first ones (smallest symbols) fill the rest;
//  - esc_sym from a 65536-bit set of the symbols in LDS;
//  - the package-merge levels built once, bottom-up. A merge is a merge path of
//    four outputs a work-item (leaf first on equal weight): one binary search,
//    four items in turn, their two pairs written as the next level's packages
//    and their leaf bits as half a byte. So a level is some fifteen LDS reads in
//    a chain and one barrier. The selection then counts leaf bits top-down;
//  - canonical codes in list order, ranked within each length by ballots;
//  - the decode table, entry by entry (prefix minus a length's first code,
//    below its count, is the code's rank), and the code word of the histogram
//    entry behind each list item.
// What bounds it is the chain of one key: a tensor has few long lists (128 past
// 512 entries of the AWQ weight below), so a key gets the work-items that make
// the chain short, and everything searched is in LDS.
//
// Weights add up as the reference's ints do. A package holds a leaf at most once
// a level, so sums stay below 11 times the key's total; a key whose sums could
// wrap, and leave the packages unsorted, is merged in sequence by one lane, as
// the reference merges.
//
// Measured on the 2,600 keys of a 4096 x 4096 AWQ weight: lists past 512 with a
// wave a key (32 outputs a lane) 343 us, with 512 work-items a key and each item
// ranked by a search of its own 142, so 39; lists past 64 104, 60, 27 us.
// ---------------------------------------------------------------------------
constexpr int kCbSmall = 64;  // keys of at most this many entries and no ESC: codebook_small_kernel
constexpr int kCbMaxL = 11;

__device__ __forceinline__ uint32_t cb_count(uint64_t k) { return key_count(k); }
__device__ __forceinline__ uint32_t cb_sym(uint64_t k) { return (uint32_t)(k & 0xFFFFu); }

// NMAX bounds the coded list, min(ni, 2^L); a level holds fewer than 2 NMAX items.
template <int NMAX, int NT>
struct CbShared {
  int32_t lw[NMAX];   // list weights
  int32_t sw[NMAX];   // ascending weights for the package-merge (kEscAwqByScale ESC lists)
  int32_t hidx[NMAX];
  uint16_t ls[NMAX];  // list symbols
  uint16_t code[NMAX];
  uint8_t lens[NMAX];
  union {
    struct {
      int32_t pack[2][NMAX];  // a level's items in pairs, this level's and the last one's
      uint32_t masks[kCbMaxL * (NMAX / 16)];
    } pm;
    uint32_t symset[65536 / 32];
    uint16_t by_code[NMAX];  // list positions in code order
  } u;
  uint32_t red[NT / 64];
  uint32_t cnt[NT / 64][16];  // a wave's items of each length
  uint32_t flag;
};

// Sum and minimum over the workgroup, returned to every work-item (two barriers).
template <int NT>
__device__ __forceinline__ uint32_t cb_sum(uint32_t *red, uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += (uint32_t)__shfl_xor((int)v, o);
  if ((threadIdx.x & 63u) == 0u) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) v += red[w];
  __syncthreads();
  return v;
}
template <int NT>
__device__ __forceinline__ uint32_t cb_min(uint32_t *red, uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t w = (uint32_t)__shfl_xor((int)v, o);
    v = w < v ? w : v;
  }
  if ((threadIdx.x & 63u) == 0u) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) v = red[w] < v ? red[w] : v;
  __syncthreads();
  return v;
}

// First of n ascending counts in LDS that is >= c (lower) or > c (upper).
__device__ __forceinline__ uint32_t cb_bound(const int32_t *counts, uint32_t n, int32_t c, bool upper) {
  uint32_t lo = 0, hi = n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    const int32_t x = counts[mid];
    if (upper ? x <= c : x < c) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

template <int NMAX, int NT>
__device__ __forceinline__ void codebook_key(CbShared<NMAX, NT> &S, const CodebookArgs &a, uint32_t g,
                                             const uint64_t *__restrict__ skeys,
                                             const uint32_t *__restrict__ sslots) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const int L = a.L;
  const uint32_t T = 1u << L;
  const uint32_t tk = a.gid_tkey[g];
  const uint32_t off = a.toff[tk];
  const uint32_t ni = a.tcount[tk];
  const uint64_t *keys = skeys + off;
  auto slot_of = [&](uint32_t t) { return sslots ? sslots[off + t] : off + t; };
  uint32_t *dsyms = reinterpret_cast<uint32_t *>(a.decode_syms + (uint64_t)g * T);  // pairs of entries
  uint8_t *dlens = a.decode_lens + (uint64_t)g * (T / 2);
  if (tid == 0) {
    a.table_scale[g] = a.scale_values[tk >> 8];
    a.table_fp8[g] = (uint16_t)(tk & 0xFF);
    S.flag = 0;
  }

  // --- the coded list ---
  const bool use_esc = ni > T;
  const uint32_t keep = T - 1;
  uint32_t nl, s0 = 0, s1 = 0, r = 0, esc_sym = 0, esc_pos = 0;
  int32_t esc_w = 0;
  if (!use_esc) {
    for (uint32_t p = tid; p < ni; p += NT) {
      const uint64_t k = keys[p];
      S.lw[p] = (int32_t)cb_count(k);
      S.ls[p] = (uint16_t)cb_sym(k);
    }
    nl = ni;
  } else {
    // kept: [s0, s0 + r) and [s1, ni), the top 2^L - 1 by (count desc, sym asc)
    const uint32_t c = cb_count(keys[ni - keep]);
    uint32_t tot = 0, kept = 0;
    for (uint32_t t = tid; t < ni; t += NT) {
      const uint32_t cnt = cb_count(keys[t]);
      tot += cnt;
      kept += (int32_t)cnt > (int32_t)c ? cnt : 0u;
      s0 += (int32_t)cnt < (int32_t)c ? 1u : 0u;
      s1 += (int32_t)cnt <= (int32_t)c ? 1u : 0u;
    }
    s0 = cb_sum<NT>(S.red, s0);
    s1 = cb_sum<NT>(S.red, s1);
    r = keep - (ni - s1);
    tot = cb_sum<NT>(S.red, tot);
    kept = cb_sum<NT>(S.red, kept) + r * c;
    const uint32_t ew = tot - kept;  // int sums as in the reference
    // esc_sym: the smallest u16 absent from the key's symbols (kEscAwqByScale) or
    // from the kept ones (the other builders)
    for (uint32_t i = tid; i < 65536 / 32; i += NT) S.u.symset[i] = 0u;
    __syncthreads();
    for (uint32_t t = tid; t < ni; t += NT) {
      const bool in = a.esc_mode == kEscAwqByScale || t >= s1 || (t >= s0 && t < s0 + r);
      if (in) {
        const uint32_t sy = cb_sym(keys[t]);
        atomicOr(&S.u.symset[sy >> 5], 1u << (sy & 31));
      }
    }
    __syncthreads();
    uint32_t cand = 0xFFFFFFFFu;
    for (uint32_t i = tid; i < 65536 / 32; i += NT) {
      const uint32_t wv = ~S.u.symset[i];
      if (wv != 0u && cand == 0xFFFFFFFFu) cand = 32u * i + (uint32_t)__builtin_ctz(wv);
    }
    cand = cb_min<NT>(S.red, cand);
    __syncthreads();
    if (a.esc_mode == kEscAwqByScale) {
      esc_sym = cand == 0xFFFFFFFFu ? 0xFFFFu : cand;
      esc_w = (int32_t)ew;
      // The kept counts, ascending: entry j of a run [j0, j1) of one count sits at
      // keep - j1 + (j - j0) in the list, which is (count desc, sym asc), ESC last.
      // The package-merge's weights are the same counts with the ESC weight merged
      // in (ties: any order gives the same list).
      int32_t *asc = S.u.pm.pack[0];
      uint32_t e_pos = 0;  // kept counts < the ESC weight (as int)
      for (uint32_t j = tid; j < keep; j += NT) {
        const int32_t c = (int32_t)cb_count(keys[j < r ? s0 + j : s1 + (j - r)]);
        asc[j] = c;
        e_pos += c < esc_w ? 1u : 0u;
      }
      e_pos = cb_sum<NT>(S.red, e_pos);
      for (uint32_t j = tid; j < keep; j += NT) {
        const uint32_t t = j < r ? s0 + j : s1 + (j - r);
        const int32_t c = asc[j];
        const uint32_t j0 = cb_bound(asc, keep, c, false), j1 = cb_bound(asc, keep, c, true);
        const uint32_t pos = keep - j1 + (j - j0);
        S.sw[j + (j >= e_pos ? 1u : 0u)] = c;
        S.lw[pos] = c;
        S.ls[pos] = (uint16_t)cb_sym(keys[t]);
        S.hidx[pos] = (int32_t)t;
      }
      if (tid == 0) {
        S.sw[e_pos] = esc_w;
        S.lw[keep] = esc_w;
        S.ls[keep] = (uint16_t)esc_sym;
        S.hidx[keep] = -1;
      }
      esc_pos = keep;
    } else {
      esc_sym = cand & 0xFFFFu;
      esc_w = (a.esc_mode == kEscAwqBucket && (int32_t)ew <= 0) ? 1 : (int32_t)ew;
      // (count asc, sym asc): the kept entries in sorted order with the ESC item
      // inserted at its key's place
      const uint64_t ek = item_key((uint32_t)esc_w, esc_sym);
      uint32_t below = 0;
      for (uint32_t j = tid; j < keep; j += NT) {
        const uint32_t t = j < r ? s0 + j : s1 + (j - r);
        below += item_key(cb_count(keys[t]), cb_sym(keys[t])) < ek ? 1u : 0u;
      }
      esc_pos = cb_sum<NT>(S.red, below);
      for (uint32_t j = tid; j < keep; j += NT) {
        const uint32_t t = j < r ? s0 + j : s1 + (j - r);
        const uint32_t p = j + (j >= esc_pos ? 1u : 0u);
        const uint64_t k = keys[t];
        S.lw[p] = (int32_t)cb_count(k);
        S.ls[p] = (uint16_t)cb_sym(k);
        S.hidx[p] = (int32_t)t;
      }
      if (tid == 0) {
        S.lw[esc_pos] = esc_w;
        S.ls[esc_pos] = (uint16_t)esc_sym;
        S.hidx[esc_pos] = -1;
      }
    }
    nl = T;
    if (tid == 0) atomicAdd(&a.esc_stats[0], 1u);
  }
  __syncthreads();

  // --- package-merge lengths (see package_merge_lengths) ---
  const int32_t *W = (use_esc && a.esc_mode == kEscAwqByScale) ? S.sw : S.lw;
  const uint32_t n = nl, keep_pm = 4u * (n - 1u);
  uint32_t xs[kCbMaxL];  // leaves among each level's selected prefix
  {
    uint32_t sum = 0;
    for (uint32_t i = tid; i < n; i += NT) sum += (uint32_t)W[i];
    const bool wraps = cb_sum<NT>(S.red, sum) >= (1u << 31) / 12u;
    int32_t *from = S.u.pm.pack[0], *to = S.u.pm.pack[1];
    uint32_t have = n < keep_pm ? n : keep_pm;
    uint32_t sizes[kCbMaxL];
    constexpr uint32_t kWords = NMAX / 16;  // of a level's mask
    static_assert(4 * NT == 2 * NMAX, "four outputs of a level a work-item");
    for (uint32_t b = tid; b < have / 2u; b += NT) from[b] = (int32_t)((uint32_t)W[2u * b] + (uint32_t)W[2u * b + 1u]);
    for (uint32_t i = tid; i < kWords; i += NT) {
      const uint32_t lo = 32u * i;
      S.u.pm.masks[i] = have >= lo + 32u ? 0xFFFFFFFFu : have > lo ? (1u << (have - lo)) - 1u : 0u;
    }
    sizes[0] = have;
    __syncthreads();
#pragma unroll
    for (int j = 1; j < kCbMaxL; ++j) {
      sizes[j] = 0;
      if (j >= L) continue;
      const uint32_t np = have / 2u;
      uint8_t *mk = reinterpret_cast<uint8_t *>(S.u.pm.masks + j * kWords);
      have = n + np < keep_pm ? n + np : keep_pm;
      sizes[j] = have;
      if (wraps) {
        if (tid == 0) {
          uint32_t bits = 0, last = 0;
          for (uint32_t o = 0, x = 0, b = 0; o < have; ++o) {
            const bool leaf = x < n && (b >= np || W[x] <= from[b]);
            const uint32_t v = (uint32_t)(leaf ? W[x++] : from[b++]);
            bits = (bits >> 1) | (leaf ? 0x80u : 0u);
            if (o & 1u) to[o >> 1] = (int32_t)(last + v);
            last = v;
            if ((o & 7u) == 7u) mk[o >> 3] = (uint8_t)bits;
            else if (o + 1u == have) mk[o >> 3] = (uint8_t)((bits & 0xFFu) >> (7u - (o & 7u)));
          }
        }
      } else {
        const uint32_t o = 4u * tid;  // this work-item's outputs: [o, o + 4)
        uint32_t bits = 0;
        if (o < have) {
          uint32_t lo = o > np ? o - np : 0u, hi = o < n ? o : n;
          while (lo < hi) {  // how many leaves are among the first o
            const uint32_t mid = (lo + hi) >> 1;
            if (W[mid] <= from[o - 1u - mid]) lo = mid + 1u;
            else hi = mid;
          }
          uint32_t x = lo, b = o - lo;
          int32_t wv = W[x < n ? x : n - 1u], pv = from[b], v[4];
#pragma unroll
          for (uint32_t i = 0; i < 4u; ++i) {
            const bool leaf = x < n && (b >= np || wv <= pv);
            v[i] = leaf ? wv : pv;
            bits |= leaf ? 1u << i : 0u;
            x += leaf ? 1u : 0u;
            b += leaf ? 0u : 1u;
            if (i < 3u) {
              const int32_t next = *(leaf ? W + (x < n ? x : n - 1u) : from + (b < np ? b : 0u));
              wv = leaf ? next : wv;
              pv = leaf ? pv : next;
            }
          }
          if (o + 1u < have) to[2u * tid] = v[0] + v[1];
          if (o + 3u < have) to[2u * tid + 1u] = v[2] + v[3];
        }
        const uint32_t other = (uint32_t)__shfl_xor((int)bits, 1);
        if (!(tid & 1u)) mk[tid >> 1] = (uint8_t)(bits | (other << 4));
      }
      int32_t *const swap = from;
      from = to;
      to = swap;
      __syncthreads();
    }
    // top-down, by every wave for itself
    uint32_t c = 2u * (n - 1u);
#pragma unroll
    for (int j = kCbMaxL - 1; j >= 0; --j) {
      xs[j] = 0;
      if (j >= L || c == 0u) continue;
      const uint32_t cc = c < sizes[j] ? c : sizes[j];
      const uint32_t *mk = S.u.pm.masks + j * kWords;
      uint32_t x = 0;
      for (uint32_t i = lane; i < (cc + 31u) / 32u; i += 64u) {
        const uint32_t rem = cc - 32u * i;
        x += (uint32_t)__popc(rem >= 32u ? mk[i] : (mk[i] & ((1u << rem) - 1u)));
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x += (uint32_t)__shfl_xor((int)x, o);
      xs[j] = x;
      c = 2u * (cc - x);
    }
  }

  // --- canonical codes (build_huffman.cu:171-203), handed out in list order ---
  // Wave w has the items [w * per, + per): counts first, then codes.
  const uint32_t per = (n + NT - 1u) / NT * 64u;
  const uint32_t p0 = wave * per, p1 = p0 + per < n ? p0 + per : n;
  uint32_t mine = 0;  // lane v: this wave's items of length v
  for (uint32_t b = p0; b < p1; b += 64u) {
    const uint32_t p = b + lane;
    int len = 0;
    if (p < p1) {
#pragma unroll
      for (int j = 0; j < kCbMaxL; ++j) len += p < xs[j] ? 1 : 0;
      if (len <= 0 || len > L) S.flag = 1;
      if (use_esc && a.esc_mode != kEscFp8 && (uint32_t)S.ls[p] == esc_sym) len = L;  // AWQ: ESC code has length L
      S.lens[p] = (uint8_t)len;
    }
#pragma unroll
    for (int v = 1; v <= kCbMaxL; ++v) {
      const uint32_t c = (uint32_t)__popcll(__ballot(len == v));
      mine += lane == (uint32_t)v ? c : 0u;
    }
  }
  if (lane < 16u) S.cnt[wave][lane] = mine;
  __syncthreads();  // (the masks are read: by_code may take their place)
  if (S.flag) {
    if (tid == 0) atomicOr(a.err, 2u);
    return;
  }
  uint32_t all = 0, before = 0;  // lane v: items of length v in all, and in the waves before
  if (lane < 16u) {
#pragma unroll
    for (uint32_t w = 0; w < NT / 64; ++w) {
      const uint32_t c = S.cnt[w][lane];
      all += c;
      before += w < wave ? c : 0u;
    }
  }
  uint32_t first[kCbMaxL + 1], num[kCbMaxL + 1], base[kCbMaxL + 1];  // of a length: first code, codes, codes before it
  first[0] = num[0] = base[0] = 0;
  uint32_t next = 0, at_code = 0;  // lane v: the wave's next code of length v, and its place in code order
#pragma unroll
  for (int v = 1; v <= kCbMaxL; ++v) {
    num[v] = (uint32_t)__builtin_amdgcn_readlane((int)all, v);
    first[v] = (first[v - 1] + num[v - 1]) << 1;
    base[v] = base[v - 1] + num[v - 1];
    if (lane == (uint32_t)v) {
      next = first[v] + before;
      at_code = base[v] + before;
    }
  }
  const uint64_t below = lane == 0u ? 0ull : (~0ull >> (64u - lane));
  for (uint32_t b = p0; b < p1; b += 64u) {
    const uint32_t p = b + lane;
    const int len = p < p1 ? S.lens[p] : 0;
    uint32_t rank = 0, got = 0;
#pragma unroll
    for (int v = 1; v <= kCbMaxL; ++v) {
      const uint64_t m = __ballot(len == v);
      if (len == v) rank = (uint32_t)__popcll(m & below);
      if (lane == (uint32_t)v) got = (uint32_t)__popcll(m);
    }
    const uint32_t c = (uint32_t)__shfl((int)next, len) + rank, at = (uint32_t)__shfl((int)at_code, len) + rank;
    if (p < p1) {
      S.code[p] = (uint16_t)c;
      S.u.by_code[at] = (uint16_t)p;
    }
    next += got;
    at_code += got;
  }
  __syncthreads();

  // --- decode table, two entries a work-item ---
  for (uint32_t p = tid; p < T / 2u; p += NT) {
    uint32_t s2 = 0, l2 = 0;
#pragma unroll
    for (uint32_t h = 0; h < 2u; ++h) {
      const uint32_t e = 2u * p + h;
      uint32_t at = 0, len = 0;
#pragma unroll
      for (int v = 1; v <= kCbMaxL; ++v) {
        const uint32_t r = v <= L ? (e >> (L - v)) - first[v] : ~0u;  // wraps when the prefix lies below
        if (r < num[v]) {
          at = base[v] + r;
          len = (uint32_t)v;
        }
      }
      if (len) {
        const uint32_t sy = S.ls[S.u.by_code[at]];
        const uint32_t nib = use_esc && sy == esc_sym ? (a.esc_mode == kEscFp8 ? (len | 0x8u) : 15u) : len;
        s2 |= sy << (16u * h);
        l2 |= (nib & 0xFu) << (4u * h);
      }
    }
    dsyms[p] = s2;
    dlens[p] = (uint8_t)l2;
  }
  const uint32_t esc_cw = use_esc ? ((uint32_t)S.lens[esc_pos] << 16) | (S.code[esc_pos] & 0xFFFFu) : 0u;

  // --- code word of every histogram entry, from its list position ---
  for (uint32_t p = tid; p < n; p += NT) {
    const int32_t t = use_esc ? S.hidx[p] : (int32_t)p;
    if (t >= 0) a.cw_slot[slot_of((uint32_t)t)] = ((uint32_t)S.lens[p] << 16) | (S.code[p] & 0xFFFFu);
  }
  if (!use_esc) return;
  for (uint32_t i = tid; i < ni - keep; i += NT) {  // the entries left out: [0, s0) and [s0 + r, s1)
    const uint32_t t = i < s0 ? i : i + r;
    const bool coded = cb_sym(keys[t]) == esc_sym;  // a data symbol equal to esc_sym: the ESC code alone
    if (coded) atomicAdd(&a.esc_stats[1], cb_count(keys[t]));
    a.cw_slot[slot_of(t)] = coded ? esc_cw : esc_cw | kRaw;  // else ESC code + raw16
  }
}

// The codebooks of the *n keys in `list` (a size class).
template <int NMAX, int NT>
__global__ __launch_bounds__(NT) void codebook_key_kernel(CodebookArgs a, const uint64_t *__restrict__ skeys,
                                                          const uint32_t *__restrict__ sslots,
                                                          const uint32_t *__restrict__ list,
                                                          const uint32_t *__restrict__ n) {
  __shared__ CbShared<NMAX, NT> S;
  const uint32_t count = *n;
  for (uint32_t i = blockIdx.x; i < count; i += gridDim.x) {
    codebook_key<NMAX, NT>(S, a, list[i], skeys, sslots);
    __syncthreads();
  }
}

// Keys of at most 64 entries and no ESC (of an FP8 weight's keys nearly all: a
// normal bin of 8 holds 16 symbols), a wave a key and a list item a lane, held
// in registers: a level's merge is a rank a lane, leaf i lands after the i leaves and the packages lighter than it,
// package b after the b packages and the leaves no heavier (leaf first on equal
// weight), both by binary search in LDS. The leaves' places stay in registers,
// so the selection counts them with a ballot a level, and the canonical codes
// follow from one ballot a length. A decode table entry finds its code by
// length: prefix minus first code below the count.
// Weights add up as the reference's ints do. A package of a level holds a leaf
// at most once a level, so sums stay below 11 x 64 x the largest count; a key
// with a count of 2^21 or more, whose sums could wrap and leave the packages
// unsorted, is merged in sequence by one lane, as the reference merges.
// Measured: 22,000 keys of a 14336 x 4096 FP8 weight 196 -> 50 us, 12,000 of a
// 1024 x 4096 one 122 -> 32 us.
constexpr int kCbWaves = 4;  // waves (keys) a workgroup
__global__ __launch_bounds__(64 * kCbWaves) void codebook_small_kernel(CodebookArgs a,
                                                                       const uint64_t *__restrict__ skeys,
                                                                       const uint32_t *__restrict__ sslots,
                                                                       const uint32_t *__restrict__ list,
                                                                       const uint32_t *__restrict__ n_list) {
  constexpr int kMaxL = kCbMaxL;
  __shared__ int32_t s_leaf[kCbWaves][64], s_pack[kCbWaves][64], s_cur[kCbWaves][128];
  __shared__ uint32_t s_sym[kCbWaves][64];  // symbols in code order
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  int32_t *leaf = s_leaf[wave], *pack = s_pack[wave], *cur = s_cur[wave];
  uint32_t *by_code = s_sym[wave];
  auto lds_sync = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  const int L = a.L;
  const uint32_t T = 1u << L, count = *n_list;
  for (uint32_t at = blockIdx.x * kCbWaves + wave; at < count; at += gridDim.x * kCbWaves) {
    const uint32_t g = list[at];
    const uint32_t tk = a.gid_tkey[g];
    const uint32_t off = a.toff[tk];
    const uint32_t n = a.tcount[tk];
    const bool in = lane < n;
    const uint64_t key = in ? skeys[off + lane] : 0ull;
    const uint32_t slot = in ? (sslots ? sslots[off + lane] : off + lane) : 0u;
    const uint32_t sym = cb_sym(key);
    uint32_t *dsyms = reinterpret_cast<uint32_t *>(a.decode_syms + (uint64_t)g * T);  // pairs of entries
    uint8_t *dlens = a.decode_lens + (uint64_t)g * (T / 2);
    if (lane == 0) {
      a.table_scale[g] = a.scale_values[tk >> 8];
      a.table_fp8[g] = (uint16_t)(tk & 0xFF);
    }
    int len = 1;
    if (n > 1) {
      // --- package-merge (see package_merge_lengths) ---
      const int32_t w = (int32_t)cb_count(key);
      const uint32_t keep = 4u * (n - 1u);
      const bool wraps = __ballot(in && (uint32_t)w >= (1u << 21)) != 0;
      leaf[lane] = w;
      if (in && lane < keep) cur[lane] = w;
      uint32_t have = n < keep ? n : keep;  // items of the level
      uint32_t sizes[kMaxL], place[kMaxL];  // a level's items; this lane's leaf's place in it
      sizes[0] = have;
      place[0] = lane;
      lds_sync();
#pragma unroll
      for (int j = 1; j < kMaxL; ++j) {
        if (j < L) {
          const uint32_t np = have / 2u;
          int32_t pw = 0;
          if (lane < np) pw = (int32_t)((uint32_t)cur[2u * lane] + (uint32_t)cur[2u * lane + 1u]);
          pack[lane] = pw;
          lds_sync();
          if (wraps) {
            by_code[lane] = keep;  // (a leaf that is not merged has no place)
            lds_sync();
            if (lane == 0) {
              for (uint32_t o = 0, x = 0, b = 0; o < keep && (x < n || b < np); ++o) {
                if (x < n && (b >= np || leaf[x] <= pack[b])) {
                  cur[o] = leaf[x];
                  by_code[x++] = o;
                } else {
                  cur[o] = pack[b++];
                }
              }
            }
            have = n + np < keep ? n + np : keep;
            sizes[j] = have;
            lds_sync();
            place[j] = by_code[lane];
            lds_sync();
            continue;
          }
          uint32_t lo = 0, hi = np, lo2 = 0, hi2 = n;
          while (__ballot(lo < hi || lo2 < hi2)) {
            const uint32_t mid = (lo + hi) >> 1, mid2 = (lo2 + hi2) >> 1;
            const int32_t x = pack[mid & 63u], x2 = leaf[mid2 & 63u];
            if (lo < hi) {  // packages lighter than this leaf
              if (x < w) lo = mid + 1u;
              else hi = mid;
            }
            if (lo2 < hi2) {  // leaves no heavier than this package
              if (x2 <= pw) lo2 = mid2 + 1u;
              else hi2 = mid2;
            }
          }
          const uint32_t mine = lane + lo, theirs = lane + lo2;
          if (in && mine < keep) cur[mine] = w;
          if (lane < np && theirs < keep) cur[theirs] = pw;
          have = n + np < keep ? n + np : keep;
          sizes[j] = have;
          place[j] = mine;
          lds_sync();
        }
      }
      // top-down: a leaf is coded once more in every level whose selected prefix holds it
      uint32_t c = 2u * (n - 1u);
      len = 0;
#pragma unroll
      for (int j = kMaxL - 1; j >= 0; --j) {
        if (j < L && c > 0u) {
          const uint32_t cc = c < sizes[j] ? c : sizes[j];
          const bool sel = in && place[j] < cc;
          const uint32_t x = (uint32_t)__popcll(__ballot(sel));
          len += sel ? 1 : 0;
          c = 2u * (cc - x);
        }
      }
    }
    if (__ballot(in && (len <= 0 || len > L))) {
      if (lane == 0) atomicOr(a.err, 2u);
      continue;
    }
    // --- canonical codes (build_huffman.cu:171-203), handed out in list order ---
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64u - lane));
    uint32_t first[kMaxL + 1], num[kMaxL + 1], base[kMaxL + 1];  // of a length: first code, codes, codes before it
    uint32_t code = 0, cd = 0, before = 0;
    first[0] = num[0] = base[0] = 0;
#pragma unroll
    for (int v = 1; v <= kMaxL; ++v) {
      const uint64_t m = v <= L ? __ballot(in && len == v) : 0ull;
      cd = (cd + num[v - 1]) << 1;
      first[v] = cd;
      num[v] = (uint32_t)__popcll(m);
      base[v] = before;
      if (in && len == v) {
        const uint32_t r = (uint32_t)__popcll(m & below);
        code = cd + r;
        by_code[before + r] = sym;
      }
      before += num[v];
    }
    if (in) a.cw_slot[slot] = ((uint32_t)len << 16) | (n > 1 ? code & 0xFFFFu : 0u);
    lds_sync();
    // --- decode table: two entries a lane ---
    for (uint32_t p = lane; p < T / 2u; p += 64u) {
      uint32_t s2 = 0, l2 = 0;
#pragma unroll
      for (uint32_t h = 0; h < 2u; ++h) {
        const uint32_t e = 2u * p + h;
        uint32_t at_sym = 0, v_len = 0;
#pragma unroll
        for (int v = 1; v <= kMaxL; ++v) {
          const uint32_t r = v <= L ? (e >> (L - v)) - first[v] : ~0u;  // wraps when the prefix lies below
          if (r < num[v]) {
            at_sym = base[v] + r;
            v_len = (uint32_t)v;
          }
        }
        if (n == 1) {  // one symbol: every entry, length 1
          at_sym = 0;
          v_len = 1;
        }
        if (v_len) {
          s2 |= by_code[at_sym] << (16u * h);
          l2 |= v_len << (4u * h);
        }
      }
      dsyms[p] = s2;
      dlens[p] = (uint8_t)l2;
    }
    lds_sync();  // the next key's lists overwrite these
  }
}

// Size class of a key with ni entries and T = 2^L codes: 0 (at most kCbSmall
// entries, no ESC), 1 (a coded list of at most 512) or 2.
__device__ __forceinline__ int cb_class(uint32_t ni, uint32_t T) {
  const uint32_t nmax = ni < T ? ni : T;
  return ni <= (uint32_t)kCbSmall && ni <= T ? 0 : nmax <= 512u ? 1 : 2;
}

// Appends gid to its class's list (lists: [3][cap]); one atomic per wave and class.
__device__ __forceinline__ void cb_append(uint32_t gid, int cls, uint32_t *lists, uint32_t cap, uint32_t *n3) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const uint64_t m = __ballot(cls == c);
    if (!m) continue;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(n3 + c, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, 0);
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (cls == c) lists[(uint64_t)c * cap + base + (uint32_t)__popcll(m & below)] = gid;
  }
}

__global__ void codebook_classes_kernel(const uint32_t *gid_tkey, const uint32_t *tcount, uint32_t G, uint32_t T,
                                        uint32_t *lists, uint32_t *n3) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  cb_append(g, g < G ? cb_class(tcount[gid_tkey[g]], T) : -1, lists, G, n3);
}

__global__ void item_keys_kernel(const uint16_t *__restrict__ sym, const uint32_t *__restrict__ cnt, uint64_t n,
                                 uint64_t *__restrict__ keys) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) keys[i] = item_key(cnt[i], sym[i]);
}

__global__ void segment_bounds_kernel(const uint32_t *gid_tkey, const uint32_t *toff, const uint32_t *tcount,
                                      uint32_t G, uint32_t *beg, uint32_t *end) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= G) return;
  const uint32_t tk = gid_tkey[g];
  beg[g] = toff[tk];
  end[g] = toff[tk] + tcount[tk];
}

__global__ void ws_size_kernel(const uint32_t *gid_tkey, const uint32_t *tcount, uint32_t G, uint32_t T,
                               uint32_t *sz) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= G) return;
  const uint32_t ni = tcount[gid_tkey[g]];
  const uint32_t n = kWsSort * ni + kWsPerItem * (ni < T ? ni : T) + kWsFixed;
  sz[g] = (n + 1u) & ~1u;  // even, so that every key's 64-bit sort keys are 8-byte aligned
}

// ---------------------------------------------------------------------------
// 4. bucket_table, U / unique gids / fp8 -> uidx (one work-item per bucket)
// ---------------------------------------------------------------------------
// qvals = 256 (FP8 bytes; also U/uniq/uidx): a workgroup a bucket, a work-item
// a byte; or 16 (AWQ int4 values, build_huffman.cu:1973-1982): a work-item an
// entry. (A work-item a bucket walking its 256 bytes took 172 us for 70 to 180
// buckets, all of it latency; this takes 5 us.)
__global__ __launch_bounds__(256) void bucket_table_kernel(const uint16_t *bucket_sidx, uint32_t B, int qvals,
                                                           const uint32_t *tcount, const uint32_t *tgid, int32_t *btab,
                                                           int32_t *bU, int32_t *uniq, int16_t *uidx) {
  __shared__ uint32_t s_tmp[16];
  if (qvals != 256) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (uint64_t)B * qvals) return;
    const uint64_t t = (uint64_t)bucket_sidx[i / qvals] * 256 + i % qvals;
    btab[i] = tcount[t] ? (int32_t)tgid[t] : -1;
    return;
  }
  const uint32_t b = blockIdx.x, c = threadIdx.x;
  const uint64_t t = (uint64_t)bucket_sidx[b] * 256 + c;
  const bool has = tcount[t] != 0;
  const int32_t gid = has ? (int32_t)tgid[t] : -1;
  // gids of one bucket are distinct (one scale, distinct fp8 bytes): first-appearance order is fp8 order
  uint32_t U = 0;
  const uint32_t at = block_exclusive_scan(has ? 1u : 0u, s_tmp, &U);
  btab[(uint64_t)b * 256 + c] = gid;
  uidx[(uint64_t)b * 256 + c] = has ? (int16_t)at : (int16_t)-1;
  if (has) uniq[(uint64_t)b * 256 + at] = gid;
  if (c >= U) uniq[(uint64_t)b * 256 + c] = -1;
  if (c == 0) bU[b] = (int32_t)U;
}

// ---------------------------------------------------------------------------
// 5. Bitstream
// ---------------------------------------------------------------------------
struct LaneArgs {
  const uint16_t *bf16;
  const uint8_t *fp8;
  ScaleMap S;
  int64_t m;
  const int32_t *row_offsets;
  const int32_t *row_indices;
  const int32_t *col_start;
  const int32_t *col_len;
  const int32_t *row_col;     // per-row column start (groups of the by-scale layout) or null
  uint32_t qmask;
  const uint32_t *lane_base;  // [B+1] cumulative k_eff
  uint32_t B;
  int64_t k;
  const uint64_t *keys;
  const uint32_t *cw_slot;
  uint64_t cap_mask;
  uint32_t *cw_elem;    // [numel]
  uint32_t *lane_bits;  // [B, k+1] (count of lane t at [b][t+1])
  uint32_t *err;
};

__device__ __forceinline__ uint32_t find_bucket(const uint32_t *lane_base, uint32_t B, uint32_t g) {
  uint32_t lo = 0, hi = B;  // largest b with lane_base[b] <= g
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (lane_base[mid] <= g) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ void lane_bits_kernel(LaneArgs a) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= a.lane_base[a.B]) return;
  const uint32_t b = find_bucket(a.lane_base, a.B, g);
  const uint32_t t = g - a.lane_base[b];
  const int32_t ra = a.row_offsets[b], rows = a.row_offsets[b + 1] - ra;
  const int32_t c0 = a.row_col ? 0 : a.col_start[b], cl = a.col_len[b];
  const int64_t total = (int64_t)rows * cl;
  const int64_t k_eff = a.lane_base[b + 1] - a.lane_base[b];
  uint64_t bits = 0;
  for (int64_t e = t; e < total; e += k_eff) {
    const int64_t rr = e / cl, cc = e - rr * cl;
    const int64_t row = a.row_indices[ra + rr];
    const int64_t col = (a.row_col ? a.row_col[ra + rr] : c0) + cc;
    const int64_t idx = row * a.m + col;
    const uint64_t k = key40(sidx_of(a.S, row, col), a.fp8[idx] & a.qmask, a.bf16[idx]);
    uint64_t h = hash64(k) & a.cap_mask;
    while (a.keys[h] != k) {
      if (a.keys[h] == kEmpty) {
        atomicOr(a.err, 4u);
        return;
      }
      h = (h + 1) & a.cap_mask;
    }
    const uint32_t cw = a.cw_slot[h];
    a.cw_elem[idx] = cw;
    bits += cw_len(cw) + ((cw & kRaw) ? 16u : 0u);
  }
  a.lane_bits[(uint64_t)b * (a.k + 1) + t + 1] = (uint32_t)bits;
}

// per bucket: inclusive scan of lane bits -> u32 starts; inactive lanes -> starts[k_eff]
__global__ __launch_bounds__(1024) void lane_starts_kernel(uint32_t *startbit, const uint32_t *lane_base, int64_t k,
                                                           uint32_t *bucket_bits) {
  __shared__ uint32_t s_tmp[16];
  const uint32_t b = blockIdx.x;
  const int64_t k_eff = lane_base[b + 1] - lane_base[b];
  uint32_t *sb = startbit + (uint64_t)b * (k + 1);
  const int t = threadIdx.x;
  const uint32_t v = t < k_eff ? sb[t + 1] : 0u;
  uint32_t total = 0;
  const uint32_t ex = block_exclusive_scan(v, s_tmp, &total);
  __syncthreads();
  if (t == 0) sb[0] = 0;
  if (t < k) sb[t + 1] = t < k_eff ? ex + v : total;
  if (t == 0) bucket_bits[b] = total;
}

struct PackArgs {
  const uint16_t *bf16;
  int64_t m;
  const int32_t *row_offsets;
  const int32_t *row_indices;
  const int32_t *col_start;
  const int32_t *col_len;
  const int32_t *row_col;  // as LaneArgs::row_col
  const uint32_t *lane_base;
  uint32_t B;
  int64_t k;
  const uint32_t *cw_elem;
  const uint32_t *startbit;
  const int64_t *bit_base;
  unsigned long long *bits;  // zeroed
};

__device__ __forceinline__ void flush_word(unsigned long long *bits, uint64_t w, uint64_t v, uint64_t first_w,
                                           uint64_t last_w) {
  if (v == 0) return;
  if (w == first_w || w == last_w) atomicOr(bits + w, (unsigned long long)v);
  else bits[w] = v;
}

__global__ void pack_kernel(PackArgs a) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= a.lane_base[a.B]) return;
  const uint32_t b = find_bucket(a.lane_base, a.B, g);
  const uint32_t t = g - a.lane_base[b];
  const int32_t ra = a.row_offsets[b], rows = a.row_offsets[b + 1] - ra;
  const int32_t c0 = a.row_col ? 0 : a.col_start[b], cl = a.col_len[b];
  const int64_t total = (int64_t)rows * cl;
  const int64_t k_eff = a.lane_base[b + 1] - a.lane_base[b];
  const uint32_t *sb = a.startbit + (uint64_t)b * (a.k + 1);
  const uint64_t p0 = (uint64_t)a.bit_base[b] + sb[t];
  const uint64_t p1 = (uint64_t)a.bit_base[b] + sb[t + 1];
  if (p1 == p0) return;
  const uint64_t first_w = p0 >> 6, last_w = (p1 - 1) >> 6;
  uint64_t w = first_w;
  uint64_t acc = 0;          // current word, MSB-first
  uint32_t used = (uint32_t)(p0 & 63);  // bits of the current word already taken by earlier lanes
  auto put = [&](uint32_t v, uint32_t n) {  // append the low n bits of v
    while (n > 0) {
      const uint32_t room = 64 - used;
      const uint32_t take = n < room ? n : room;
      const uint64_t part = (uint64_t)((v >> (n - take)) & ((take == 32) ? 0xFFFFFFFFu : ((1u << take) - 1u)));
      acc |= part << (room - take);
      used += take;
      n -= take;
      if (used == 64) {
        flush_word(a.bits, w, acc, first_w, last_w);
        ++w;
        acc = 0;
        used = 0;
      }
    }
  };
  for (int64_t e = t; e < total; e += k_eff) {
    const int64_t rr = e / cl, cc = e - rr * cl;
    const int64_t idx = (int64_t)a.row_indices[ra + rr] * a.m + (a.row_col ? a.row_col[ra + rr] : c0) + cc;
    const uint32_t cw = a.cw_elem[idx];
    put(cw & 0xFFFF, cw_len(cw));
    if (cw & kRaw) put(a.bf16[idx], 16);
  }
  if (used > 0) flush_word(a.bits, w, acc, first_w, last_w);
}

#include "encode_units.h"

// ---------------------------------------------------------------------------
// Host orchestration
// ---------------------------------------------------------------------------
// The codebook launches, one a size class that has keys (at most most[c]; n3 on
// the device says how many).
void launch_codebooks(const CodebookArgs &cba, const uint64_t *skeys, const uint32_t *sslots, const uint32_t *lists,
                      uint32_t cap, const uint32_t *n3, const uint32_t *most, hipStream_t s) {
  if (most[0])
    hipLaunchKernelGGL(codebook_small_kernel, dim3(std::min((most[0] + kCbWaves - 1) / kCbWaves, 2048u)),
                       dim3(64 * kCbWaves), 0, s, cba, skeys, sslots, lists, n3);
  if (most[1])
    hipLaunchKernelGGL((codebook_key_kernel<512, 256>), dim3(std::min(most[1], 2048u)), dim3(256), 0, s, cba, skeys,
                       sslots, lists + cap, n3 + 1);
  if (most[2])
    hipLaunchKernelGGL((codebook_key_kernel<2048, 1024>), dim3(std::min(most[2], 512u)), dim3(1024), 0, s, cba, skeys,
                       sslots, lists + 2 * (size_t)cap, n3 + 2);
}

template <typename T>
struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  ~DevBuf() { reset(); }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t alloc(size_t count) {
    reset();
    n = count;
    return hipMalloc(&p, sizeof(T) * (count > 0 ? count : 1));
  }
};

hipError_t device_scan(const uint32_t *in, uint32_t *out, uint64_t n, hipStream_t s, uint32_t *total_out) {
  // exclusive scan; total (sum of all) written to host *total_out when non-null (synchronises)
  if (n == 0) {
    if (total_out) *total_out = 0;
    return hipSuccess;
  }
  const uint64_t tiles = (n + kScanTile - 1) / kScanTile;
  DevBuf<uint32_t> sums, sums_ex;
  hipError_t e = sums.alloc(tiles + 1);
  if (e != hipSuccess) return e;
  if ((e = sums_ex.alloc(tiles + 1)) != hipSuccess) return e;
  hipLaunchKernelGGL(scan_tiles, dim3((unsigned)tiles), dim3(kScanBlock), 0, s, in, out, n, sums.p);
  if (tiles > 1) {
    if ((e = device_scan(sums.p, sums_ex.p, tiles, s, nullptr)) != hipSuccess) return e;
    hipLaunchKernelGGL(scan_add, dim3((unsigned)tiles), dim3(kScanBlock), 0, s, out, n, sums_ex.p);
  }
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (total_out) {
    uint32_t last_in = 0, last_out = 0;
    if ((e = hipMemcpyAsync(&last_in, in + n - 1, 4, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipMemcpyAsync(&last_out, out + n - 1, 4, hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
    *total_out = last_in + last_out;
  }
  return hipSuccess;
}

}  // namespace
}  // namespace mps

using namespace mps;

// A handle's result: device arrays in the reference's 17-output order.
struct mps_fp8_sidecar {
  void *out[17] = {};
  int64_t sizes[17] = {};
  int64_t stats[4] = {};  // esc keys, esc collision elements, distinct (key, symbol) pairs, hash capacity
  std::vector<void *> work;
  ~mps_fp8_sidecar() {
    for (void *p : out)
      if (p) (void)hipFree(p);
    free_work();
  }
  void free_work() {
    for (void *p : work) (void)hipFree(p);
    work.clear();
  }
};

namespace mps {
namespace {

enum : int { kFmtFp8 = kEscFp8, kFmtAwqBucket = kEscAwqBucket, kFmtAwqByScale = kEscAwqByScale };

// One builder run, after the entry point's own argument checks.
struct EncodeSpec {
  const uint16_t *bf16;
  const uint8_t *q;  // FP8 bytes, or AWQ int4 values (low nibble)
  const uint16_t *scales;
  int64_t n, m, scale_numel;
  bool scalar, per_row, block2d;
  int64_t nb0, nb1, sb0, sb1;
  int64_t L, k, group_cap;
  int format;
};

constexpr int kOutBytes[17] = {2, 1, 2, 2, 2, 4, 4, 4, 4, 4, 4, 8, 8, 8, 4, 4, 2};  // of an element of each output

// Arrays built on the host travel in one block; those that are outputs are
// copied from it to their own buffers by one launch.
struct Placed {
  const char *src[6];
  char *dst[6];
  uint64_t bytes[6];
};
__global__ void place_kernel(Placed p) {
  const int a = (int)blockIdx.y;
  const uint64_t n = p.bytes[a], at = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (at + 4 <= n) *reinterpret_cast<uint32_t *>(p.dst[a] + at) = *reinterpret_cast<const uint32_t *>(p.src[a] + at);
  else if (at + 2 <= n) *reinterpret_cast<uint16_t *>(p.dst[a] + at) = *reinterpret_cast<const uint16_t *>(p.src[a] + at);
}

// Rows (groups) from which rank_sort deals them to their scales: two more
// launches and their gaps against 2 ns a row on the host and its copies. A build
// with the host's loop and with rank_sort: 4096 groups 352, 361 us; 8192 groups
// 364, 369; 8192 FP8 rows 336, 321; 14,336 rows 542, 527; 32,768 groups 435, 403.
constexpr int64_t kDealMin = 8192;
static_assert(kDealMin >= kSortRanks, "a list of scales holds the values of a sort's ranks");

// Runs the builder. Device memory comes from `alloc` (the 17 outputs by slot,
// workspaces as slot -1); the last kernels may still run when this returns.
int encode_impl(const EncodeSpec &sp, hipStream_t s, mps_encode_alloc alloc, void *ctx, int64_t *sizes17,
                int64_t *stats4) {
  const int64_t n = sp.n, m = sp.m, numel = n * m, L = sp.L, kth = sp.k, scale_numel = sp.scale_numel;
  const bool scale_scalar = sp.scalar, scale_block2d = sp.block2d;
  const int64_t nb0 = sp.nb0, nb1 = sp.nb1, sb0 = sp.sb0, sb1 = sp.sb1;
  const uint32_t qmask = sp.format == kFmtFp8 ? 0xFFu : 0x0Fu;
  const int qvals = sp.format == kFmtFp8 ? 256 : 16;
  hipError_t e;
#define HC(x)                                                   \
  do {                                                          \
    if ((e = (x)) != hipSuccess) return hip_fail(e, #x);        \
  } while (0)
// The output of a slot: `count` elements from the caller's allocator (null for none).
#define OUT(name, T, slot, count)                                                                   \
  T *name = nullptr;                                                                                \
  {                                                                                                 \
    const size_t out_n = (count);                                                                   \
    if (out_n && !(name = static_cast<T *>(alloc(ctx, slot, (int64_t)(sizeof(T) * out_n)))))        \
      return fail(MPS_ERR_NO_MEMORY, "no device memory for output %d of the sidecar builder", slot); \
  }

  // --- the scales' ranks among their sorted distinct values ---
  // [0] how many values; items of each rank, where they are dealt here; the values, ascending;
  // the scales' ranks; the tiles' counts
  const bool by_scale = sp.format == kFmtAwqByScale;
  const int64_t width = scale_block2d ? sb1 : m;               // columns of a row (group) of a bucket
  const int64_t per_row = by_scale && scale_block2d ? nb1 : 1;  // groups of a row
  // Many rows (groups) with a scale each are dealt to their scales by rank_sort;
  // then only their counts and the values come to the host. (The sort's tiles
  // count in 16 bits, up to 2^23 items. It leaves more than kSortRanks values to
  // the host.)
  bool dealt = (scale_block2d ? by_scale && sb0 == 1 : !scale_scalar) && scale_numel >= kDealMin &&
               scale_numel <= ((int64_t)1 << 23);
  const uint32_t tile = (uint32_t)std::max<int64_t>(2048, (scale_numel / 256 + 1023) / 1024 * 1024);
  const uint32_t tiles = dealt ? (uint32_t)((scale_numel + tile - 1) / tile) : 0;
  auto up256 = [](size_t x) { return (x + 255) & ~(size_t)255; };
  const size_t o_counts = 256, o_values = o_counts + (dealt ? 4 * (size_t)kSortRanks : 0);
  const size_t o_ranks = up256(o_values + 2 * std::min<size_t>((size_t)scale_numel, 65536));
  const size_t o_hist = up256(o_ranks + 2 * (size_t)scale_numel);
  std::vector<char> ranked(o_ranks + 2 * (size_t)scale_numel);
  char *d_ranked = static_cast<char *>(alloc(ctx, -1, (int64_t)(o_hist + 4 * (size_t)kSortRanks * tiles)));
  if (!d_ranked) return fail(MPS_ERR_NO_MEMORY, "no device memory for the sidecar builder's scales");
  size_t here = 0;  // bytes of it on the host
  auto fetch_ranked = [&](size_t end) -> int {
    if (end <= here) return MPS_OK;
    HC(hipMemcpyAsync(ranked.data() + here, d_ranked + here, end - here, hipMemcpyDeviceToHost, s));
    HC(hipStreamSynchronize(s));
    here = end;
    return MPS_OK;
  };
  auto *d_count = reinterpret_cast<uint32_t *>(d_ranked);
  auto *d_ranks = reinterpret_cast<uint16_t *>(d_ranked + o_ranks);
  hipLaunchKernelGGL(scale_ranks, dim3(1), dim3(kUnitThreads), 0, s, sp.scales, (uint64_t)scale_numel, d_count, d_ranks,
                     reinterpret_cast<uint16_t *>(d_ranked + o_values));
  int32_t *dealt_rows = nullptr, *dealt_cols = nullptr;
  if (dealt) {
    OUT(x6, int32_t, 6, (size_t)scale_numel);
    OUT(x8, int32_t, 8, by_scale ? (size_t)scale_numel : (size_t)0);
    dealt_rows = x6;
    dealt_cols = x8;
    auto *d_hist = reinterpret_cast<uint32_t *>(d_ranked + o_hist);
    hipLaunchKernelGGL(rank_hist, dim3(tiles), dim3(kUnitThreads), 0, s, d_ranks, (uint32_t)scale_numel, tile, d_count,
                       d_hist);
    hipLaunchKernelGGL(rank_sort, dim3(tiles), dim3(kUnitThreads), 0, s, d_ranks, (uint32_t)scale_numel, tile, d_count,
                       d_hist, reinterpret_cast<uint32_t *>(d_ranked + o_counts), (uint32_t)per_row, (uint32_t)width,
                       dealt_rows, dealt_cols);
  }
  HC(hipGetLastError());
  int ranked_rc = fetch_ranked(dealt ? o_values + 2 * (size_t)kSortRanks : ranked.size());
  if (ranked_rc != MPS_OK) return ranked_rc;
  const uint32_t S = *reinterpret_cast<const uint32_t *>(ranked.data());
  dealt = dealt && S <= kSortRanks;
  if (!dealt && (ranked_rc = fetch_ranked(ranked.size())) != MPS_OK) return ranked_rc;
  const uint16_t *rank = reinterpret_cast<const uint16_t *>(ranked.data() + o_ranks);  // of scale i
  const uint16_t *uniq_sc = reinterpret_cast<const uint16_t *>(ranked.data() + o_values);

  // --- buckets (build_huffman.cu:611-696), host ---
  // Rows (groups, by scale) are dealt to their scales by counting: ascending
  // scales, rows in order within one, which is the reference's stable sort.
  std::vector<int32_t> row_offsets{0};
  std::vector<uint32_t> lane_base{0};
  std::vector<uint16_t> bucket_sidx, bucket_scale;
  std::vector<int32_t> row_indices, cols;  // cols: by bucket, or (by scale) by group
  if (by_scale || !scale_block2d) {
    std::vector<int64_t> at(S + 1, 0);  // first row (group) of each scale
    if (dealt)
      std::copy_n(reinterpret_cast<const uint32_t *>(ranked.data() + o_counts), S, at.begin() + 1);
    else if (scale_block2d)
      for (int64_t i = 0; i < scale_numel; ++i) at[rank[i] + 1] += sb0;
    else if (scale_scalar) at[1] = n;
    else
      for (int64_t i = 0; i < scale_numel; ++i) at[rank[i] + 1] += 1;
    const int64_t cap_rows = by_scale ? sp.group_cap : 128;
    for (uint32_t i = 0; i < S; ++i) {
      const int64_t rows = at[i + 1];
      for (int64_t off = 0; off < rows; off += std::min(cap_rows, rows - off)) {
        bucket_sidx.push_back((uint16_t)i);
        row_offsets.push_back(row_offsets.back() + (int32_t)std::min(cap_rows, rows - off));
      }
      at[i + 1] += at[i];
    }
    if (!dealt) row_indices.resize((size_t)(n * per_row));
    if (by_scale) cols.resize(row_indices.size());
    for (int64_t r = 0; r < n && !dealt; ++r) {
      const uint16_t *rk = rank + (scale_scalar ? 0 : scale_block2d ? r / sb0 * nb1 : r);
      for (int64_t c = 0; c < per_row; ++c) {
        const size_t to = (size_t)at[rk[c]]++;
        row_indices[to] = (int32_t)r;
        if (by_scale) cols[to] = (int32_t)(c * width);
      }
    }
    if (!by_scale) cols.assign(bucket_sidx.size(), 0);
  } else {
    for (int64_t br = 0; br < nb0; ++br) {
      for (int64_t bc = 0; bc < nb1; ++bc) {
        for (int64_t off = 0; off < sb0; off += 128) {
          const int64_t take = std::min<int64_t>(128, sb0 - off);
          for (int64_t q = 0; q < take; ++q) row_indices.push_back((int32_t)(br * sb0 + off + q));
          bucket_sidx.push_back(rank[br * nb1 + bc]);
          cols.push_back((int32_t)(bc * sb1));
          row_offsets.push_back((int32_t)row_indices.size());
        }
      }
    }
  }
  const uint32_t B = (uint32_t)bucket_sidx.size();
  const std::vector<int32_t> col_len(B, (int32_t)width);
  for (uint32_t b = 0; b < B; ++b) {
    const int64_t total = (int64_t)(row_offsets[b + 1] - row_offsets[b]) * width;
    lane_base.push_back(lane_base[b] + (uint32_t)std::min<int64_t>(kth, std::max<int64_t>(1, total)));
    bucket_scale.push_back(uniq_sc[bucket_sidx[b]]);
  }
  const size_t num_rows = dealt ? (size_t)scale_numel : row_indices.size();
  const size_t num_cols = dealt && by_scale ? (size_t)scale_numel : cols.size();
  const bool fp8 = sp.format == kFmtFp8;
  const int64_t shape[4] = {n, m, kth, by_scale ? width : 0};
  const size_t nshape = by_scale ? 4 : 3;

  // --- one device block: the host-built arrays (`put`), then work memory (`take`) ---
  // flags: [0] overflow, [1] error bits, [2..3] esc stats, [4] compact count, [5..7] codebook
  // classes, [8..10] keys, entries and most entries of a scale (number_keys), [11] finished
  // workgroups and [12..13] the stream's end (bucket_starts)
  constexpr int kFlags = 16;
  uint32_t hflags[kFlags] = {};
  std::vector<char> host;
  size_t bytes = 0;
  auto take = [&](size_t sz) {
    const size_t at = bytes;
    bytes += (sz + 255) & ~(size_t)255;
    return at;
  };
  auto put = [&](const void *src, size_t sz) {
    const size_t at = take(sz);
    host.resize(bytes);
    std::memcpy(host.data() + at, src, sz);
    return at;
  };
  const size_t o_flags = put(hflags, sizeof(hflags)), o_scale_values = put(uniq_sc, 2 * (size_t)S),
               o_sidx = put(bucket_sidx.data(), 2 * (size_t)B), o_lane_base = put(lane_base.data(), 4 * lane_base.size()),
               o_bscale = put(bucket_scale.data(), 2 * (size_t)B),
               o_rowoff = put(row_offsets.data(), 4 * row_offsets.size()),
               o_rows = put(row_indices.data(), 4 * row_indices.size()), o_cols = put(cols.data(), 4 * cols.size()),
               o_clen = put(col_len.data(), 4 * (size_t)B), o_shape = put(shape, 8 * nshape);
  char *blk = nullptr;
  uint32_t *flags = nullptr, *d_lane_base = nullptr, *tcount = nullptr, *tgid = nullptr, *gid_tkey = nullptr;
  int32_t *d_row_offsets = nullptr, *d_row_indices = nullptr, *d_cols = nullptr, *d_col_len = nullptr;
  auto at32 = [&](size_t o) { return reinterpret_cast<uint32_t *>(blk + o); };
  // Allocates the block as laid out so far, uploads it and places the outputs it holds.
  // (Where the unit passes gave up after theirs, that block stays: the general path
  // uses its host-built arrays, and clears the flags itself.)
  auto upload = [&]() -> int {
    if (blk) return MPS_OK;
    if (!(blk = static_cast<char *>(alloc(ctx, -1, (int64_t)bytes))))
      return fail(MPS_ERR_NO_MEMORY, "no device memory for the sidecar builder's workspace (%zu bytes)", bytes);
    HC(hipMemcpyAsync(blk, host.data(), host.size(), hipMemcpyHostToDevice, s));
    flags = at32(o_flags);
    d_lane_base = at32(o_lane_base);
    d_row_offsets = reinterpret_cast<int32_t *>(blk + o_rowoff);
    d_row_indices = dealt ? dealt_rows : reinterpret_cast<int32_t *>(blk + o_rows);
    d_cols = dealt && by_scale ? dealt_cols : reinterpret_cast<int32_t *>(blk + o_cols);
    d_col_len = reinterpret_cast<int32_t *>(blk + o_clen);
    OUT(x4, uint16_t, 4, (size_t)B);
    OUT(x5, int32_t, 5, row_offsets.size());
    int32_t *x6 = dealt_rows, *x8 = dealt_cols;  // (or their buffers, where the sort had too many scales)
    if (!x6) {
      OUT(own, int32_t, 6, row_indices.size());
      x6 = own;
    }
    if (!x8) {
      OUT(own, int32_t, 8, cols.size());
      x8 = own;
    }
    OUT(x9, int32_t, 9, by_scale ? (size_t)0 : (size_t)B);
    OUT(x13, int64_t, 13, nshape);
    Placed pl = {{blk + o_bscale, blk + o_rowoff, blk + o_rows, blk + o_cols, blk + o_clen, blk + o_shape},
                 {(char *)x4, (char *)x5, (char *)x6, (char *)x8, (char *)x9, (char *)x13},
                 {2ull * B, 4 * row_offsets.size(), 4 * row_indices.size(), 4 * cols.size(), by_scale ? 0ull : 4ull * B,
                  8 * nshape}};
    const uint64_t longest = *std::max_element(pl.bytes, pl.bytes + 6);
    hipLaunchKernelGGL(place_kernel, dim3((unsigned)((longest + 1023) / 1024), 6), dim3(256), 0, s, pl);
    HC(hipGetLastError());
    return MPS_OK;
  };

  uint32_t D = 0, G = 0;
  uint64_t cap = 0;
  int64_t W = 0;
  const uint64_t T = (uint64_t)S * 256;
  const uint32_t Tsz = 1u << L;
  const uint32_t packed = Tsz / 2 > 0 ? Tsz / 2 : 1;
  CodebookArgs cba{};
  int32_t *btab = nullptr, *bU = nullptr, *uniq = nullptr;
  int16_t *uidx = nullptr;
  auto alloc_tables = [&]() -> int {  // the outputs whose sizes follow from G
    OUT(syms, uint16_t, 0, (size_t)G * Tsz);
    OUT(lens, uint8_t, 1, (size_t)G * packed);
    OUT(tscale, uint16_t, 2, (size_t)G);
    OUT(tq, uint16_t, 3, (size_t)G);
    OUT(x7, int32_t, 7, (size_t)B * qvals);
    OUT(x14, int32_t, 14, fp8 ? (size_t)B : 0);
    OUT(x15, int32_t, 15, fp8 ? (size_t)B * 256 : 0);
    OUT(x16, int16_t, 16, fp8 ? (size_t)B * 256 : 0);
    btab = x7;
    bU = x14;
    uniq = x15;
    uidx = x16;
    cba.gid_tkey = gid_tkey;
    cba.tcount = tcount;
    cba.scale_values = reinterpret_cast<const uint16_t *>(blk + o_scale_values);
    cba.decode_syms = syms;
    cba.decode_lens = lens;
    cba.table_scale = tscale;
    cba.table_fp8 = tq;
    cba.G = G;
    cba.L = (int)L;
    cba.esc_mode = sp.format;
    cba.err = flags + 1;
    cba.esc_stats = flags + 2;
    return MPS_OK;
  };
  auto bucket_tables = [&]() -> int {
    if (B)
      hipLaunchKernelGGL(bucket_table_kernel, dim3(fp8 ? B : (B * 16 + 255) / 256), dim3(256), 0, s,
                         reinterpret_cast<const uint16_t *>(blk + o_sidx), B, qvals, tcount, tgid, btab, bU, uniq, uidx);
    HC(hipGetLastError());
    return MPS_OK;
  };
  auto check_errors = [&]() -> int {
    if (hflags[1] & 2u) return fail(MPS_ERR_RUNTIME, "invalid code length");
    if (hflags[1] & 4u)
      return fail(MPS_ERR_RUNTIME,
                  fp8 ? "missing enc table for (scale,fp8) key" : "missing enc table for (scale,qv) key");
    return MPS_OK;
  };

  // --- the unit passes (encode_units.h) ---
  // Taken when code words fit 16 bits (L <= 11), a workgroup's pieces of a
  // substream stay few (k >= 32), element indexes have room in 32 bits, and the
  // buckets are not so small that a workgroup's LDS set-up outweighs its unit
  // (1024 elements). It gives up (kGeneral) when a unit's or a scale's pairs
  // overflow their LDS tables, as random bit patterns do.
  constexpr int kGeneral = 1;
  auto unit_path = [&]() -> int {
    if (L > 11 || kth < 32 || numel > ((int64_t)1 << 31)) return kGeneral;
    // A unit: about 1/1024 of the tensor, so that four go to a CU; at least 16 Ki
    // elements beside the 64 KiB of LDS each pass sets up.
    const uint64_t target = std::min<uint64_t>(std::max<uint64_t>((uint64_t)numel / 1024, 16384), 1u << 20);
    std::vector<Unit> units;
    std::vector<uint32_t> bucket_unit(B + 1, 0), bucket_elem(B), list_off, scale_units(S + 1, 0);
    std::vector<uint64_t> scale_elems(S, 0);
    uint64_t elem = 0, lists_n = 0;
    for (uint32_t b = 0; b < B; ++b) {
      const uint64_t cl = (uint64_t)width, total = (uint64_t)(row_offsets[b + 1] - row_offsets[b]) * cl;
      const uint64_t ke = lane_base[b + 1] - lane_base[b];
      const uint64_t steps = (total + ke - 1) / ke;
      const uint64_t most = std::max<uint64_t>(1, std::min<uint64_t>(target, (uint64_t)kUnitRows * cl) / ke);
      const uint64_t parts = (steps + most - 1) / most, per = (steps + parts - 1) / parts;
      bucket_unit[b] = (uint32_t)units.size();
      bucket_elem[b] = (uint32_t)elem;
      for (uint64_t i = 0; i < steps; i += per) {
        const uint64_t end = std::min(steps, i + per);
        units.push_back(Unit{b, (uint32_t)i, (uint32_t)end, bucket_sidx[b]});
        list_off.push_back((uint32_t)lists_n);
        lists_n += std::min<uint64_t>((end - i) * ke, kPairSlots);
        ++scale_units[bucket_sidx[b] + 1];
      }
      elem += total;
      scale_elems[bucket_sidx[b]] += total;
    }
    const size_t U = units.size();
    bucket_unit[B] = (uint32_t)U;
    if (U == 0 || (U > 4096 && (uint64_t)numel / U < 1024)) return kGeneral;
    for (uint32_t i = 0; i < S; ++i) scale_units[i + 1] += scale_units[i];
    std::vector<uint32_t> unit_of_scale(U), fill(scale_units.begin(), scale_units.end() - 1);
    for (size_t u = 0; u < U; ++u) unit_of_scale[fill[units[u].sidx]++] = (uint32_t)u;
    // Parts: q ranges of a scale merged by workgroups of their own, two a CU in all.
    const uint32_t P = std::min<uint32_t>((uint32_t)qvals, std::max<uint32_t>(1, std::min<uint32_t>(16, 512 / S)));
    std::vector<uint32_t> part_off((size_t)S * P);
    uint64_t entries = 0;
    for (size_t i = 0; i < part_off.size(); ++i) {
      part_off[i] = (uint32_t)entries;
      entries += std::min<uint64_t>(scale_elems[i / P], kPairSlots);
    }
    // One device block: the host-built arrays, then the passes' own.
    const size_t o_units = put(units.data(), sizeof(Unit) * U), o_bunit = put(bucket_unit.data(), 4 * bucket_unit.size()),
                 o_belem = put(bucket_elem.data(), 4 * (size_t)B), o_loff = put(list_off.data(), 4 * U),
                 o_sunit = put(scale_units.data(), 4 * scale_units.size()),
                 o_uos = put(unit_of_scale.data(), 4 * U), o_poff = put(part_off.data(), 4 * part_off.size());
    const size_t o_ln = take(4 * U), o_pn = take(4 * part_off.size()), o_pk = take(4 * part_off.size()),
                 o_lists = take(8 * lists_n), o_skeys = take(8 * entries), o_cw = take(4 * entries),
                 o_toff = take(4 * T), o_tcount = take(4 * T), o_tgid = take(4 * T), o_tkey = take(4 * T),
                 o_cbl = take(12 * T), o_codes = take(2 * (size_t)numel), o_pieces = take(4 * (size_t)kUnitThreads * U),
                 o_bbits = take(4 * (size_t)B);
    int rc = upload();
    if (rc != MPS_OK) return rc;
    tcount = at32(o_tcount);
    tgid = at32(o_tgid);
    gid_tkey = at32(o_tkey);
    uint32_t *cb_lists = at32(o_cbl);
    UnitArgs ua;
    ua.units = reinterpret_cast<const Unit *>(blk + o_units);
    ua.bf16 = sp.bf16;
    ua.q = sp.q;
    ua.m = (uint32_t)m;
    ua.qmask = qmask;
    ua.row_offsets = d_row_offsets;
    ua.row_indices = d_row_indices;
    ua.col_start = by_scale ? nullptr : d_cols;
    ua.col_len = d_col_len;
    ua.row_col = by_scale ? d_cols : nullptr;
    ua.k = (uint32_t)kth;
    // every row's column range starts and ends on 8 elements (columns start at multiples of the range's width)
    ua.vec8 = m % 8 == 0 && width % 8 == 0 && reinterpret_cast<uintptr_t>(sp.bf16) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(sp.q) % 8 == 0;
    auto *lists = reinterpret_cast<uint2 *>(blk + o_lists);
    auto *skeys = reinterpret_cast<uint64_t *>(blk + o_skeys);
    auto *codes = reinterpret_cast<uint16_t *>(blk + o_codes);
    hipLaunchKernelGGL(unit_hist, dim3((unsigned)U), dim3(kUnitThreads), 0, s, ua, at32(o_loff), lists, at32(o_ln),
                       flags);
    hipLaunchKernelGGL(merge_lists, dim3(S * P), dim3(kUnitThreads), 0, s, at32(o_sunit), at32(o_uos), at32(o_loff),
                       at32(o_ln), lists, P, (uint32_t)qvals, at32(o_poff), skeys, tcount, at32(o_toff), at32(o_pn),
                       at32(o_pk), flags);
    hipLaunchKernelGGL(number_keys, dim3(S), dim3(256), 0, s, tcount, at32(o_pk), at32(o_pn), S, P, Tsz, (uint32_t)qvals,
                       tgid, gid_tkey, cb_lists, (uint32_t)T, flags + 5, flags + 8);
    HC(hipGetLastError());
    HC(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, s));
    HC(hipStreamSynchronize(s));
    const uint32_t most = hflags[10];  // entries of the scale that has most
    if (hflags[0] || most > 12288) return kGeneral;
    G = hflags[8];
    D = hflags[9];
    cap = (uint64_t)S * P * kPairSlots;
    if ((rc = alloc_tables()) != MPS_OK) return rc;
    cba.toff = at32(o_toff);
    cba.cw_slot = at32(o_cw);
    launch_codebooks(cba, skeys, nullptr, cb_lists, (uint32_t)T, flags + 5, hflags + 5, s);
    HC(hipGetLastError());
    if ((rc = bucket_tables()) != MPS_OK) return rc;
    OUT(startbit, uint32_t, 10, (size_t)B * (kth + 1));
    OUT(bit_base, int64_t, 11, (size_t)B + 1);
    // the smaller table (two workgroups a CU) while it is at most 3/4 full
    auto codes_pass = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)U), dim3(kUnitThreads), 0, s, ua, P, at32(o_poff), at32(o_pn), skeys,
                         at32(o_cw), at32(o_belem), codes, at32(o_pieces), flags + 1);
    };
    if (most <= 6144) codes_pass(unit_codes<8192>);
    else codes_pass(unit_codes<16384>);
    hipLaunchKernelGGL(bucket_starts, dim3(B), dim3(kUnitThreads), 0, s, ua.units, at32(o_bunit), d_lane_base,
                       (uint32_t)kth, at32(o_pieces), startbit, at32(o_bbits), bit_base, flags + 11,
                       reinterpret_cast<int64_t *>(flags + 12));
    HC(hipGetLastError());
    HC(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, s));
    HC(hipStreamSynchronize(s));
    if ((rc = check_errors()) != MPS_OK) return rc;
    int64_t end = 0;  // of the bitstream, in bits
    std::memcpy(&end, hflags + 12, sizeof(end));
    W = (end + 63) >> 6;
    OUT(bitstream, uint64_t, 12, (size_t)W);
    if (W) {
      auto pack = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(U + 7) / 8 * 8), dim3(kUnitThreads), 0, s, ua, (uint32_t)U,
                           at32(o_belem), codes, at32(o_pieces), startbit, bit_base,
                           reinterpret_cast<uint32_t *>(bitstream));
      };
      if (L <= 7) pack(unit_pack<4>);
      else pack(unit_pack<2>);
      HC(hipGetLastError());
    }
    return MPS_OK;
  };

  // --- the general path: hash tables in global memory, a work-item a substream ---
  auto general_path = [&]() -> int {
    int rc = upload();
    if (rc != MPS_OK) return rc;
    if ((rc = fetch_ranked(ranked.size())) != MPS_OK) return rc;
    std::vector<uint16_t> row_sidx, block_sidx;
    if (scale_block2d) {
      block_sidx.resize((size_t)(nb0 * nb1));
      for (size_t i = 0; i < block_sidx.size(); ++i) block_sidx[i] = rank[i];
    } else {
      row_sidx.resize((size_t)n);
      for (size_t r = 0; r < row_sidx.size(); ++r) row_sidx[r] = rank[scale_scalar ? 0 : r];
    }
    DevBuf<uint16_t> d_row_sidx, d_block_sidx;
    HC(d_row_sidx.alloc(row_sidx.size()));
    HC(d_block_sidx.alloc(block_sidx.size()));
    if (!row_sidx.empty())
      HC(hipMemcpyAsync(d_row_sidx.p, row_sidx.data(), 2 * row_sidx.size(), hipMemcpyHostToDevice, s));
    if (!block_sidx.empty())
      HC(hipMemcpyAsync(d_block_sidx.p, block_sidx.data(), 2 * block_sidx.size(), hipMemcpyHostToDevice, s));
    ScaleMap smap;
    smap.mode = scale_block2d ? 1 : 0;
    smap.row_sidx = d_row_sidx.p;
    smap.block_sidx = d_block_sidx.p;
    smap.sb0 = sb0;
    smap.sb1 = sb1;
    smap.nb1 = nb1;

    // --- 1. histogram (retry with a larger table on overflow) ---
    DevBuf<uint64_t> keys;
    DevBuf<uint32_t> counts;
    cap = 1u << 16;
    while (cap < (uint64_t)std::min<int64_t>(numel, (int64_t)1 << 22) * 2) cap <<= 1;
    const int64_t per_block = 1 << 14;
    const unsigned hist_blocks = (unsigned)((numel + per_block - 1) / per_block);
    for (;;) {
      HC(keys.alloc(cap));
      HC(counts.alloc(cap));
      HC(hipMemsetAsync(keys.p, 0xFF, sizeof(uint64_t) * cap, s));
      HC(hipMemsetAsync(counts.p, 0, sizeof(uint32_t) * cap, s));
      HC(hipMemsetAsync(flags, 0, sizeof(uint32_t) * kFlags, s));
      hipLaunchKernelGGL(hist_kernel, dim3(hist_blocks), dim3(kHistBlock), 0, s, sp.bf16, sp.q, n, m, smap,
                         qmask, per_block, keys.p, counts.p, cap - 1, flags);
      HC(hipGetLastError());
      HC(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, s));
      HC(hipStreamSynchronize(s));
      if (!hflags[0]) break;
      if (cap >= ((uint64_t)1 << 34)) return fail(MPS_ERR_RUNTIME, "histogram table overflow");
      cap <<= 1;
    }

    // --- 2. compaction and grouping by (scale, fp8) key ---
    DevBuf<uint64_t> ckey;
    DevBuf<uint32_t> ccount, cslot;
    // bound for the compact arrays: count first
    {
      HC(ckey.alloc(cap));
      HC(ccount.alloc(cap));
      HC(cslot.alloc(cap));
      hipLaunchKernelGGL(compact_kernel, dim3((unsigned)((cap + 255) / 256)), dim3(256), 0, s, keys.p, counts.p, cap,
                         ckey.p, ccount.p, cslot.p, flags + 4);
      HC(hipGetLastError());
      HC(hipMemcpyAsync(&D, flags + 4, 4, hipMemcpyDeviceToHost, s));
      HC(hipStreamSynchronize(s));
    }
    DevBuf<uint32_t> toff, tfill, tnz, d_tcount, d_tgid, d_tkey, cb_lists;
    HC(d_tcount.alloc(T));
    tcount = d_tcount.p;
    HC(toff.alloc(T));
    HC(tfill.alloc(T));
    HC(tnz.alloc(T));
    HC(d_tgid.alloc(T));
    tgid = d_tgid.p;
    HC(hipMemsetAsync(tcount, 0, 4 * T, s));
    HC(hipMemsetAsync(tfill.p, 0, 4 * T, s));
    hipLaunchKernelGGL(table_count_kernel, dim3((D + 255) / 256), dim3(256), 0, s, ckey.p, D, tcount);
    HC(hipGetLastError());
    uint32_t D_check = 0;
    G = 0;
    HC(device_scan(tcount, toff.p, T, s, &D_check));
    hipLaunchKernelGGL(nonzero_kernel, dim3((unsigned)((T + 255) / 256)), dim3(256), 0, s, tcount, T, tnz.p);
    HC(hipGetLastError());
    HC(device_scan(tnz.p, tgid, T, s, &G));
    if (D_check != D) return fail(MPS_ERR_RUNTIME, "internal error: histogram grouping mismatch");
    DevBuf<uint16_t> seg_sym;
    DevBuf<uint32_t> seg_cnt, seg_slot, ws_off, cw_slot;
    HC(seg_sym.alloc(D));
    HC(seg_cnt.alloc(D));
    HC(seg_slot.alloc(D));
    HC(d_tkey.alloc(G));
    gid_tkey = d_tkey.p;
    hipLaunchKernelGGL(scatter_kernel, dim3((D + 255) / 256), dim3(256), 0, s, ckey.p, ccount.p, cslot.p, D, toff.p,
                       tfill.p, seg_sym.p, seg_cnt.p, seg_slot.p);
    hipLaunchKernelGGL(table_list_kernel, dim3((unsigned)((T + 255) / 256)), dim3(256), 0, s, tcount, tgid, T,
                       gid_tkey);
    HC(hipGetLastError());

    // --- 3. code books ---
    if ((rc = alloc_tables()) != MPS_OK) return rc;
    HC(cw_slot.alloc(cap));
    // Codebooks. L <= 11 (the FP8 and AWQ formats): the keys' histogram entries
    // are sorted for all keys at once, then built in LDS (launch_codebooks).
    // Longer codes (L up to 15, reachable through the op's max_len)
    // keep the work-item-per-key kernel and its global workspace.
    const bool wave_cb = L <= 11;
    DevBuf<uint64_t> keys_in, keys_sorted;
    DevBuf<uint32_t> slots_sorted, seg_beg, seg_end;
    DevBuf<char> sort_tmp;
    if (wave_cb && G) {
      HC(keys_in.alloc(D));
      HC(keys_sorted.alloc(D));
      HC(slots_sorted.alloc(D));
      HC(seg_beg.alloc(G));
      HC(seg_end.alloc(G));
      if (D)
        hipLaunchKernelGGL(item_keys_kernel, dim3((D + 255) / 256), dim3(256), 0, s, seg_sym.p, seg_cnt.p, (uint64_t)D,
                           keys_in.p);
      hipLaunchKernelGGL(segment_bounds_kernel, dim3((G + 255) / 256), dim3(256), 0, s, gid_tkey, toff.p, tcount, G,
                         seg_beg.p, seg_end.p);
      HC(hipGetLastError());
      size_t tmp_bytes = 0;
      HC(rocprim::segmented_radix_sort_pairs(nullptr, tmp_bytes, keys_in.p, keys_sorted.p, seg_slot.p, slots_sorted.p,
                                             D, G, seg_beg.p, seg_end.p, 0, 48, s));
      HC(sort_tmp.alloc(tmp_bytes));
      HC(rocprim::segmented_radix_sort_pairs(sort_tmp.p, tmp_bytes, keys_in.p, keys_sorted.p, seg_slot.p,
                                             slots_sorted.p, D, G, seg_beg.p, seg_end.p, 0, 48, s));
    }
    // per-key workspace of the work-item-per-key kernel, sized by each key's list length
    DevBuf<uint32_t> ws_sz;
    HC(ws_sz.alloc(G));
    HC(ws_off.alloc(G));
    uint32_t ws_total = 0;
    if (G && !wave_cb) {
      hipLaunchKernelGGL(ws_size_kernel, dim3((G + 255) / 256), dim3(256), 0, s, gid_tkey, tcount, G, Tsz,
                         ws_sz.p);
      HC(hipGetLastError());
      HC(device_scan(ws_sz.p, ws_off.p, G, s, &ws_total));
    }
    DevBuf<int32_t> ws;
    HC(ws.alloc(ws_total));
    cba.toff = toff.p;
    cba.seg_sym = seg_sym.p;
    cba.seg_cnt = seg_cnt.p;
    cba.seg_slot = seg_slot.p;
    cba.ws = ws.p;
    cba.ws_off = ws_off.p;
    cba.cw_slot = cw_slot.p;
    if (G && wave_cb) {
      HC(cb_lists.alloc(3 * (size_t)G));
      HC(hipMemsetAsync(flags + 5, 0, 12, s));
      hipLaunchKernelGGL(codebook_classes_kernel, dim3((G + 255) / 256), dim3(256), 0, s, gid_tkey, tcount, G, Tsz,
                         cb_lists.p, flags + 5);
      const uint32_t any[3] = {G, G, G};
      launch_codebooks(cba, keys_sorted.p, slots_sorted.p, cb_lists.p, G, flags + 5, any, s);
    } else if (G) {
      hipLaunchKernelGGL(codebook_kernel, dim3((G + 63) / 64), dim3(64), 0, s, cba);
    }
    HC(hipGetLastError());

    // --- 4. bucket tables ---
    if ((rc = bucket_tables()) != MPS_OK) return rc;

    // --- 5. bitstream ---
    OUT(startbit, uint32_t, 10, (size_t)B * (kth + 1));
    HC(hipMemsetAsync(startbit, 0, 4 * (size_t)B * (kth + 1), s));
    DevBuf<uint32_t> cw_elem, bucket_bits;
    HC(cw_elem.alloc((size_t)numel));
    HC(bucket_bits.alloc(B));
    const uint32_t lanes = lane_base[B];
    LaneArgs la;
    la.bf16 = sp.bf16;
    la.fp8 = sp.q;
    la.qmask = qmask;
    la.row_col = by_scale ? d_cols : nullptr;
    la.S = smap;
    la.m = m;
    la.row_offsets = d_row_offsets;
    la.row_indices = d_row_indices;
    la.col_start = d_cols;
    la.col_len = d_col_len;
    la.lane_base = d_lane_base;
    la.B = B;
    la.k = kth;
    la.keys = keys.p;
    la.cw_slot = cw_slot.p;
    la.cap_mask = cap - 1;
    la.cw_elem = cw_elem.p;
    la.lane_bits = startbit;
    la.err = flags + 1;
    if (lanes) hipLaunchKernelGGL(lane_bits_kernel, dim3((lanes + 255) / 256), dim3(256), 0, s, la);
    HC(hipGetLastError());
    if (B) hipLaunchKernelGGL(lane_starts_kernel, dim3(B), dim3(1024), 0, s, startbit,
                              d_lane_base, kth, bucket_bits.p);
    HC(hipGetLastError());
    std::vector<uint32_t> h_bucket_bits(B);
    if (B) HC(hipMemcpyAsync(h_bucket_bits.data(), bucket_bits.p, 4 * (size_t)B, hipMemcpyDeviceToHost, s));
    HC(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, s));
    HC(hipStreamSynchronize(s));
    if ((rc = check_errors()) != MPS_OK) return rc;
    // 64-bit aligned bucket bases (build_huffman.cu:813-818), final cursor unaligned
    std::vector<int64_t> bit_base(B + 1, 0);
    int64_t pos = 0;
    for (uint32_t b = 0; b < B; ++b) {
      if (pos & 63) pos = (pos + 63) & ~(int64_t)63;
      bit_base[b] = pos;
      pos += h_bucket_bits[b];
    }
    bit_base[B] = pos;
    W = (pos + 63) >> 6;
    OUT(d_bit_base, int64_t, 11, (size_t)B + 1);
    HC(hipMemcpyAsync(d_bit_base, bit_base.data(), 8 * (size_t)(B + 1), hipMemcpyHostToDevice, s));
    OUT(bitstream, uint64_t, 12, (size_t)W);
    if (W) HC(hipMemsetAsync(bitstream, 0, 8 * (size_t)W, s));
    PackArgs pa;
    pa.bf16 = sp.bf16;
    pa.row_col = by_scale ? d_cols : nullptr;
    pa.m = m;
    pa.row_offsets = d_row_offsets;
    pa.row_indices = d_row_indices;
    pa.col_start = d_cols;
    pa.col_len = d_col_len;
    pa.lane_base = d_lane_base;
    pa.B = B;
    pa.k = kth;
    pa.cw_elem = cw_elem.p;
    pa.startbit = startbit;
    pa.bit_base = d_bit_base;
    pa.bits = reinterpret_cast<unsigned long long *>(bitstream);
    if (lanes && W) hipLaunchKernelGGL(pack_kernel, dim3((lanes + 255) / 256), dim3(256), 0, s, pa);
    HC(hipGetLastError());
    HC(hipStreamSynchronize(s));
    return MPS_OK;
  };

  int path_rc = unit_path();
  if (path_rc == kGeneral) path_rc = general_path();
  if (path_rc != MPS_OK) return path_rc;

  // by scale, slots 5, 6 and 8 hold the group offsets, group rows and group column starts
  const int64_t sizes[17] = {(int64_t)G * Tsz, (int64_t)G * packed, G, G, B, B + 1, (int64_t)num_rows,
                             (int64_t)B * qvals, (int64_t)num_cols, by_scale ? 0 : B, (int64_t)B * (kth + 1), B + 1,
                             W, (int64_t)nshape, fp8 ? B : 0, fp8 ? (int64_t)B * 256 : 0, fp8 ? (int64_t)B * 256 : 0};
  std::memcpy(sizes17, sizes, sizeof(sizes));
  stats4[0] = hflags[2];
  stats4[1] = hflags[3];
  stats4[2] = D;
  stats4[3] = (int64_t)cap;
  return MPS_OK;
#undef OUT
#undef HC
}

// The handle's allocator: hipMalloc, outputs by slot, workspaces freed when the build ends.
void *handle_alloc(void *ctx, int32_t slot, int64_t bytes) {
  auto *sc = static_cast<mps_fp8_sidecar *>(ctx);
  void *p = nullptr;
  if (hipMalloc(&p, (size_t)bytes) != hipSuccess) return nullptr;
  if (slot >= 0) sc->out[slot] = p;
  else sc->work.push_back(p);
  return p;
}

// A builder run into a new handle.
int encode_handle(const EncodeSpec &sp, hipStream_t s, mps_fp8_sidecar **out) {
  auto sc = std::make_unique<mps_fp8_sidecar>();
  const int rc = encode_impl(sp, s, handle_alloc, sc.get(), sc->sizes, sc->stats);
  const hipError_t e = hipStreamSynchronize(s);  // before the workspaces go, also after a failure
  if (rc != MPS_OK) return rc;
  if (e != hipSuccess) return hip_fail(e, "sidecar builder");
  sc->free_work();
  *out = sc.release();
  return MPS_OK;
}

// No C++ exception (a host array too large for memory) leaves a C entry.
template <typename F>
int no_throw(F &&f) {
  try {
    return f();
  } catch (const std::exception &x) {
    return fail(MPS_ERR_NO_MEMORY, "sidecar builder: %s", x.what());
  }
}

}  // namespace
}  // namespace mps

namespace {
// The argument checks of mps_fp8_encode: the run to make, or an error.
int fp8_spec(const mps_fp8_encode_in *in, EncodeSpec *spec) {
  const int64_t L = in->max_len, kth = in->threads_per_block;
  if (L <= 0 || L > 15) return fail(MPS_ERR_INVALID_ARGUMENT, "max_len must be in [1, 15]");
  if (kth <= 0 || kth > 1024) return fail(MPS_ERR_INVALID_ARGUMENT, "threads_per_block must be in [1, 1024]");
  const int64_t numel = in->numel;
  if (in->ndim < 0 || in->ndim > 8 || in->scale_ndim < 0 || in->scale_ndim > 8)
    return fail(MPS_ERR_INVALID_ARGUMENT, "too many dimensions");
  // scale modes (build_huffman.cu:325-366)
  const int64_t scale_numel = in->scale_numel;
  const bool scale_scalar = scale_numel == 1;
  const bool scale_per_elem = scale_numel == numel;
  bool scale_per_row = false, scale_block2d = false;
  int64_t n_rows = -1, n_cols = -1, sb0 = -1, sb1 = -1, nb0 = -1, nb1 = -1;
  if (!scale_scalar && !scale_per_elem && in->ndim == 2) {
    n_rows = in->dims[0];
    n_cols = in->dims[1];
    scale_per_row = scale_numel == n_rows;
    if (!scale_per_row && in->scale_ndim == 2) {
      nb0 = in->scale_dims[0];
      nb1 = in->scale_dims[1];
      if (nb0 > 0 && nb1 > 0 && n_rows % nb0 == 0 && n_cols % nb1 == 0) {
        sb0 = n_rows / nb0;
        sb1 = n_cols / nb1;
        if (sb0 > 0 && sb1 > 0) scale_block2d = true;
      }
    }
  }
  if (!scale_scalar && !scale_per_elem && !scale_per_row && !scale_block2d)
    return fail(MPS_ERR_INVALID_ARGUMENT,
                "unsupported scales shape: use scalar, per-row (n,), per-element (numel), or 2D block-wise "
                "[n/bs0,m/bs1]");
  // The reference builds the tables before it checks the bucket layout; the
  // checks below raise the same errors without the wasted work.
  if (in->ndim != 2) return fail(MPS_ERR_INVALID_ARGUMENT, "bucket packing requires bf16_params to be 2D [n,m]");
  const int64_t n = in->dims[0], m = in->dims[1];
  if (n <= 0 || m <= 0) return fail(MPS_ERR_INVALID_ARGUMENT, "bf16_params shape must be non-empty");
  if (!scale_block2d && !(scale_scalar || (!scale_per_elem && scale_per_row)))
    return fail(MPS_ERR_INVALID_ARGUMENT,
                "bucket packing requires scales to be scalar, per-row (n,), or 2D block-wise");
  if (numel != n * m) return fail(MPS_ERR_INVALID_ARGUMENT, "bf16_params and fp8_params must have same numel");
  if (numel >= (int64_t)1 << 32) return fail(MPS_ERR_INVALID_ARGUMENT, "tensor too large for the GPU builder");
  *spec = EncodeSpec{in->bf16, in->fp8, in->scales, n, m, scale_numel, scale_scalar, scale_per_row, scale_block2d,
                     nb0, nb1, sb0, sb1, L, kth, 0, kFmtFp8};
  return MPS_OK;
}

// The argument checks of mps_awq_encode.
int awq_spec(const mps_awq_encode_in *in, EncodeSpec *spec) {
  // checks of build_huffman.cu:1097-1153 (by scale) and :1605-1650, in order
  const int64_t L = in->max_len, kth = in->threads_per_block, n = in->n, m = in->m;
  if (L <= 0 || L > 15) return fail(MPS_ERR_INVALID_ARGUMENT, "max_len must be in (0,15]");
  if (kth <= 0 || kth > 1024) return fail(MPS_ERR_INVALID_ARGUMENT, "threads_per_block must be in [1,1024]");
  if (in->by_scale && in->group_cap <= 0) return fail(MPS_ERR_INVALID_ARGUMENT, "group_cap must be > 0");
  if (n <= 0 || m <= 0) return fail(MPS_ERR_INVALID_ARGUMENT, "bf16_params shape must be non-empty");
  if (in->scale_ndim < 0 || in->scale_ndim > 2) return fail(MPS_ERR_INVALID_ARGUMENT,
      "unsupported scales_u16 shape: use scalar, per-row (n,), or 2D block-wise [n/bs0,m/bs1]");
  const int64_t scale_numel = in->scale_numel;
  const bool scalar = scale_numel == 1;
  const bool per_row = !scalar && in->scale_ndim == 1 && scale_numel == n;
  bool block2d = false;
  int64_t nb0 = -1, nb1 = -1, sb0 = -1, sb1 = -1;
  if (!scalar && !per_row && in->scale_ndim == 2) {
    nb0 = in->scale_dims[0];
    nb1 = in->scale_dims[1];
    if (nb0 > 0 && nb1 > 0 && n % nb0 == 0 && m % nb1 == 0) {
      sb0 = n / nb0;
      sb1 = m / nb1;
      block2d = sb0 > 0 && sb1 > 0;
    }
  }
  if (!scalar && !per_row && !block2d)
    return fail(MPS_ERR_INVALID_ARGUMENT,
                "unsupported scales_u16 shape: use scalar, per-row (n,), or 2D block-wise [n/bs0,m/bs1]");
  if (n * m >= (int64_t)1 << 32) return fail(MPS_ERR_INVALID_ARGUMENT, "tensor too large for the GPU builder");
  if (in->by_scale && n * (block2d ? nb1 : 1) >= (int64_t)1 << 31)
    return fail(MPS_ERR_INVALID_ARGUMENT, "too many quantisation groups for the GPU builder");
  *spec = EncodeSpec{in->bf16, in->int4, in->scales, n, m, scale_numel, scalar, per_row, block2d, nb0, nb1, sb0, sb1,
                     L, kth, in->group_cap, in->by_scale ? kFmtAwqByScale : kFmtAwqBucket};
  return MPS_OK;
}

template <typename In>
int to_handle(const In *in, int (*make)(const In *, EncodeSpec *), void *stream, mps_fp8_sidecar **out) {
  last_error().clear();
  if (!in || !out) return fail(MPS_ERR_INVALID_ARGUMENT, "inputs must be defined");
  *out = nullptr;
  EncodeSpec sp;
  const int rc = make(in, &sp);
  return rc != MPS_OK ? rc : no_throw([&] { return encode_handle(sp, reinterpret_cast<hipStream_t>(stream), out); });
}

template <typename In>
int to_alloc(const In *in, int (*make)(const In *, EncodeSpec *), void *stream, mps_encode_alloc alloc, void *ctx,
             int64_t *sizes17, int64_t *stats4) {
  last_error().clear();
  if (!in || !alloc || !sizes17 || !stats4) return fail(MPS_ERR_INVALID_ARGUMENT, "inputs must be defined");
  EncodeSpec sp;
  int rc = make(in, &sp);
  if (rc != MPS_OK) return rc;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  rc = no_throw([&] { return encode_impl(sp, s, alloc, ctx, sizes17, stats4); });
  // After a failure nothing runs on: the caller frees what it gave, and its inputs.
  if (rc != MPS_OK) (void)hipStreamSynchronize(s);
  return rc;
}
}  // namespace

extern "C" {

int mps_fp8_encode(const mps_fp8_encode_in *in, void *stream, mps_fp8_sidecar **out) {
  return to_handle(in, fp8_spec, stream, out);
}

int mps_awq_encode(const mps_awq_encode_in *in, void *stream, mps_fp8_sidecar **out) {
  return to_handle(in, awq_spec, stream, out);
}

int mps_fp8_encode_alloc(const mps_fp8_encode_in *in, void *stream, mps_encode_alloc alloc, void *ctx,
                         int64_t *sizes17, int64_t *stats4) {
  return to_alloc(in, fp8_spec, stream, alloc, ctx, sizes17, stats4);
}

int mps_awq_encode_alloc(const mps_awq_encode_in *in, void *stream, mps_encode_alloc alloc, void *ctx,
                         int64_t *sizes17, int64_t *stats4) {
  return to_alloc(in, awq_spec, stream, alloc, ctx, sizes17, stats4);
}

int mps_fp8_sidecar_sizes(const mps_fp8_sidecar *sc, int64_t *sizes17) {
  if (!sc || !sizes17) return fail(MPS_ERR_INVALID_ARGUMENT, "NULL argument");
  std::memcpy(sizes17, sc->sizes, sizeof(sc->sizes));
  return MPS_OK;
}

int mps_fp8_sidecar_stats(const mps_fp8_sidecar *sc, int64_t *stats4) {
  if (!sc || !stats4) return fail(MPS_ERR_INVALID_ARGUMENT, "NULL argument");
  std::memcpy(stats4, sc->stats, sizeof(sc->stats));
  return MPS_OK;
}

int mps_fp8_sidecar_copy(const mps_fp8_sidecar *sc, void *const *dst17, void *stream) {
  last_error().clear();
  if (!sc || !dst17) return fail(MPS_ERR_INVALID_ARGUMENT, "NULL argument");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  for (int i = 0; i < 17; ++i) {
    const size_t bytes = (size_t)sc->sizes[i] * kOutBytes[i];
    if (bytes == 0) continue;
    if (!dst17[i]) return fail(MPS_ERR_INVALID_ARGUMENT, "NULL destination %d", i);
    MPS_HIP_CHECK(hipMemcpyAsync(dst17[i], sc->out[i], bytes, hipMemcpyDefault, s));
  }
  MPS_HIP_CHECK(hipStreamSynchronize(s));
  return MPS_OK;
}

int mps_fp8_sidecar_free(mps_fp8_sidecar *sc) {
  delete sc;
  return MPS_OK;
}

}  // extern "C"
