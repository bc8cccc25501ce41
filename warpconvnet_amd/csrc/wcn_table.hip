// Coordinate table of 4x4x4-voxel blocks: build and point queries (gfx950).
//
// Build pipeline (all on the caller's stream, no host round trip).  The keys are grouped by bins of one to two thousand (a bin is
// a hash of the key's 16x16x16-voxel cell, so every 4x4x4 block lies in exactly one bin); one workgroup per bin then sees all
// voxels of its blocks and builds their masks with LDS atomics:
//   table_sort     per part of the keys (a workgroup): the part's keys in the order of their bins, where each bin begins among them, and
//                  the part's bounding box
//   table_bins     per bin: its stretches of all parts, the box and the keys of the bins before; block masks and entry counts in
//                  an LDS table, their prefix sums; that table is the bin's region of the table in memory; then per key: its
//                  place in block order and perm[base + rank] = row
// Up to 16,384 keys one launch does all of it (table_small).
//
// HBM traffic per key: 16 B read (12 where the keys are made here, and 16 written), 20 B written and read (grouped entry), 8 B written
// (entry in block order) + 4 B (perm), plus 16 B per table slot.
// What it took over 1 M voxels of rooms, us: with bins laid out one behind the other (a launch for the parts' counts per bin 10.5, one for
// their sums 4.9, the scatter 21.2, table_bins over contiguous entries 26) 62.6; as it is, 14.6 + 32.4, of which the stretches of
// eight keys in 245 parts are 6.  456,000: 38.1 -> 30.2; 60,000 and 24,000 voxels of a network's levels 48.2 -> 40.6 together.  The regions written
// whole against slots of 32 bytes anywhere in the table, cleared by the first launch and claimed with a 64-bit compare-and-swap per block:
// the probe passes of a 3x3x3 map 86 -> 59 and of a 5x5x5 map 189 -> 140; 1,800 voxels: 14.4 in two launches -> 10.2 in one.
#include <stdlib.h>
#include <string.h>

#include <chrono>
#include <mutex>
#include <thread>
#include <type_traits>
#include <vector>

#include <algorithm>

#include "wcn_common.h"

namespace {

// Bin of a key (wcn_cell_* in wcn_common.h).
__device__ __forceinline__ uint32_t bin_of(const int4 c, uint32_t bin_mask) {
  return wcn_cell_hash(wcn_cell_batch((uint32_t)c.x) + wcn_cell_x(c.y >> 2) + wcn_cell_y(c.z >> 2) + wcn_cell_z(c.w >> 2)) & bin_mask;
}

struct PartRange {
  int64_t lo, hi;
};
__device__ __forceinline__ PartRange part_range(int64_t n_keys, int part) {
  const int64_t chunk = (n_keys + gridDim.x - 1) / gridDim.x;
  PartRange r;
  r.lo = (int64_t)part * chunk;
  r.hi = r.lo + chunk < n_keys ? r.lo + chunk : n_keys;
  return r;
}

// Bins: capacity / 2048, at most WCN_MAX_BINS.  The sort keeps one counter per bin in LDS (dynamic: 4 bytes per bin, 128 KB at the
// most), and a thread of it adds up BPT of them: 4 up to 4096 bins, 32 beyond.
constexpr int SMALL_BINS = 4096;

// The keys of one part in the order of their bins, within the part's own stretch of memory; where each bin begins there, and the
// part's bounding box.  A part of up to 4,096 keys (up to a million altogether) is read once.  What its workgroup writes lies in 80 KB,
// in whole lines.
// ITEMS: the keys are made here too, [batch item, x, y, z] of three columns, and written on the way.
struct KeysOfItems {
  const int32_t* coords;  // (n, 3)
  int4* rows;
  WcnItemStarts starts;
  int32_t batch_size;
};

template <int BPT, bool ITEMS>
__global__ void __launch_bounds__(1024) table_sort(const int4* __restrict__ keys, int64_t n_keys, int32_t bins,
                                                   int32_t* __restrict__ part_start, int32_t* __restrict__ part_box,
                                                   int4* __restrict__ bin_coords, int32_t* __restrict__ bin_row, KeysOfItems of) {
  extern __shared__ __attribute__((aligned(16))) int s_cur[];  // [bins], then (BPT 4) the part's keys and their numbers in it
  __shared__ int64_t s_start[ITEMS ? WCN_VOXEL_MAX_BATCH + 1 : 1];
  __shared__ int s_mn[16][4], s_mx[16][4], s_wave[16];
  const int tid = threadIdx.x, lane = wcn_lane(), wave = tid >> 6;
  const int parts = gridDim.x, part = wcn_xcd_tile((int)blockIdx.x, parts);
  const PartRange r = part_range(n_keys, part);
  const uint32_t bin_mask = (uint32_t)bins - 1u;
  if (ITEMS && tid <= WCN_VOXEL_MAX_BATCH) s_start[tid] = of.starts.start[tid];
  for (int b = tid; b < bins; b += 1024) s_cur[b] = 0;
  __syncthreads();
  constexpr int PER = 4;  // keys a thread has in flight together
  auto load = [&](int64_t i) {
    return ITEMS ? make_int4(0, of.coords[3 * i], of.coords[3 * i + 1], of.coords[3 * i + 2]) : keys[i];
  };
  const bool kept = r.hi - r.lo <= 1024 * PER;  // a thread's keys stay in registers
  int4 c[PER];
  int rank[PER] = {};
  int mn[4] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MAX};
  int mx[4] = {INT32_MIN, INT32_MIN, INT32_MIN, INT32_MIN};
  for (int64_t i0 = r.lo + tid; i0 < r.hi; i0 += 1024 * PER) {
#pragma unroll
    for (int t = 0; t < PER; ++t) c[t] = load(i0 + t * 1024 < r.hi ? i0 + t * 1024 : i0);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      if (ITEMS) {
        const int64_t i = i0 + t * 1024 < r.hi ? i0 + t * 1024 : i0;
        c[t].x = wcn_item_of(s_start, of.batch_size, i);
        of.rows[i] = c[t];
      }
      if (i0 + t * 1024 < r.hi) rank[t] = atomicAdd(&s_cur[bin_of(c[t], bin_mask)], 1);
      mn[0] = min(mn[0], c[t].x); mx[0] = max(mx[0], c[t].x);
      mn[1] = min(mn[1], c[t].y); mx[1] = max(mx[1], c[t].y);
      mn[2] = min(mn[2], c[t].z); mx[2] = max(mx[2], c[t].z);
      mn[3] = min(mn[3], c[t].w); mx[3] = max(mx[3], c[t].w);
    }
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
      mn[d] = min(mn[d], __shfl_xor(mn[d], s, 64));
      mx[d] = max(mx[d], __shfl_xor(mx[d], s, 64));
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      s_mn[wave][d] = mn[d];
      s_mx[wave][d] = mx[d];
    }
  }
  __syncthreads();
  int v[BPT], sum = 0;
#pragma unroll
  for (int t = 0; t < BPT; ++t) {
    v[t] = tid * BPT + t < bins ? s_cur[tid * BPT + t] : 0;
    sum += v[t];
  }
  const int incl = wcn_wave_inclusive_sum(sum);
  if (lane == 63) s_wave[wave] = incl;
  if (tid < 4) {
    int a = s_mn[0][tid], b = s_mx[0][tid];
    for (int w = 1; w < 16; ++w) {
      a = min(a, s_mn[w][tid]);
      b = max(b, s_mx[w][tid]);
    }
    part_box[part * 8 + tid] = a;
    part_box[part * 8 + 4 + tid] = b;
  }
  __syncthreads();
  int run = incl - sum;
  for (int w = 0; w < wave; ++w) run += s_wave[w];
#pragma unroll
  for (int t = 0; t < BPT; ++t) {
    const int b = tid * BPT + t;
    if (b < bins) {
      s_cur[b] = run;
      part_start[(int64_t)b * parts + part] = run;
    }
    run += v[t];
  }
  if (tid == 0) part_start[(int64_t)bins * parts + part] = r.hi > r.lo ? (int32_t)(r.hi - r.lo) : 0;
  __syncthreads();
  auto put = [&](int64_t i, const int4 key, int at) {
    bin_coords[r.lo + at] = key;
    bin_row[r.lo + at] = (int32_t)i;
  };
  if (kept) {
    // through LDS, for whole lines: written one by one a part's keys are as many requests (1 M voxels 19.8 us, 14.6 so)
    int4* const s_key = reinterpret_cast<int4*>(s_cur + bins);
    uint16_t* const s_row = reinterpret_cast<uint16_t*>(s_key + 1024 * PER);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      if (r.lo + tid + t * 1024 >= r.hi) continue;
      const int at = s_cur[bin_of(c[t], bin_mask)] + rank[t];
      if (BPT == 4) {
        s_key[at] = c[t];
        s_row[at] = (uint16_t)(tid + t * 1024);
      } else {
        put(r.lo + tid + t * 1024, c[t], at);
      }
    }
    if (BPT != 4) return;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < PER; ++t)
      if (r.lo + tid + t * 1024 < r.hi) put(r.lo + s_row[tid + t * 1024], s_key[tid + t * 1024], tid + t * 1024);
    return;
  }
  for (int64_t i0 = r.lo + tid; i0 < r.hi; i0 += 1024 * PER) {
#pragma unroll
    for (int t = 0; t < PER; ++t) c[t] = load(i0 + t * 1024 < r.hi ? i0 + t * 1024 : i0);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      const int64_t i = i0 + t * 1024;
      if (i >= r.hi) continue;
      if (ITEMS) c[t].x = wcn_item_of(s_start, of.batch_size, i);
      put(i, c[t], atomicAdd(&s_cur[bin_of(c[t], bin_mask)], 1));
    }
  }
}

// One workgroup per bin.  LDS holds an open-addressing table of the bin's blocks: key, occupancy
// mask, number of entries (keys, duplicates included), later their prefix sums.
struct BinLds {
  unsigned long long key[WCN_BIN_SLOTS];
  unsigned long long mask[WCN_BIN_SLOTS];
  uint32_t cursor[WCN_BIN_SLOTS];   // entries of the block, then the next free place among them
  uint32_t base[WCN_BIN_SLOTS];     // voxels of the blocks before this one
  int32_t low[WCN_BIN_SLOTS];       // lowest row per voxel when keys repeat
  int32_t index[WCN_BIN_SLOTS];     // the block's number in the bin's block list
  int32_t part[3][16];
  uint32_t passed[WCN_BIN_SLOTS / 32];  // slots that the search for a block that is there has gone on from
  int32_t lost;                     // a block has found no place
};

// A key of the bin: claims / finds its block in the LDS table, sets its bit, counts itself.  The search goes as a look-up's
// will.  Returns the block's place, or -1 if the table is full.
__device__ __forceinline__ int bin_insert(BinLds* s, unsigned long long key, uint32_t home, uint32_t bit) {
  for (int p = 0; p <= WCN_BIN_SLOTS; ++p) {
    const uint32_t h = wcn_probe_slot(home, p);
    unsigned long long seen = s->key[h];
    if (seen == WCN_EMPTY_KEY) {
      seen = atomicCAS(&s->key[h], WCN_EMPTY_KEY, key);
      if (seen == WCN_EMPTY_KEY) {
        seen = key;
        for (int q = 0; q < p; ++q) {
          const uint32_t on = wcn_probe_slot(home, q);
          atomicOr(&s->passed[on >> 5], 1u << (on & 31u));
        }
      }
    }
    if (seen == key) {
      atomicOr(&s->mask[h], 1ull << bit);
      atomicAdd(&s->cursor[h], 1u);
      return (int)h;
    }
  }
  return -1;
}
__device__ __forceinline__ int bin_find(const BinLds* s, unsigned long long key, uint32_t home) {
  for (int p = 0; p <= WCN_BIN_SLOTS; ++p) {
    const uint32_t h = wcn_probe_slot(home, p);
    if (s->key[h] == key) return (int)h;
  }
  return -1;
}
// Where the block of a key is looked for in its bin's region.
__device__ __forceinline__ uint32_t home_in_bin(const int4 c) { return wcn_home_slot_of(c.x, c.y >> 2, c.z >> 2, c.w >> 2, 0u); }

// Where a bin's entries [lo, hi) come from: at(e) is what coords() and row() are asked with.
constexpr int MAX_PARTS = 256;
struct PartedEntries {  // as table_sort left them, a stretch in every part
  const int4* __restrict__ keys;
  const int32_t* __restrict__ rows;
  const int32_t* first;  // [MAX_PARTS] LDS: entries of the bin in the parts before; INT32_MAX past the last part
  const int32_t* shift;  // [MAX_PARTS] LDS: where the part's first lies, less that
  int lo;
  template <int N>
  __device__ __forceinline__ void at(int (&e)[N]) const {  // N searches abreast
    int part[N];
#pragma unroll
    for (int t = 0; t < N; ++t) part[t] = 0;
#pragma nounroll
    for (int step = MAX_PARTS / 2; step >= 1; step >>= 1) {
#pragma unroll
      for (int t = 0; t < N; ++t) part[t] += first[part[t] + step] <= e[t] - lo ? step : 0;
    }
#pragma unroll
    for (int t = 0; t < N; ++t) e[t] += shift[part[t]] - lo;
  }
  __device__ __forceinline__ int at(int e) const {
    int one[1] = {e};
    at(one);
    return one[0];
  }
  __device__ __forceinline__ int4 coords(int i) const { return keys[i]; }
  __device__ __forceinline__ int32_t row(int i) const { return rows[i]; }
};
template <class Keys>
struct ListedEntries {  // the rows of a few keys, listed in LDS
  Keys keys;
  const uint16_t* list;
  int lo;
  template <int N>
  __device__ __forceinline__ void at(int (&e)[N]) const {
#pragma unroll
    for (int t = 0; t < N; ++t) e[t] = list[e[t] - lo];
  }
  __device__ __forceinline__ int at(int e) const { return list[e - lo]; }
  __device__ __forceinline__ int4 coords(int i) const { return keys(i); }
  __device__ __forceinline__ int32_t row(int i) const { return i; }
};

// The layout of a box in LDS, in scalar registers.
__device__ __forceinline__ WcnLayout layout_of(const WcnTableHeader& box) {
  WcnTableHeader h;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    h.mn[d] = __builtin_amdgcn_readfirstlane(box.mn[d]);
    h.mx[d] = __builtin_amdgcn_readfirstlane(box.mx[d]);
  }
  return wcn_make_layout(&h);
}

template <bool WANT_SLOT_OF, int E, class Entries>
__device__ __forceinline__ void build_bin(const Entries& in, int bin, int lo, int hi, const WcnLayout& L, BinLds* s,
                                          WcnSlot* __restrict__ slots, unsigned long long* __restrict__ wide_keys,
                                          int32_t* __restrict__ order_tag,
                                          int32_t* __restrict__ order_row, WcnBlock* __restrict__ block_list,
                                          int32_t* __restrict__ perm, int32_t* __restrict__ slot_of,
                                          int32_t* __restrict__ bin_stats) {
  const int tid = threadIdx.x, lane = wcn_lane(), wave = tid >> 6;
  uint4* const region = reinterpret_cast<uint4*>(slots + (size_t)bin * WCN_BIN_SLOTS);
  if (lo >= hi) {
    if (tid == 0) bin_stats[2 * bin] = bin_stats[2 * bin + 1] = 0;
    for (int h = tid; h < WCN_BIN_SLOTS; h += 1024) region[h] = make_uint4(WCN_EMPTY_TAG, 0u, 0u, 0u);
    return;
  }
  // A thread keeps its first E entries in registers from the first pass to the last (bins hold
  // one to two thousand keys: one or two entries per thread); entries beyond that are read again.
  int4 c[E];
  int32_t row[E];
  int where[E];  // place of the key's block << 6 | voxel bit, or -1
#pragma unroll
  for (int t = 0; t < E; ++t) where[t] = lo + tid + t * 1024 < hi ? lo + tid + t * 1024 : lo;
  in.at(where);
#pragma unroll
  for (int t = 0; t < E; ++t) {
    row[t] = in.row(where[t]);
    c[t] = in.coords(where[t]);
  }
  if (!L.ok) {
    if (tid == 0) bin_stats[2 * bin] = bin_stats[2 * bin + 1] = 0;
#pragma nounroll
    for (int e = lo + tid; e < hi; e += 1024) {
      const int32_t rw = in.row(in.at(e));
      if (WANT_SLOT_OF) slot_of[rw] = -1;
      order_row[e] = rw;
      order_tag[e] = 0;
    }
    return;
  }
  for (int h = tid; h < WCN_BIN_SLOTS; h += 1024) {
    s->key[h] = WCN_EMPTY_KEY;
    s->mask[h] = 0ull;
    s->cursor[h] = 0u;
  }
  if (tid < WCN_BIN_SLOTS / 32) s->passed[tid] = 0u;
  if (tid == 0) s->lost = 0;
  __syncthreads();
  // masks and entry counts
  bool lost = false;
#pragma unroll
  for (int t = 0; t < E; ++t) {
    where[t] = -1;
    if (lo + tid + t * 1024 < hi) {
      uint32_t r[4];
      wcn_relative(L, c[t].x, c[t].y, c[t].z, c[t].w, r);  // always inside: the box was built from these keys
      const int h = bin_insert(s, wcn_block_key(L, r), home_in_bin(c[t]), wcn_block_bit(r));
      lost |= h < 0;
      where[t] = h < 0 ? -1 : h << 6 | (int)wcn_block_bit(r);
    }
  }
#pragma nounroll
  for (int e = lo + tid + E * 1024; e < hi; e += 1024) {
    const int4 ce = in.coords(in.at(e));
    uint32_t r[4];
    wcn_relative(L, ce.x, ce.y, ce.z, ce.w, r);
    lost |= bin_insert(s, wcn_block_key(L, r), home_in_bin(ce), wcn_block_bit(r)) < 0;
  }
  if (lost) s->lost = 1;  // more distinct blocks in this bin than its table holds
  __syncthreads();
  // Prefix sums over the table's slots, entries and voxels.  Thread t owns slots t, t + 1024, ...
  // and counts them as neighbours in the order of the sums (any fixed order will do, and this one
  // reads LDS without bank conflicts and spreads the occupied slots over the threads).
  constexpr int PER = WCN_BIN_SLOTS / 1024;
  uint32_t ne[PER], nv[PER], se = 0, sv = 0, sb = 0;
  unsigned long long bkey[PER], bmask[PER];
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int h = tid + t * 1024;
    bkey[t] = s->key[h];
    bmask[t] = s->mask[h];
    ne[t] = s->cursor[h];
    nv[t] = (uint32_t)__popcll(bmask[t]);
    se += ne[t];
    sv += nv[t];
    sb += bkey[t] != WCN_EMPTY_KEY ? 1u : 0u;
  }
  const int ie = wcn_wave_inclusive_sum((int)se), iv = wcn_wave_inclusive_sum((int)sv);
  const int ib = wcn_wave_inclusive_sum((int)sb);
  if (lane == 63) {
    s->part[0][wave] = ie;
    s->part[1][wave] = iv;
    s->part[2][wave] = ib;
  }
  __syncthreads();
  int be = 0, bv = 0, bb = 0, total_v = 0, total_b = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) {
      be += s->part[0][w];
      bv += s->part[1][w];
      bb += s->part[2][w];
    }
    total_v += s->part[1][w];
    total_b += s->part[2][w];
  }
  const bool repeats = total_v != hi - lo;          // some key of this bin came more than once
  const bool low_in_lds = total_v <= WCN_BIN_SLOTS;  // room for one word per voxel
  uint32_t re = (uint32_t)(be + ie) - se, rv = (uint32_t)(bv + iv) - sv;
  int rb = bb + ib - (int)sb;
  // The LDS table's places are the region's slots.
#pragma unroll
  for (int t = 0; t < PER; ++t) {
    const int h = tid + t * 1024;
    s->cursor[h] = re;
    s->base[h] = rv;
    const bool there = bkey[t] != WCN_EMPTY_KEY;
    region[h] = there ? make_uint4(wcn_block_tag(L, bkey[t]), (uint32_t)(lo + (int32_t)rv) | (s->passed[h >> 5] >> (h & 31)) << 31, (uint32_t)bmask[t],
                                    (uint32_t)(bmask[t] >> 32))
                      : make_uint4(WCN_EMPTY_TAG, 0u, 0u, 0u);
    if (there) {
      if (L.wide) wide_keys[(size_t)bin * WCN_BIN_SLOTS + h] = bkey[t];
      // the block's line of the bin's block list (two 16-byte stores)
      uint4* line = reinterpret_cast<uint4*>(&block_list[lo + rb]);
      line[0] = make_uint4((uint32_t)bkey[t], (uint32_t)(bkey[t] >> 32), (uint32_t)bmask[t], (uint32_t)(bmask[t] >> 32));
      line[1] = make_uint4((uint32_t)(lo + (int32_t)rv), re, 0u, 0u);
      s->index[h] = rb;
      ++rb;
    }
    re += ne[t];
    rv += nv[t];
  }
  if (repeats) {
    if (low_in_lds) {
      for (int j = tid; j < total_v; j += 1024) s->low[j] = INT32_MAX;
    } else {
      for (int j = lo + tid; j < lo + total_v; j += 1024) perm[j] = INT32_MAX;
      __threadfence();
    }
  }
  __syncthreads();
  // every key to its place in block order; the row of every voxel into perm
  auto place = [&](int32_t rw, int where, int e) {
    if (where < 0) {  // its block did not fit (overflow is flagged): the entry stays where it is
      order_tag[e] = 0;
      order_row[e] = rw;
      if (WANT_SLOT_OF) slot_of[rw] = -1;
      return;
    }
    const int h = where >> 6;
    const uint32_t bit = (uint32_t)where & 63u;
    if (WANT_SLOT_OF) slot_of[rw] = bin * WCN_BIN_SLOTS + h;
    const int v = (int)s->base[h] + wcn_rank_below(s->mask[h], bit);
    // without repeated keys the entries of a block are its voxels: block order is perm's order
    const int q = lo + (repeats ? (int)atomicAdd(&s->cursor[h], 1u) : v);
    order_tag[q] = (s->index[h] << 6) | (int32_t)bit;
    order_row[q] = rw;
    if (!repeats) perm[lo + v] = rw;
    else if (low_in_lds) atomicMin(&s->low[v], rw);
    else atomicMin(&perm[lo + v], rw);
  };
#pragma unroll
  for (int t = 0; t < E; ++t) {
    const int e = lo + tid + t * 1024;
    if (e < hi) place(row[t], where[t], e);
  }
#pragma nounroll
  for (int e = lo + tid + E * 1024; e < hi; e += 1024) {
    const int i = in.at(e);
    const int4 ce = in.coords(i);
    uint32_t r[4];
    wcn_relative(L, ce.x, ce.y, ce.z, ce.w, r);
    const int h = bin_find(s, wcn_block_key(L, r), home_in_bin(ce));
    place(in.row(i), h < 0 ? -1 : h << 6 | (int)wcn_block_bit(r), e);
  }
  __syncthreads();
  if (repeats && low_in_lds)
    for (int j = tid; j < total_v; j += 1024) perm[lo + j] = s->low[j];
  if (tid == 0) {
    bin_stats[2 * bin] = total_v;
    bin_stats[2 * bin + 1] = total_b | (s->lost ? WCN_BIN_LOST : 0);
  }
}

struct BinsLds {
  BinLds bin;
  WcnTableHeader box;
  int32_t first[MAX_PARTS], shift[MAX_PARTS];
  int32_t wave[2][4], part[16][8];
};

// A bin's keys in front of it, its own and where they lie follow from two rows of the parts' starts (the keys of a part in the bins
// before are its start), the box from the parts' boxes: every workgroup finds both, and no launch stands between the sort and this one.
template <bool WANT_SLOT_OF, bool TWO>
__global__ void __launch_bounds__(1024, TWO ? 8 : 4) table_bins(WcnTableHeader* __restrict__ hdr, int64_t n_keys, int64_t stats_offset,
                                                   WcnSlot* __restrict__ slots, unsigned long long* __restrict__ wide_keys,
                                                   const int32_t* __restrict__ part_start, const int32_t* __restrict__ part_box,
                                                   int32_t parts, int32_t* __restrict__ bin_start,
                                                   const int4* __restrict__ bin_coords,
                                                   const int32_t* __restrict__ bin_row,
                                                   int32_t* __restrict__ order_tag,
                                                   int32_t* __restrict__ order_row,
                                                   WcnBlock* __restrict__ block_list,
                                                   int32_t* __restrict__ perm,
                                                   int32_t* __restrict__ slot_of,
                                                   int32_t* __restrict__ bin_stats) {
  extern __shared__ __attribute__((aligned(16))) unsigned char bin_smem[];
  BinsLds* const s = reinterpret_cast<BinsLds*>(bin_smem);
  const int tid = threadIdx.x, lane = wcn_lane(), wave = tid >> 6, bin = (int)blockIdx.x;
  int before = 0, n = 0, incl = 0;
  if (tid < MAX_PARTS) {  // a thread per part
    const int32_t* const at = part_start + (int64_t)bin * parts + (tid < parts ? tid : 0);
    before = tid < parts ? at[0] : 0;
    n = tid < parts ? at[parts] - before : 0;
  }
  // (columns of the boxes lane & 7: the values of a thread are of one column)
  const int column = lane & 7;
  int v = column < 4 ? INT32_MAX : INT32_MIN;
#pragma unroll
  for (int t = 0; t < MAX_PARTS * 8 / 1024; ++t) {
    const int i = tid + t * 1024, x = part_box[i < parts * 8 ? i : column];
    v = column < 4 ? min(v, x) : max(v, x);
  }
#pragma unroll
  for (int d = 8; d < 64; d <<= 1) {
    const int o = __shfl_xor(v, d, 64);
    v = column < 4 ? min(v, o) : max(v, o);
  }
  if (lane < 8) s->part[wave][lane] = v;
  if (tid < MAX_PARTS) {
    incl = wcn_wave_inclusive_sum(n);
    const int all_before = wcn_wave_inclusive_sum(before);
    if (lane == 63) {
      s->wave[0][wave] = incl;
      s->wave[1][wave] = all_before;
    }
  }
  __syncthreads();
  if (tid < 8) {
    int a = s->part[0][tid];
    for (int w = 1; w < 16; ++w) a = tid < 4 ? min(a, s->part[w][tid]) : max(a, s->part[w][tid]);
    *(tid < 4 ? &s->box.mn[tid] : &s->box.mx[tid - 4]) = a;
    if (bin == 0) *(tid < 4 ? &hdr->mn[tid] : &hdr->mx[tid - 4]) = a;
  }
  if (tid < MAX_PARTS) {
    int first = incl - n;
    for (int w = 0; w < wave; ++w) first += s->wave[0][w];
    const int64_t chunk = (n_keys + parts - 1) / parts;
    s->first[tid] = tid < parts ? first : INT32_MAX;
    s->shift[tid] = tid < parts ? (int32_t)(tid * chunk) + before - first : 0;
  }
  const int lo = __builtin_amdgcn_readfirstlane(s->wave[1][0] + s->wave[1][1] + s->wave[1][2] + s->wave[1][3]);
  const int hi = __builtin_amdgcn_readfirstlane(lo + s->wave[0][0] + s->wave[0][1] + s->wave[0][2] + s->wave[0][3]);
  if (tid == 0) {
    bin_start[bin] = lo;
    if (bin == (int)gridDim.x - 1) bin_start[bin + 1] = (int32_t)n_keys;
    if (bin == 0) {
      hdr->num_keys = (int32_t)n_keys;
      hdr->bins = (int32_t)gridDim.x;
      hdr->stats_offset = stats_offset;
    }
  }
  __syncthreads();
  const PartedEntries in{bin_coords, bin_row, s->first, s->shift, lo};
  build_bin<WANT_SLOT_OF, TWO ? 2 : 4>(in, bin, lo, hi, layout_of(s->box), &s->bin, slots, wide_keys, order_tag, order_row,
                          block_list, perm, slot_of, bin_stats);
}

// ---- few keys -----------------------------------------------------------------------------------
// Of few keys the two launches above are mostly start, end and the wait between them.  Up to SMALL_KEYS keys one launch does both:
// every workgroup reads all of them (a quarter of a megabyte at the most, out of its die's L2), finds the box, lists the rows of its
// own bin and counts those of the bins before it.  What each reads grows with the keys, and the list takes LDS.  us of a build,
// spheres, two launches / one:
//     keys        500         2,000        8,000        12,000       16,384       20,000       24,000       30,000
//             14.0 /  9.1  14.7 / 10.1  15.6 / 11.9  15.9 / 13.4  16.9 / 15.4  17.8 / 17.1  18.6 / 18.9  19.7 / 22.7
constexpr int64_t SMALL_KEYS = 16384;
constexpr int SMALL_KEY_BINS = 64;  // more bins (a table that was grown) would read the keys too often

struct SmallLds {
  BinLds bin;
  uint16_t list[SMALL_KEYS];
  WcnTableHeader box;
  int64_t item_start[WCN_VOXEL_MAX_BATCH + 1];
  int part[16][10];  // per wave: least and greatest value of every column, keys of earlier bins
  int listed;
};

struct KeyRows {
  const int4* __restrict__ keys;
  __device__ __forceinline__ int4 operator()(int i) const { return keys[i]; }
};
struct KeyItems {  // made here, as in table_sort
  const int32_t* __restrict__ coords;
  const int64_t* start;
  int32_t batch_size;
  __device__ __forceinline__ int4 operator()(int i) const {
    return make_int4(wcn_item_of(start, batch_size, i), coords[3 * i], coords[3 * i + 1], coords[3 * i + 2]);
  }
};

template <bool WANT_SLOT_OF, bool ITEMS>
__global__ void __launch_bounds__(1024) table_small(const int4* __restrict__ rows, KeysOfItems of, int32_t n_keys, int32_t bins,
                                                    WcnTableHeader* __restrict__ hdr, int64_t stats_offset,
                                                    WcnSlot* __restrict__ slots, unsigned long long* __restrict__ wide_keys,
                                                    int32_t* __restrict__ bin_start,
                                                    int32_t* __restrict__ order_tag, int32_t* __restrict__ order_row,
                                                    WcnBlock* __restrict__ block_list, int32_t* __restrict__ perm,
                                                    int32_t* __restrict__ slot_of, int32_t* __restrict__ bin_stats) {
  extern __shared__ __attribute__((aligned(16))) unsigned char bin_smem[];
  SmallLds* s = reinterpret_cast<SmallLds*>(bin_smem);
  const int tid = threadIdx.x, lane = wcn_lane(), wave = tid >> 6, bin = (int)blockIdx.x;
  const uint32_t bin_mask = (uint32_t)bins - 1u;
  typedef typename std::conditional<ITEMS, KeyItems, KeyRows>::type Keys;
  Keys keys;
  if constexpr (ITEMS) {
    if (tid <= WCN_VOXEL_MAX_BATCH) s->item_start[tid] = of.starts.start[tid];
    keys = Keys{of.coords, s->item_start, of.batch_size};
  } else {
    keys = Keys{rows};
  }
  if (tid == 0) s->listed = 0;
  __syncthreads();
  int v[9] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN, INT32_MIN, 0};
  constexpr int PER = 4;
  for (int i0 = tid; i0 < n_keys; i0 += 1024 * PER) {
    int4 c[PER];
#pragma unroll
    for (int t = 0; t < PER; ++t) c[t] = keys(i0 + t * 1024 < n_keys ? i0 + t * 1024 : i0);
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      const int i = i0 + t * 1024;
      v[0] = min(v[0], c[t].x); v[4] = max(v[4], c[t].x);
      v[1] = min(v[1], c[t].y); v[5] = max(v[5], c[t].y);
      v[2] = min(v[2], c[t].z); v[6] = max(v[6], c[t].z);
      v[3] = min(v[3], c[t].w); v[7] = max(v[7], c[t].w);
      const int b = (int)bin_of(c[t], bin_mask);
      const bool live = i < n_keys;
      if (ITEMS && live && ((uint32_t)i >> 10 & bin_mask) == (uint32_t)bin) of.rows[i] = c[t];
      v[8] += live && b < bin ? 1 : 0;
      if (live && b == bin) s->list[atomicAdd(&s->listed, 1)] = (uint16_t)i;
    }
  }
#pragma unroll
  for (int d = 0; d < 9; ++d) {
#pragma unroll
    for (int x = 32; x > 0; x >>= 1) {
      const int o = __shfl_xor(v[d], x, 64);
      v[d] = d < 4 ? min(v[d], o) : d < 8 ? max(v[d], o) : v[d] + o;
    }
    if (lane == 0) s->part[wave][d] = v[d];
  }
  __syncthreads();
  if (tid < 9) {
    int a = s->part[0][tid];
    for (int w = 1; w < 16; ++w) {
      const int o = s->part[w][tid];
      a = tid < 4 ? min(a, o) : tid < 8 ? max(a, o) : a + o;
    }
    int* const field = tid < 4 ? &s->box.mn[tid] : tid < 8 ? &s->box.mx[tid - 4] : &s->box.total;
    *field = a;
    if (bin == 0 && tid < 8) *(tid < 4 ? &hdr->mn[tid] : &hdr->mx[tid - 4]) = a;
  }
  __syncthreads();
  const int lo = __builtin_amdgcn_readfirstlane(s->box.total), hi = __builtin_amdgcn_readfirstlane(lo + s->listed);
  if (tid == 0) {
    bin_start[bin] = lo;
    if (bin == bins - 1) bin_start[bins] = n_keys;
    if (bin == 0) {
      hdr->num_keys = n_keys;
      hdr->bins = bins;
      hdr->stats_offset = stats_offset;
    }
  }
  const ListedEntries<Keys> in{keys, s->list, lo};
  build_bin<WANT_SLOT_OF, 4>(in, bin, lo, hi, layout_of(s->box), &s->bin, slots, wide_keys, order_tag, order_row,
                          block_list, perm, slot_of, bin_stats);
}

// Sums the bins' voxel and block counts into the header (for the host's status read; the
// kernel-map builder adds them up itself).
__global__ void __launch_bounds__(1024) table_sum_stats(WcnTableHeader* __restrict__ hdr) {
  __shared__ int s_v[16], s_b[16];
  const int32_t bins = hdr->bins;
  const int32_t* bin_stats = reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(hdr) + hdr->stats_offset);
  __shared__ int s_lost[16];
  const int status = wcn_table_status(hdr, (int)threadIdx.x, 1024, s_lost);
  int v = 0, b = 0;
  for (int i = threadIdx.x; i < bins; i += 1024) {
    v += bin_stats[2 * i];
    b += bin_stats[2 * i + 1] & ~WCN_BIN_LOST;
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) {
    v += __shfl_xor(v, s, 64);
    b += __shfl_xor(b, s, 64);
  }
  if (wcn_lane() == 0) {
    s_v[threadIdx.x >> 6] = v;
    s_b[threadIdx.x >> 6] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    v = b = 0;
    for (int w = 0; w < 16; ++w) {
      v += s_v[w];
      b += s_b[w];
    }
    hdr->total = v;
    hdr->num_blocks = b;
    hdr->status = status;
  }
}

__global__ void __launch_bounds__(256) table_query(const WcnTableHeader* __restrict__ hdr,
                                                   WcnTableRef table,
                                                   const int32_t* __restrict__ perm,
                                                   const int4* __restrict__ queries,
                                                   int64_t num_queries,
                                                   int32_t* __restrict__ results) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_queries) return;
  const WcnLayout L = wcn_make_layout(hdr);
  const int4 c = queries[i];
  uint32_t r[4];
  int32_t res = -1;
  if (L.ok && wcn_relative(L, c.x, c.y, c.z, c.w, r)) {
    int32_t base;
    const unsigned long long mask = wcn_lookup_block(L, table, r, &base);
    const uint32_t bit = wcn_block_bit(r);
    if ((mask >> bit) & 1ull) res = perm[base + wcn_rank_below(mask, bit)];
  }
  results[i] = res;
}

inline bool is_pow2(int64_t x) { return x > 0 && (x & (x - 1)) == 0; }

// One-item-per-thread kernels take the uncapped grid (a grid's x extent reaches 2^31 - 1 blocks, and
// item counts here stay below 2^31); a cap is for kernels that loop with a grid stride.
inline int grid_for(int64_t n, int block, int cap = 0x7fffffff) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

}  // namespace

// LDS beyond the default limit: lifted once per device and kernel.
static int allow_lds(const void* kernel, size_t bytes, int which) {
  static std::mutex mu;
  static bool allowed[12][64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return WCN_ERR_LAUNCH;
  std::lock_guard<std::mutex> hold(mu);
  if (allowed[which][device]) return WCN_OK;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
    return WCN_ERR_LAUNCH;
  allowed[which][device] = true;
  return WCN_OK;
}

// Enqueue the build kernels.  Shared with the strided-coordinate path, which also wants the slot of
// every key (`want_slot_of`).
static int table_build_from(const int32_t* keys, int64_t n_keys, const WcnTableView& v, const KeysOfItems* items,
                            bool want_slot_of, hipStream_t s) {
  const int4* k4 = (const int4*)keys;
  if (v.bins < 1 || v.bins > WCN_MAX_BINS || (v.bins & (v.bins - 1))) return WCN_ERR_INVALID_ARGUMENT;
  const int64_t stats = (int64_t)((const char*)v.bin_stats - (const char*)v.hdr);
  if (n_keys >= 1 && n_keys <= SMALL_KEYS && v.bins <= SMALL_KEY_BINS) {
    auto small = want_slot_of ? (items ? table_small<true, true> : table_small<true, false>)
                              : (items ? table_small<false, true> : table_small<false, false>);
    const int which = 7 + (want_slot_of ? 2 : 0) + (items ? 1 : 0);
    if (allow_lds((const void*)small, sizeof(SmallLds), which) != WCN_OK) return WCN_ERR_LAUNCH;
    hipLaunchKernelGGL(small, dim3(v.bins), dim3(1024), sizeof(SmallLds), s, k4, items ? *items : KeysOfItems{}, (int32_t)n_keys,
                       v.bins, v.hdr, stats, v.slots, v.wide_keys, v.bin_start, v.order_tag, v.order_row, v.block_list, v.perm,
                       v.slot_of, v.bin_stats);
    WCN_LAUNCH_CHECK();
    return WCN_OK;
  }
  const bool many_bins = v.bins > SMALL_BINS;
  auto sort = items ? (many_bins ? table_sort<WCN_MAX_BINS / 1024, true> : table_sort<SMALL_BINS / 1024, true>)
                    : (many_bins ? table_sort<WCN_MAX_BINS / 1024, false> : table_sort<SMALL_BINS / 1024, false>);
  const bool two = v.bins > 256;  // more than one per CU: 64 registers let two share it (fewer bins: 15.7 -> 22 us of 500 k voxels)
  auto fn = want_slot_of ? (two ? table_bins<true, true> : table_bins<true, false>)
                         : (two ? table_bins<false, true> : table_bins<false, false>);
  if (allow_lds((const void*)fn, sizeof(BinsLds), (want_slot_of ? 1 : 0) + (two ? 3 : 0)) != WCN_OK) return WCN_ERR_LAUNCH;
  // (up to 4096 bins beside the counters a part's keys, 16 and 2 bytes each)
  const size_t sort_lds = sizeof(int) * (size_t)v.bins + (many_bins ? 0 : 4096 * 18);
  if (allow_lds((const void*)sort, many_bins ? sizeof(int) * WCN_MAX_BINS : sizeof(int) * SMALL_BINS + 4096 * 18,
                many_bins ? (items ? 6 : 2) : (items ? 11 : 5)) != WCN_OK)
    return WCN_ERR_LAUNCH;
  hipLaunchKernelGGL(sort, dim3(v.parts), dim3(1024), sort_lds, s, k4, n_keys, v.bins, v.part_start, v.part_box,
                     (int4*)v.bin_coords, v.bin_row, items ? *items : KeysOfItems{});
  hipLaunchKernelGGL(fn, dim3(v.bins), dim3(1024), sizeof(BinsLds), s, v.hdr, n_keys, stats, v.slots, v.wide_keys, v.part_start,
                     v.part_box, v.parts, v.bin_start, (const int4*)v.bin_coords, v.bin_row, v.order_tag, v.order_row,
                     v.block_list, v.perm, v.slot_of, v.bin_stats);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_table_build_impl(const int32_t* keys, int64_t n_keys, const WcnTableView& v, bool want_slot_of, hipStream_t s) {
  return table_build_from(keys, n_keys, v, nullptr, want_slot_of, s);
}


// Host waits are polls (a blocking stream synchronisation wakes the host tens of microseconds
// late) with an upper bound: WCN_WAIT_LIMIT_MS milliseconds (environment, default 60000), after
// which the call gives up with WCN_ERR_LAUNCH instead of spinning for ever on a stream that is
// stuck.  After a short spin the poll yields the core between looks.
namespace {
int64_t wait_limit_ns() {
  static const int64_t limit = [] {
    const char* e = getenv("WCN_WAIT_LIMIT_MS");
    const long long ms = e ? atoll(e) : 0;
    return (int64_t)(ms > 0 ? ms : 60000) * 1000000;
  }();
  return limit;
}
struct BoundedPoll {
  std::chrono::steady_clock::time_point start = std::chrono::steady_clock::now();
  unsigned looks = 0;
  // false once the time limit has passed
  bool again() {
    if ((++looks & 0xFFu) != 0) return true;
    const int64_t ns = std::chrono::duration_cast<std::chrono::nanoseconds>(
                           std::chrono::steady_clock::now() - start).count();
    if (ns > wait_limit_ns()) return false;
    if (ns > 200000) std::this_thread::yield();
    return true;
  }
};
int wait_for_event(hipEvent_t ev) {
  BoundedPoll poll;
  for (;;) {
    const hipError_t e = hipEventQuery(ev);
    if (e == hipSuccess) return WCN_OK;
    if (e != hipErrorNotReady || !poll.again()) return WCN_ERR_LAUNCH;
  }
}
// per-thread pinned staging of wcn_read_small (released by wcn_thread_release)
thread_local void* g_small_staging = nullptr;
thread_local hipEvent_t g_small_done = nullptr;
thread_local int g_small_device = -1;
}  // namespace

int wcn_read_small(void* host_dst, const void* device_src, size_t bytes, hipStream_t stream) {
  constexpr size_t kStaging = 16384;
  void*& staging = g_small_staging;
  hipEvent_t& done = g_small_done;
  int& staging_device = g_small_device;
  if (bytes > kStaging) return WCN_ERR_INVALID_ARGUMENT;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return WCN_ERR_LAUNCH;
  if (!staging) {
    if (hipHostMalloc(&staging, kStaging, hipHostMallocDefault) != hipSuccess) {
      staging = nullptr;
      return WCN_ERR_LAUNCH;
    }
  }
  if (!done || staging_device != device) {  // events belong to the device they were created on
    if (done) (void)hipEventDestroy(done);
    if (hipEventCreateWithFlags(&done, hipEventDisableTiming) != hipSuccess) {
      done = nullptr;
      return WCN_ERR_LAUNCH;
    }
    staging_device = device;
  }
  if (hipMemcpyAsync(staging, device_src, bytes, hipMemcpyDeviceToHost, stream) != hipSuccess)
    return WCN_ERR_LAUNCH;
  if (hipEventRecord(done, stream) != hipSuccess) return WCN_ERR_LAUNCH;
  if (wait_for_event(done) != WCN_OK) return WCN_ERR_LAUNCH;
  memcpy(host_dst, staging, bytes);
  return WCN_OK;
}

// A read that is requested where the data is produced and collected later: the copy into the
// thread's second staging buffer is enqueued at once (so that it runs before whatever the caller
// enqueues next), the wait happens in wcn_read_early_end.  One pending read per host thread; an
// end without a matching begin is a plain wcn_read_small.
namespace {
constexpr size_t kEarlyStaging = 16384;
thread_local void* g_early_staging = nullptr;
thread_local hipEvent_t g_early_done = nullptr;
thread_local int g_early_device = -1;
thread_local const void* g_early_src = nullptr;
thread_local size_t g_early_bytes = 0;
}  // namespace

int wcn_read_early_begin(const void* device_src, size_t bytes, hipStream_t stream) {
  g_early_src = nullptr;
  if (bytes > kEarlyStaging) return WCN_ERR_INVALID_ARGUMENT;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return WCN_ERR_LAUNCH;
  if (!g_early_staging &&
      hipHostMalloc(&g_early_staging, kEarlyStaging, hipHostMallocDefault) != hipSuccess) {
    g_early_staging = nullptr;
    return WCN_ERR_LAUNCH;
  }
  if (!g_early_done || g_early_device != device) {
    if (g_early_done) (void)hipEventDestroy(g_early_done);
    if (hipEventCreateWithFlags(&g_early_done, hipEventDisableTiming) != hipSuccess) {
      g_early_done = nullptr;
      return WCN_ERR_LAUNCH;
    }
    g_early_device = device;
  }
  if (hipMemcpyAsync(g_early_staging, device_src, bytes, hipMemcpyDeviceToHost, stream) != hipSuccess)
    return WCN_ERR_LAUNCH;
  if (hipEventRecord(g_early_done, stream) != hipSuccess) return WCN_ERR_LAUNCH;
  g_early_src = device_src;
  g_early_bytes = bytes;
  return WCN_OK;
}

int wcn_read_early_end(void* host_dst, const void* device_src, size_t bytes, hipStream_t stream) {
  if (g_early_src != device_src || g_early_bytes != bytes)
    return wcn_read_small(host_dst, device_src, bytes, stream);
  g_early_src = nullptr;
  if (wait_for_event(g_early_done) != WCN_OK) return WCN_ERR_LAUNCH;
  memcpy(host_dst, g_early_staging, bytes);
  return WCN_OK;
}

namespace {
// Events that maps have given back, by device, for the mailbox writes to come: created and destroyed with every map they took
// 2 us of the host.  An event may be recorded again while an earlier record is still waited for: the wait is for that one.
constexpr size_t kIdleEvents = 64;  // of a device; more are destroyed
struct IdleEvents {
  std::mutex mu;
  std::vector<hipEvent_t> of[64];
};
IdleEvents& idle_events() {
  static IdleEvents* const pool = new IdleEvents;  // (never destroyed: maps may outlive static objects)
  return *pool;
}
hipError_t event_for(int device, hipEvent_t* event) {
  if (device >= 0 && device < 64) {
    IdleEvents& pool = idle_events();
    std::lock_guard<std::mutex> hold(pool.mu);
    if (!pool.of[device].empty()) {
      *event = pool.of[device].back();
      pool.of[device].pop_back();
      return hipSuccess;
    }
  }
  return hipEventCreateWithFlags(event, hipEventDisableTiming);
}

constexpr size_t kMailboxBytes = 16384;
thread_local int64_t* g_box = nullptr;        // pinned, coherent, mapped
thread_local hipEvent_t g_box_done = nullptr;
thread_local int g_box_device = -1;
thread_local int64_t g_box_sequence = 0;
thread_local int64_t g_box_open = 0;  // the sequence of a write that is on its way and that nobody has collected
}  // namespace

int wcn_mailbox_begin(int64_t** device_visible_box, int64_t* sequence) {
  // A write that nobody has collected (an error between a call and its read) may be on its way still, on another stream
  // than this call's: its words would land among this call's.  Until it has landed there is no mailbox.
  if (g_box_open != 0 && *(volatile int64_t*)g_box != g_box_open) {
    const hipError_t earlier = hipPeekAtLastError();  // of the caller's launches: not to be lost
    const hipError_t e = hipEventQuery(g_box_done);
    if (e != hipSuccess && earlier == hipSuccess) (void)hipGetLastError();
    if (e == hipErrorNotReady) return WCN_ERR_LAUNCH;
  }
  g_box_open = 0;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return WCN_ERR_LAUNCH;
  if (!g_box) {
    void* p = nullptr;
    if (hipHostMalloc(&p, kMailboxBytes, hipHostMallocCoherent | hipHostMallocMapped) != hipSuccess)
      return WCN_ERR_LAUNCH;
    g_box = (int64_t*)p;
    g_box[0] = 0;
  }
  if (!g_box_done || g_box_device != device) {
    if (g_box_done) (void)hipEventDestroy(g_box_done);
    if (event_for(device, &g_box_done) != hipSuccess) {
      g_box_done = nullptr;
      return WCN_ERR_LAUNCH;
    }
    g_box_device = device;
  }
  void* dev = nullptr;
  if (hipHostGetDevicePointer(&dev, g_box, 0) != hipSuccess) return WCN_ERR_LAUNCH;
  *device_visible_box = (int64_t*)dev;
  *sequence = ++g_box_sequence;
  return WCN_OK;
}

int wcn_mailbox_mark(hipStream_t stream) {
  if (!g_box_done || hipEventRecord(g_box_done, stream) != hipSuccess) return WCN_ERR_LAUNCH;
  g_box_open = g_box_sequence;
  return WCN_OK;
}

int wcn_mailbox_end(void* host_dst, size_t payload_bytes, int64_t sequence, bool kernel_over) {
  if (!g_box || !g_box_done || payload_bytes + 8 > kMailboxBytes) return WCN_ERR_INVALID_ARGUMENT;
  volatile int64_t* word0 = g_box;
  BoundedPoll poll;
  for (;;) {
    if (!kernel_over && *word0 == sequence) break;
    const hipError_t e = hipEventQuery(g_box_done);
    if (e == hipErrorNotReady) {
      if (!poll.again()) return WCN_ERR_LAUNCH;
      continue;
    }
    if (e != hipSuccess) return WCN_ERR_LAUNCH;
    // the kernel is over: its write must be there by now, or it never happened
    if (*word0 == sequence) break;
    return WCN_ERR_LAUNCH;
  }
  __atomic_thread_fence(__ATOMIC_ACQUIRE);
  memcpy(host_dst, (const void*)(g_box + 1), payload_bytes);
  if (g_box_open == sequence) g_box_open = 0;
  return WCN_OK;
}

// The event behind the thread's last write, which has been collected, is the caller's from here on (the next write gets another).
void* wcn_mailbox_take_event(int32_t* device) {
  if (g_box_open != 0) return nullptr;
  void* const event = (void*)g_box_done;
  g_box_done = nullptr;
  *device = g_box_device;
  return event;
}

int wcn_table_status_from_bits(int32_t bits) {
  if (bits & WCN_DEV_RANGE) return WCN_ERR_COORD_RANGE;
  if (bits & WCN_DEV_OVERFLOW) return WCN_ERR_TABLE_OVERFLOW;
  return WCN_OK;
}

extern "C" {

int wcn_version(void) { return 200; }

void wcn_kmap_return_event(void* event, int32_t device) {
  if (!event) return;
  if (device >= 0 && device < 64) {
    IdleEvents& pool = idle_events();
    std::lock_guard<std::mutex> hold(pool.mu);
    if (pool.of[device].size() < kIdleEvents) {
      pool.of[device].push_back((hipEvent_t)event);
      return;
    }
  }
  (void)hipEventDestroy((hipEvent_t)event);
}

int wcn_thread_release(void) {
  int st = WCN_OK;
  {
    IdleEvents& pool = idle_events();
    std::lock_guard<std::mutex> hold(pool.mu);
    for (auto& events : pool.of) {
      for (hipEvent_t e : events)
        if (hipEventDestroy(e) != hipSuccess) st = WCN_ERR_LAUNCH;
      events.clear();
    }
  }
  if (g_small_done && hipEventDestroy(g_small_done) != hipSuccess) st = WCN_ERR_LAUNCH;
  if (g_early_done && hipEventDestroy(g_early_done) != hipSuccess) st = WCN_ERR_LAUNCH;
  if (g_box_done && hipEventDestroy(g_box_done) != hipSuccess) st = WCN_ERR_LAUNCH;
  if (g_small_staging && hipHostFree(g_small_staging) != hipSuccess) st = WCN_ERR_LAUNCH;
  if (g_early_staging && hipHostFree(g_early_staging) != hipSuccess) st = WCN_ERR_LAUNCH;
  if (g_box && hipHostFree(g_box) != hipSuccess) st = WCN_ERR_LAUNCH;
  g_small_done = g_early_done = g_box_done = nullptr;
  g_small_staging = g_early_staging = nullptr;
  g_box = nullptr;
  g_box_open = 0;
  g_small_device = g_early_device = g_box_device = -1;
  g_early_src = nullptr;
  return st;
}

const char* wcn_status_string(int status) {
  switch (status) {
    case WCN_OK: return "success";
    case WCN_ERR_INVALID_ARGUMENT: return "invalid argument";
    case WCN_ERR_LAUNCH: return "HIP launch or copy failed";
    case WCN_ERR_TABLE_OVERFLOW: return "a bin of the coordinate table holds more blocks than it has slots (capacity too small)";
    case WCN_ERR_COORD_RANGE: return "coordinate bounding box does not fit the 63-bit block key";
    case WCN_ERR_TOO_MANY_PAIRS: return "kernel map exceeds 2^31-1 pairs";
    case WCN_ERR_WORKSPACE: return "workspace too small";
    default: return "unknown status";
  }
}

int64_t wcn_table_default_capacity(int64_t n_keys) {
  // Blocks hold up to 64 voxels; surface-like data fills ~10 per block.  The power of two above the key count makes bins of one
  // to two thousand keys (2,048 slots each): a bin overflows only where almost every voxel is alone in its block and more than
  // the average falls to it; the build then reports WCN_ERR_TABLE_OVERFLOW and the caller retries with 4x the slots.
  int64_t want = n_keys + 1;
  int64_t cap = 1024;
  while (cap < want) cap <<= 1;
  return cap;
}

size_t wcn_table_bytes(int64_t n_keys, int64_t capacity) {
  if (n_keys < 0 || capacity <= 0) return 0;
  return wcn_table_layout(nullptr, n_keys, capacity, nullptr);
}

int wcn_table_build(const int32_t* keys, int64_t n_keys, void* table, int64_t capacity,
                    void* stream) {
  if (!table || n_keys < 0 || (n_keys > 0 && !keys)) return WCN_ERR_INVALID_ARGUMENT;
  if (!is_pow2(capacity) || capacity < 64 || capacity > (1ll << 31)) return WCN_ERR_INVALID_ARGUMENT;
  if (n_keys >= (1ll << 31)) return WCN_ERR_INVALID_ARGUMENT;
  WcnTableView v;
  wcn_table_layout(table, n_keys, capacity, &v);
  return wcn_table_build_impl(keys, n_keys, v, false, (hipStream_t)stream);
}

int wcn_table_build_items(const int32_t* coords, int64_t n_rows, const int64_t* host_batch_offsets, int32_t batch_size,
                          int32_t* rows, void* table, int64_t capacity, void* stream) {
  KeysOfItems of = {coords, (int4*)rows, {}, batch_size};
  if (!table || n_rows < 1 || n_rows >= (1ll << 31) || !coords || !rows || (uintptr_t)rows % 16 != 0 || !is_pow2(capacity) ||
      capacity < 64 || capacity > (1ll << 31) || !wcn_item_starts(host_batch_offsets, batch_size, n_rows, &of.starts))
    return WCN_ERR_INVALID_ARGUMENT;
  WcnTableView v;
  wcn_table_layout(table, n_rows, capacity, &v);
  return table_build_from(rows, n_rows, v, &of, false, (hipStream_t)stream);
}

int wcn_table_query(const void* table, int64_t n_keys, int64_t capacity, const int32_t* queries,
                    int64_t num_queries, int32_t* results, void* stream) {
  if (!table || num_queries < 0 || (num_queries > 0 && (!queries || !results)))
    return WCN_ERR_INVALID_ARGUMENT;
  if (!is_pow2(capacity) || capacity < 64 || n_keys < 0) return WCN_ERR_INVALID_ARGUMENT;
  if (num_queries == 0) return WCN_OK;
  WcnTableView v;
  wcn_table_layout(const_cast<void*>(table), n_keys, capacity, &v);
  hipLaunchKernelGGL(table_query, dim3(grid_for(num_queries, 256)), dim3(256), 0,
                     (hipStream_t)stream, v.hdr, wcn_table_ref(v), v.perm,
                     (const int4*)queries, num_queries, results);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_table_read_status(const void* table, int32_t* host_num_blocks, void* stream) {
  if (!table) return WCN_ERR_INVALID_ARGUMENT;
  WcnTableHeader h;
  hipLaunchKernelGGL(table_sum_stats, dim3(1), dim3(1024), 0, (hipStream_t)stream,
                     reinterpret_cast<WcnTableHeader*>(const_cast<void*>(table)));
  WCN_LAUNCH_CHECK();
  if (wcn_read_small(&h, table, sizeof(h), (hipStream_t)stream) != WCN_OK) return WCN_ERR_LAUNCH;
  if (host_num_blocks) *host_num_blocks = h.num_blocks;
  return wcn_table_status_from_bits(h.status);
}

}  // extern "C"
