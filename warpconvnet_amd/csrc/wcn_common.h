// Shared host/device definitions of libwcn_hip.so (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/wcn_hip.h"

#define WCN_WAVE 64
#define WCN_EMPTY_KEY 0xFFFFFFFFFFFFFFFFull
#define WCN_EMPTY_TAG 0xFFFFFFFFu
#define WCN_MAX_OFFSETS 1024  // kernel volume bound of the kernel-map kernels

// Conditions of a table that its build records (a bit set).
#define WCN_DEV_OVERFLOW 1
#define WCN_DEV_RANGE 2

// ---- coordinate table -------------------------------------------------------------------------
// The table does not store one slot per voxel.  Space is cut into 4x4x4-voxel blocks; a slot
// holds a tag of the packed block coordinate, a 64-bit occupancy mask of the block and the rank of its
// first voxel in `perm`, the list of input rows grouped by block.  A voxel's row index is
// perm[base + popcount(mask below its bit)].  One 16-byte slot, one request, answers up to 64 probes.
// The tag is the block coordinate itself where that fits 31 bits (4096 x 4096 x 2048 voxels and 8 batch items do), else 31 bits
// of a hash of it: then the coordinates lie beside the slots, 8 bytes each, and a look-up compares them too (a second request behind
// the first: table and 3x3x3 map over 1 M rows of rooms 124 us, with one voxel far away 144; 5x5x5 231 and 256.  Slots of 32 bytes with the
// key in them took 169 and 306 either way).
// The slots come in regions of WCN_BIN_SLOTS, one per bin of the build: every block of a 16x16x16-voxel cell is in the
// region that the cell's hash names, so a region is made by one workgroup, in LDS, and written from end to end: no slot is
// cleared beforehand and none is claimed with an atomic.
struct __attribute__((aligned(16))) WcnSlot {
  uint32_t tag;             // or WCN_EMPTY_TAG
  uint32_t base;            // first position of the block's voxels in perm, | WCN_SLOT_PASSED where the search for another goes on
  unsigned long long mask;  // bit (x&3)*16 + (y&3)*4 + (z&3)
};
#define WCN_SLOT_PASSED 0x80000000u

struct __attribute__((aligned(32))) WcnBlock {  // a line of a bin's block list
  unsigned long long key;   // packed (batch, bx, by, bz) relative to the bounding box
  unsigned long long mask;
  int32_t base;
  int32_t first;            // first entry of the block, counted from the bin's first
  int32_t pad[2];
};

struct WcnTableHeader {  // first 256 bytes of a table workspace
  int32_t mn[4];         // bounding box of the keys, per column
  int32_t mx[4];
  int32_t num_blocks;    // occupied slots (valid after table_sum_stats)
  int32_t status;        // WCN_DEV_* bits (valid after table_sum_stats)
  int32_t total;         // number of distinct keys (valid after table_sum_stats)
  int32_t num_keys;      // keys inserted; more keys than set bits (`total`) means some key came twice
  int32_t bins;          // bins of the build
  int32_t pad;
  int64_t stats_offset;  // bytes from the header to the bins' (voxels, blocks) counts
  int32_t reserved[48];
};
static_assert(sizeof(WcnTableHeader) == 256, "header is 256 bytes");

struct WcnTableView {  // host-computed addresses inside a table workspace
  WcnTableHeader* hdr;
  WcnSlot* slots;         // bins regions of WCN_BIN_SLOTS
  unsigned long long* wide_keys;  // their block coordinates, where a tag does not hold them
  int32_t* perm;        // n_keys
  int32_t* slot_of;     // n_keys (slot of each key; written on request)
  // The keys in block order: every key once, the keys of one block next to each other, the blocks
  // of one bin next to each other (bin b owns entries bin_start[b] .. bin_start[b + 1]).
  int32_t* order_tag;     // n_keys: (index of the entry's block in its bin's block list) << 6 | voxel bit
  int32_t* order_row;     // n_keys: input row of each entry
  // The blocks of bin b, in the order of its entries: block_list[bin_start[b] + j], j < blocks of
  // the bin.
  WcnBlock* block_list;   // n_keys places (a bin has at most as many blocks as keys)
  // build scratch
  int32_t* bin_coords;    // (n_keys, 4) the keys of every part, grouped by bin within the part
  int32_t* bin_row;       // n_keys
  int32_t* part_start;    // (bins + 1, parts): keys of part w in the bins before b
  int32_t* bin_start;     // bins + 1
  int32_t* bin_stats;     // (bins, 2): distinct keys of each bin; its blocks, | WCN_BIN_LOST where some found no place
  int32_t* part_box;      // (parts, 8) bounding box of each part's keys
  int64_t n_keys;
  int64_t capacity;
  int32_t bins;           // power of two
  int32_t parts;          // workgroups of the sort
};

static inline size_t wcn_align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Keys are first grouped into bins of one to two thousand (a bin is a hash of the key's 16x16x16-voxel
// cell, so the 4x4x4 blocks of a cell stay together); the bin count follows the slot count, so a
// rebuild with more slots also re-deals the bins.
#define WCN_BIN_SLOTS 2048      // slots of a bin's region: the distinct blocks it can hold
#define WCN_BIN_LOST (1 << 30)
#define WCN_PART_KEYS 1024      // keys of a workgroup of the sort (more beyond 256 of them)
#define WCN_MAX_BINS 32768      // a counter per bin in LDS during the build: 128 KB
static inline int32_t wcn_table_bins(int64_t capacity) {
  int64_t b = capacity / 2048;
  if (b < 16) b = 16;
  if (b > WCN_MAX_BINS) b = WCN_MAX_BINS;
  return (int32_t)b;
}
static inline int32_t wcn_table_parts(int64_t n_keys) {
  int64_t w = (n_keys + WCN_PART_KEYS - 1) / WCN_PART_KEYS;
  if (w < 1) w = 1;
  if (w > 256) w = 256;
  return (int32_t)w;
}

static inline size_t wcn_table_layout(void* base, int64_t n_keys, int64_t capacity,
                                      WcnTableView* v) {
  char* p = (char*)base;
  size_t off = 0;
  const int32_t bins = wcn_table_bins(capacity), parts = wcn_table_parts(n_keys);
  if (v) v->hdr = (WcnTableHeader*)(p + off);
  off += 256;
  if (v) v->slots = (WcnSlot*)(p + off);
  off += sizeof(WcnSlot) * WCN_BIN_SLOTS * (size_t)bins;
  if (v) v->wide_keys = (unsigned long long*)(p + off);
  off += sizeof(unsigned long long) * WCN_BIN_SLOTS * (size_t)bins;
  if (v) v->perm = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)n_keys);
  if (v) v->slot_of = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)n_keys);
  if (v) v->order_tag = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)n_keys);
  if (v) v->order_row = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)n_keys);
  if (v) v->block_list = (WcnBlock*)(p + off);
  off += wcn_align256(sizeof(WcnBlock) * (size_t)n_keys);
  if (v) v->bin_coords = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * 4 * (size_t)n_keys);
  if (v) v->bin_row = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)n_keys);
  if (v) v->part_start = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)(bins + 1) * (size_t)parts);
  if (v) v->bin_start = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)(bins + 1));
  if (v) v->bin_stats = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * 2 * (size_t)bins);
  if (v) v->part_box = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * 8 * (size_t)parts);
  if (v) {
    v->n_keys = n_keys;
    v->capacity = capacity;
    v->bins = bins;
    v->parts = parts;
  }
  return off;
}

#ifdef __HIPCC__

// Bit layout of the packed block key, derived from the bounding box in the header.
struct WcnLayout {
  uint32_t amin[4];   // batch minimum; spatial minima rounded down to a multiple of 4
  uint32_t span[4];   // largest valid (coord - amin) per column
  uint32_t shift[4];  // left shift of each field in the key
  bool ok;            // all fields fit in 63 bits
  bool wide;          // ... but not in 31
};

__device__ __forceinline__ WcnLayout wcn_make_layout(const WcnTableHeader* __restrict__ h) {
  WcnLayout L;
  uint32_t bits[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    int32_t mn = h->mn[d], mx = h->mx[d];
    uint32_t a = d == 0 ? (uint32_t)mn : ((uint32_t)mn & ~3u);
    L.amin[d] = a;
    L.span[d] = (uint32_t)mx - a;
    uint32_t cells = d == 0 ? L.span[d] : (L.span[d] >> 2);  // largest field value
    bits[d] = cells == 0 ? 0u : 32u - (uint32_t)__builtin_clz(cells);
  }
  L.shift[3] = 0;
  L.shift[2] = bits[3];
  L.shift[1] = bits[3] + bits[2];
  L.shift[0] = bits[3] + bits[2] + bits[1];
  const uint32_t total = bits[0] + bits[1] + bits[2] + bits[3];
  L.ok = total <= 63u;
  L.wide = total > 31u;
  return L;
}

// Relative coordinates of (b,x,y,z); false if the point lies outside the bounding box.
__device__ __forceinline__ bool wcn_relative(const WcnLayout& L, int b, int x, int y, int z,
                                             uint32_t r[4]) {
  r[0] = (uint32_t)b - L.amin[0];
  r[1] = (uint32_t)x - L.amin[1];
  r[2] = (uint32_t)y - L.amin[2];
  r[3] = (uint32_t)z - L.amin[3];
  return r[0] <= L.span[0] && r[1] <= L.span[1] && r[2] <= L.span[2] && r[3] <= L.span[3];
}

__device__ __forceinline__ unsigned long long wcn_block_key(const WcnLayout& L,
                                                            const uint32_t r[4]) {
  return ((unsigned long long)r[0] << L.shift[0]) | ((unsigned long long)(r[1] >> 2) << L.shift[1]) |
         ((unsigned long long)(r[2] >> 2) << L.shift[2]) | (unsigned long long)(r[3] >> 2);
}

__device__ __forceinline__ uint32_t wcn_block_bit(const uint32_t r[4]) {
  return ((r[1] & 3u) << 4) | ((r[2] & 3u) << 2) | (r[3] & 3u);
}

// Hash of the 16x16x16-voxel cell that holds a block, from the block's absolute coordinates (block boundaries are multiples of
// four in absolute coordinates: the table's origin is rounded down to one): the sum of a term per column, finalised.  The columns'
// multipliers are the first four primes of 32-bit xxHash (any odd numbers without small relations between them would do), the last one
// is of MurmurHash3's finaliser.  One multiplication does: bins and places are as even as with two (rooms, spheres, full cubes, grids of step 8 to 64).
__device__ __forceinline__ uint32_t wcn_cell_batch(uint32_t batch) { return batch * 0x9E3779B1u; }
__device__ __forceinline__ uint32_t wcn_cell_x(int32_t block) { return (uint32_t)(block >> 2) * 0x85EBCA77u; }
__device__ __forceinline__ uint32_t wcn_cell_y(int32_t block) { return (uint32_t)(block >> 2) * 0xC2B2AE3Du; }
__device__ __forceinline__ uint32_t wcn_cell_z(int32_t block) { return (uint32_t)(block >> 2) * 0x27D4EB2Fu; }
__device__ __forceinline__ uint32_t wcn_cell_hash(uint32_t sum) {
  sum ^= sum >> 16;
  sum *= 0xC2B2AE35u;
  return sum ^ (sum >> 15);
}

// Where a block is looked for: in its bin's region, first at its place in the line of 128 bytes of its 8x8x8-voxel cell (a
// row's neighbourhood lies in 3.4 blocks but in 2 lines on average), then in another line (wcn_probe_slot).  The eight
// lines of a larger cell, and a line's eight places, are turned by the larger cell's hash (exclusive or with the sum of a word per
// dimension).  Lines that follow one another, and a search of the line's other places, were slower: the blocks
// of a dense cell stand in each other's way (up to 50 slots looked at for the slowest lane of a wave, 2 this way).  A second place
// anywhere in the region: 66 us for the probe pass of 1 M voxels of rooms instead of 59; the blocks of a cell that gives way to another
// stay in one line this way.
__device__ __forceinline__ uint32_t wcn_place_x(int32_t block) { return ((block & 2) ? 0x95u << 3 : 0u) | (uint32_t)(block & 1) << 2; }
__device__ __forceinline__ uint32_t wcn_place_y(int32_t block) { return ((block & 2) ? 0x4Eu << 3 : 0u) | (uint32_t)(block & 1) << 1; }
__device__ __forceinline__ uint32_t wcn_place_z(int32_t block) { return ((block & 2) ? 0x2Bu << 3 : 0u) | (uint32_t)(block & 1); }
__device__ __forceinline__ uint32_t wcn_home_slot(uint32_t cell, uint32_t place, uint32_t bin_mask) {
  return (cell & bin_mask) * WCN_BIN_SLOTS | (((cell >> 16) ^ place) & (WCN_BIN_SLOTS - 1));
}
static_assert(WCN_BIN_SLOTS == 2048 && WCN_MAX_BINS <= 32768, "places from bits 16 to 26 of the hash, bins from bits 0 to 14");
__device__ __forceinline__ uint32_t wcn_home_slot_of(int32_t batch, int32_t bx, int32_t by, int32_t bz, uint32_t bin_mask) {
  return wcn_home_slot(wcn_cell_hash(wcn_cell_batch((uint32_t)batch) + wcn_cell_x(bx) + wcn_cell_y(by) + wcn_cell_z(bz)),
                       wcn_place_x(bx) ^ wcn_place_y(by) ^ wcn_place_z(bz), bin_mask);
}
// The p-th slot of the search: the same place of another line, then nine slots further and further; with p up to WCN_BIN_SLOTS
// all of the region's.
__device__ __forceinline__ uint32_t wcn_probe_slot(uint32_t home, int p) {
  if (p == 0) return home;
  return (home & ~(uint32_t)(WCN_BIN_SLOTS - 1)) | (((home ^ (0xB5u << 3)) + 9u * (uint32_t)(p - 1)) & (WCN_BIN_SLOTS - 1));
}

// What a slot's tag says of a block key (never WCN_EMPTY_TAG).
__device__ __forceinline__ uint32_t wcn_block_tag(const WcnLayout& L, unsigned long long key) {
  return L.wide ? ((uint32_t)(key ^ (key >> 31)) * 0x9E3779B1u) >> 1 : (uint32_t)key;
}

struct WcnTableRef {  // what a look-up reads
  const WcnSlot* __restrict__ slots;
  const unsigned long long* __restrict__ wide_keys;  // read only where the layout is wide
  uint32_t bin_mask;
};

inline WcnTableRef wcn_table_ref(const WcnTableView& v) { return {v.slots, v.wide_keys, (uint32_t)v.bins - 1u}; }

// Finds the slot of a block key from probe `p` on.  Returns its mask (0 if the block is absent) and base.
__device__ __forceinline__ unsigned long long wcn_lookup_block_from(const WcnLayout& L, const WcnTableRef& t,
                                                                    unsigned long long key, uint32_t home, int p,
                                                                    int32_t* base) {
  const uint32_t tag = wcn_block_tag(L, key);
  for (; p <= WCN_BIN_SLOTS; ++p) {
    const uint32_t h = wcn_probe_slot(home, p);
    const uint4 s = *reinterpret_cast<const uint4*>(&t.slots[h]);
    if (s.x == tag && (!L.wide || t.wide_keys[h] == key)) {
      *base = (int32_t)(s.y & ~WCN_SLOT_PASSED);
      return ((unsigned long long)s.w << 32) | s.z;
    }
    if (!(s.y & WCN_SLOT_PASSED)) break;
  }
  *base = 0;
  return 0ull;
}

// The block at relative coordinates (batch, x, y, z in blocks) within the box.
__device__ __forceinline__ uint32_t wcn_home_of_relative(const WcnLayout& L, uint32_t rb, uint32_t bx, uint32_t by, uint32_t bz,
                                                          uint32_t bin_mask) {
  return wcn_home_slot_of((int32_t)(rb + L.amin[0]), ((int32_t)L.amin[1] >> 2) + (int32_t)bx,
                          ((int32_t)L.amin[2] >> 2) + (int32_t)by, ((int32_t)L.amin[3] >> 2) + (int32_t)bz, bin_mask);
}
// The block of a voxel at relative coordinates r.
__device__ __forceinline__ unsigned long long wcn_lookup_block(const WcnLayout& L, const WcnTableRef& t, const uint32_t r[4],
                                                               int32_t* base) {
  return wcn_lookup_block_from(L, t, wcn_block_key(L, r), wcn_home_of_relative(L, r[0], r[1] >> 2, r[2] >> 2, r[3] >> 2, t.bin_mask),
                               0, base);
}

// The table's WCN_DEV_* bits, by all `threads` (>= 64, a multiple of 64) of a workgroup; `shared`: 16 words of LDS.
__device__ __forceinline__ int wcn_table_status(const WcnTableHeader* __restrict__ h, int tid, int threads, int32_t* shared) {
  const int32_t* stats = reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(h) + h->stats_offset);
  int lost = 0;
  for (int b = tid; b < h->bins; b += threads) lost |= stats[2 * b + 1] & WCN_BIN_LOST;
  const bool any = __ballot(lost != 0) != 0ull;
  if ((tid & 63) == 0) shared[tid >> 6] = any ? 1 : 0;
  __syncthreads();
  int all = 0;
  for (int w = 0; w < threads / 64; ++w) all |= shared[w];
  return (all ? WCN_DEV_OVERFLOW : 0) | (h->num_keys > 0 && !wcn_make_layout(h).ok ? WCN_DEV_RANGE : 0);
}

__device__ __forceinline__ int wcn_rank_below(unsigned long long mask, uint32_t bit) {
  return __popcll(mask & ((1ull << bit) - 1ull));
}

// Workgroups go to the eight XCDs in turn (blockIdx % 8), each with an L2 of its own.  For kernels whose
// neighbouring tiles write into the same lines (a few bytes each) or read them: the tile of workgroup `b` of `n` so that an
// XCD works through one stretch of tiles, and the pieces of a line meet in its L2.
__device__ __forceinline__ int wcn_xcd_tile(int b, int n) {
  const int xcd = b & 7, each = n >> 3, more = n & 7;
  return xcd * each + (xcd < more ? xcd : more) + (b >> 3);
}

__device__ __forceinline__ int wcn_lane() { return (int)(threadIdx.x & 63); }

// Inclusive prefix sum over the 64 lanes of a wave: shifts inside rows of 16 lanes, then the last lane of
// a row added to the row behind it, then of the first half to the second.  Six vector instructions; the
// same steps by lane exchange are six LDS round trips.
__device__ __forceinline__ int wcn_wave_inclusive_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

#endif  // __HIPCC__

// Where the rows of every batch item begin; handed over in a launch's arguments.
struct WcnItemStarts {
  int64_t start[WCN_VOXEL_MAX_BATCH + 1];
};
// From batch_size + 1 host offsets: false if there are none, too many, or they do not ascend from 0 to num_rows.
static inline bool wcn_item_starts(const int64_t* host_offsets, int32_t batch_size, int64_t num_rows, WcnItemStarts* out) {
  if (!host_offsets || batch_size < 1 || batch_size > WCN_VOXEL_MAX_BATCH || host_offsets[0] != 0) return false;
  for (int b = 0; b <= batch_size; ++b) {
    if (b > 0 && host_offsets[b] < host_offsets[b - 1]) return false;
    out->start[b] = host_offsets[b];
  }
  for (int b = batch_size + 1; b <= WCN_VOXEL_MAX_BATCH; ++b) out->start[b] = num_rows;
  return host_offsets[batch_size] == num_rows;
}

#ifdef __HIPCC__
// The item of row i: `start` in LDS (lanes search at different places).
__device__ __forceinline__ int wcn_item_of(const int64_t* start, int batch_size, int64_t i) {
  int lo = 0, hi = batch_size;  // the item lies in [lo, hi)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= i) lo = mid; else hi = mid;
  }
  return lo;
}
#endif

// Small device-to-host reads (map offsets, table status, row counts): copied into pinned memory
// and awaited by polling an event, which returns within a few microseconds of the copy's end (a
// blocking stream synchronisation wakes the host tens of microseconds later).  One staging buffer
// and one event per host thread, created on first use and kept until the process ends.
int wcn_read_small(void* host_dst, const void* device_src, size_t bytes, hipStream_t stream);
// The same read split in two: begin enqueues the copy (before whatever is enqueued next), end waits
// for it; an end without a matching begin on this thread does the whole read.
int wcn_read_early_begin(const void* device_src, size_t bytes, hipStream_t stream);
int wcn_read_early_end(void* host_dst, const void* device_src, size_t bytes, hipStream_t stream);

// A result the device writes straight into pinned host memory (no copy command): `begin` hands out
// this thread's mailbox (device-visible address of up to 16 KiB - 8 bytes of payload behind an
// 8-byte sequence word) and a fresh sequence number; the kernel writes the payload, a system-scope
// fence, then the sequence number into word 0.  `end` polls word 0 (and `done`, an event recorded
// after the kernel, so that a kernel that never wrote cannot stall the host: it then returns
// WCN_ERR_LAUNCH and the caller reads the device copy instead) and copies the payload out.  While a write that was armed
// and not collected is on its way, `begin` returns WCN_ERR_LAUNCH: the caller reads the device copy.  With `kernel_over` it
// waits for `done` in any case (the kernel writes more than the mailbox, and the caller takes it for written).
int wcn_mailbox_begin(int64_t** device_visible_box, int64_t* sequence);
int wcn_mailbox_mark(hipStream_t stream);  // records `done` behind the writing kernel (and what was enqueued behind that)
void* wcn_mailbox_take_event(int32_t* device);  // `done` of a write that has been collected, the caller's from there on; or null
int wcn_mailbox_end(void* host_dst, size_t payload_bytes, int64_t sequence, bool kernel_over = false);

// Output-row form of a pair list (rows of the map grouped by output row, inside a row ascending
// in kernel offset): row_mask[m] has bit k set if offset k has a pair for output row m,
// row_in[row_ptr[m] .. row_ptr[m + 1]) are the input rows of those pairs.  Built by
// wcn_rows_build (wcn_conv.hip) inside a caller-provided workspace; used by the contraction to
// re-order lists that do not ascend and by the pooling kernels.
struct WcnRowsView {
  int64_t* offsets;    // K + 1, device copy of the host offsets
  uint32_t* row_mask;  // num_out * words
  int32_t* row_ptr;    // num_out + 1
  int32_t* row_in;     // pairs
  int32_t* groups;     // G + 1 (scan scratch)
  int64_t* row_total;  // 1 (scan scratch)
  int32_t words;       // ceil(K / 32)
  int64_t G;           // ceil(num_out / 64)
};
size_t wcn_rows_layout(void* base, int64_t num_out, int num_offsets, int64_t pairs, WcnRowsView* v);
// `v.offsets` must already hold the offsets; pairs whose output row is out of range are dropped.
int wcn_rows_build(const int32_t* in_maps, const int32_t* out_maps, int num_offsets, int64_t num_out,
                   int64_t pairs, const WcnRowsView& v, hipStream_t stream);

// The rows form of a builder's map in one launch (wcn_map_rows_build_grouped), which also sets `clear_words` words at `clear`
// to zero for the launches behind it.
int wcn_rows_from_groups(const int32_t* gathered_rows, const int32_t* grouping_rows, const int64_t* device_offsets,
                         const int32_t* group_start, int num_offsets, int64_t num_rows, int64_t num_pairs,
                         void* workspace, size_t workspace_bytes, int32_t* clear, int clear_words, hipStream_t stream);

// Tile plan of a map (wcn_tiles.hip): tiles of WCN_TILE_ROWS output rows with their own sets of offsets.
#define WCN_TILE_ROWS 128
#define WCN_TILE_MAX_OFFSETS 32
struct WcnTilePlan {
  uint32_t* zeros;  // 1 KiB of zeros
  int32_t* order;   // tiles * 128: output row of each place, -1 past the last
  uint32_t* mask;   // tiles: the tile's offsets
  int32_t* nbr;     // (tiles, K, 128): for the j-th offset of the tile's mask, the places' input rows (-1: none)
  int64_t tiles;
};
static inline size_t wcn_tile_plan_layout(void* base, int64_t num_out, int num_offsets, WcnTilePlan* t) {
  char* p = (char*)base;
  size_t off = 0;
  const int64_t tiles = (num_out + WCN_TILE_ROWS - 1) / WCN_TILE_ROWS;
  if (t) t->zeros = (uint32_t*)(p + off);
  off += 1024;
  if (t) t->order = (int32_t*)(p + off);
  off += wcn_align256(sizeof(int32_t) * (size_t)tiles * WCN_TILE_ROWS);
  if (t) t->mask = (uint32_t*)(p + off);
  off += wcn_align256(sizeof(uint32_t) * (size_t)tiles);
  if (t) t->nbr = (int32_t*)(p + off);
  off += sizeof(int32_t) * ((size_t)tiles * (size_t)num_offsets + 1) * WCN_TILE_ROWS;
  if (t) t->tiles = tiles;
  return off;
}

#ifdef __HIPCC__

#define WCN_LAUNCH_CHECK()                      \
  do {                                          \
    if (hipGetLastError() != hipSuccess) return WCN_ERR_LAUNCH; \
  } while (0)

#endif  // __HIPCC__
