// Voxelisation front-end of libwcn_hip.so (gfx950): points -> integer voxel rows, and the
// sorted-unique / CSR grouping of integer rows that the point-to-voxel pooling reduces over.
//
// The reference does this with torch ops: floor(points / voxel_size).int() + a batch column
// (warpconvnet/geometry/coords/ops/voxel.py:92-95), then torch.unique(dim=0, sorted,
// return_inverse, return_counts) + a stable argsort of the inverse + a cumulative sum + a scatter
// (warpconvnet/utils/unique.py:57-109).  Here every row is packed into one key whose numeric order is
// the rows' lexicographic order (fields relative to the bounding box, first column most
// significant; 32-bit words when they fit, 64-bit ones otherwise), and the keys are sorted by one
// distribution over memory:
//   unique_box      bounding box per workgroup (of points: the rows are never stored)
//   unique_split    one workgroup: the box, the field widths and the boundaries of the buckets: every
//                   8th key of a sorted sample, so that a bucket gets about 2048 rows whatever their
//                   distribution; a key that fills buckets by itself gets a bucket of its own
//   unique_assign   per part of 8192 rows: key, bucket, and place among the part's rows of that bucket
//   unique_columns  per bucket: prefix sums over the parts
//   unique_place    (key, row) to its place in its bucket
//   unique_bucket   per bucket, in LDS: the distinct keys, their order and the order of the rows
//                   (unique_bucket_large: the few buckets that are too large for it)
//   unique_finish   per bucket: the results that need the number of distinct keys in front of it
// Nothing of this waits for the host, which reads the count (and the box) once, at the end.
// 4 M points in 1.3 M voxels: 174 us over these kernels (box 16, split 26, assign 36, columns 8, place 15,
// buckets 35 + 18, finish 20), against 318 us, nine fills and two waits before, with rocPRIM's radix sort of the
// (key, row) pairs - four passes over memory for 28 bits - and its prefix sum over the heads.
// rocPRIM's radix sort and prefix sum (plain library primitives) stay for more rows than one
// workgroup can sample for, and for the improbable bucket that does not fit LDS.
#include "wcn_common.h"

#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

namespace {

constexpr int kBucketRows = 2048;  // rows of a bucket on average ...
constexpr int kBucketCap = 8192;   // ... and at most
constexpr int kMaxBuckets = 2048;
constexpr int kSamplesPerBucket = 8;
constexpr int kMaxSamples = kMaxBuckets * kSamplesPerBucket;
constexpr int kPartRows = 8192;
constexpr int kBoxParts = 256;
// The largest sample one workgroup can sort makes buckets of 2176 rows on average here; that one of
// them has more than 8192 (fewer than 8 of the samples, where 30 are due) happens once in some
// hundred calls.  Beyond, it would become the rule.
constexpr int64_t kSampleSortRows = (int64_t)kMaxBuckets * 2176;

// Field widths of the packed key: column d takes bits(mx - mn); the first column is the most
// significant.
struct KeyLayout {
  uint32_t mn[4];
  uint32_t shift[4];
  uint32_t bits[4];
  uint32_t total;
};

struct UniqueHeader {  // first 1024 bytes of the workspace
  KeyLayout layout;
  int32_t count;                           // number of distinct rows
  int32_t buckets;                         // 0 where the keys do not fit 64 bits
  int32_t overflow;                        // 1: a bucket did not fit LDS
  int32_t large;                           // buckets listed for unique_bucket_large
  int32_t item_first[WCN_VOXEL_MAX_BATCH];  // first distinct row by value of column 0 (from its minimum)
  int32_t pad[175];
};
static_assert(sizeof(UniqueHeader) == 1024, "header is 1024 bytes");
static_assert(sizeof(KeyLayout) == 52, "the fields after the layout follow it");

struct UniqueView {
  UniqueHeader* hdr;
  int32_t* boxes;      // kBoxParts x 8: least and greatest value of every column
  uint64_t* bounds;    // kMaxBuckets - 1 bucket boundaries (words of the key's width)
  uint32_t* sizes;     // kMaxBuckets
  uint32_t* starts;    // kMaxBuckets + 1
  uint32_t* large;     // kMaxBuckets: the buckets for unique_bucket_large
  uint32_t* distinct;  // kMaxBuckets: distinct keys of every bucket
  unsigned long long* keys_a;
  unsigned long long* keys_b;
  uint32_t* idx_a;  // also: row in its part | bucket << 13
  uint32_t* idx_b;
  uint32_t* rank;  // inclusive count of segment heads; also: bucket counts of the parts
  void* temp;      // rocPRIM scratch
  size_t temp_bytes;
};

struct UniqueOut {
  int32_t* rows;    // (M, columns)
  int32_t* coords;  // (M, 3): columns 1..3 of 4
  int64_t* to_orig;
  int64_t* csr_indices;
  int64_t* csr_offsets;
  int64_t* to_unique;
};

template <typename KeyT>
struct HeadFlag {  // 1 where a sorted key differs from its predecessor
  const KeyT* keys;
  __device__ uint32_t operator()(uint32_t i) const {
    return (i == 0 || keys[i] != keys[i - 1]) ? 1u : 0u;
  }
};
template <typename KeyT>
using HeadIterator =
    rocprim::transform_iterator<rocprim::counting_iterator<uint32_t>, HeadFlag<KeyT>, uint32_t>;

// rocPRIM's default switches to a comparison merge sort below a million items, which ignores how
// few key bits are in use (160 us for a million 28-bit keys against four radix passes of ~10 us).
using SortConfig = rocprim::radix_sort_config<rocprim::default_config, rocprim::default_config,
                                              rocprim::default_config, 32768>;

template <typename KeyT>
size_t prim_temp_bytes_for(int64_t n) {
  size_t sort_bytes = 0, scan_bytes = 0;
  KeyT* k = nullptr;
  uint32_t* v = nullptr;
  (void)rocprim::radix_sort_pairs<SortConfig>(nullptr, sort_bytes, k, k, v, v, (size_t)n, 0u,
                                  (unsigned)(8 * sizeof(KeyT)), (hipStream_t)0);
  HeadIterator<KeyT> heads(rocprim::counting_iterator<uint32_t>(0), HeadFlag<KeyT>{nullptr});
  (void)rocprim::inclusive_scan(nullptr, scan_bytes, heads, v, (size_t)n, rocprim::plus<uint32_t>(),
                                (hipStream_t)0);
  return sort_bytes > scan_bytes ? sort_bytes : scan_bytes;
}

// (asked for several times in a call, of the same n)
size_t prim_temp_bytes(int64_t n) {
  static thread_local int64_t last_n = -1;
  static thread_local size_t last_bytes = 0;
  if (n == last_n) return last_bytes;
  const size_t a = prim_temp_bytes_for<unsigned long long>(n), b = prim_temp_bytes_for<uint32_t>(n);
  last_n = n;
  return last_bytes = a > b ? a : b;
}

size_t unique_layout(void* base, int64_t n, UniqueView* v) {
  char* p = (char*)base;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* at = p + off;
    off += wcn_align256(bytes);
    return at;
  };
  const size_t rows = (size_t)(n > 0 ? n : 1);
  UniqueView u;
  u.hdr = (UniqueHeader*)take(sizeof(UniqueHeader));
  u.boxes = (int32_t*)take(kBoxParts * 8 * sizeof(int32_t));
  u.bounds = (uint64_t*)take(kMaxBuckets * sizeof(uint64_t));
  u.sizes = (uint32_t*)take(kMaxBuckets * sizeof(uint32_t));
  u.starts = (uint32_t*)take((kMaxBuckets + 1) * sizeof(uint32_t));
  u.large = (uint32_t*)take(kMaxBuckets * sizeof(uint32_t));
  u.distinct = (uint32_t*)take(kMaxBuckets * sizeof(uint32_t));
  u.keys_a = (unsigned long long*)take(8 * rows);
  u.keys_b = (unsigned long long*)take(8 * rows);
  u.idx_a = (uint32_t*)take(4 * rows);
  u.idx_b = (uint32_t*)take(4 * rows);
  u.rank = (uint32_t*)take(4 * rows);
  u.temp_bytes = prim_temp_bytes((int64_t)rows);
  u.temp = take(u.temp_bytes > 0 ? u.temp_bytes : 256);
  if (v) *v = u;
  return off;
}

// ---- where the rows come from -------------------------------------------------------------------
// torch divides a float tensor by a host scalar as a multiplication with the scalar's reciprocal
// (taken in double, rounded to float); the product is floored and converted to int32 the same way.
typedef WcnItemStarts BatchStarts;

struct ItemHint {
  int item;       // of a row,
  int64_t until;  // the first row of the next item that has any
};

struct PointRows {  // row i = [batch item of point i, floor(p * inv)]
  const float* points;
  float inv;
  BatchStarts starts;
  int batch_size;
  const int64_t* device_starts;  // used instead of `starts` when there are too many batch items
  __device__ __forceinline__ int64_t start(int b) const {
    return device_starts ? device_starts[b] : starts.start[b];
  }
  __device__ __forceinline__ ItemHint hint(int64_t i) const {
    int lo = 0, hi = batch_size;  // the item lies in [lo, hi)
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (start(mid) <= i) lo = mid; else hi = mid;
    }
    return ItemHint{lo, start(lo + 1)};
  }
  // `from` belongs to a row at or before i: neighbours share one search.
  template <typename I>
  __device__ __forceinline__ void load(I i, const ItemHint& from, int v[4]) const {
    columns_of(i, v);
    int item = from.item;
    if ((int64_t)i >= from.until) item = hint((int64_t)i).item;
    v[0] = item;
  }
  // the columns whose box is not known from the first and the last row
  template <typename I>
  __device__ __forceinline__ void columns_of(I i, int v[4]) const {
    const float x = points[3 * i], y = points[3 * i + 1], z = points[3 * i + 2];
    v[1] = (int)floorf(x * inv);
    v[2] = (int)floorf(y * inv);
    v[3] = (int)floorf(z * inv);
  }
  static constexpr int kFirstBoxColumn = 1;
  __device__ __forceinline__ int columns() const { return 4; }
};

struct IntRows {  // (n, columns) int32, row-major
  const int32_t* rows;
  int ncol;
  __device__ __forceinline__ ItemHint hint(int64_t) const { return ItemHint{0, INT64_MAX}; }
  template <typename I>
  __device__ __forceinline__ void load(I i, const ItemHint&, int v[4]) const { columns_of(i, v); }
  template <typename I>
  __device__ __forceinline__ void columns_of(I i, int v[4]) const {
    if (ncol == 4) {
      const int4 r = reinterpret_cast<const int4*>(rows)[i];
      v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w;
    } else {
      v[0] = v[1] = v[2] = v[3] = 0;
      for (int d = 0; d < ncol; ++d) v[d] = rows[i * ncol + d];
    }
  }
  static constexpr int kFirstBoxColumn = 0;
  __device__ __forceinline__ int columns() const { return ncol; }
};

// One thread per point: 12 bytes read (lanes read adjacent words), one 16-byte row written.
__global__ void __launch_bounds__(256) voxel_rows(PointRows src, int64_t n, int4* __restrict__ rows) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int v[4];
  src.load(i, src.hint(i), v);
  rows[i] = make_int4(v[0], v[1], v[2], v[3]);
}

// The batch column put in front of integer coordinates: row i = [batch item of row i, c[i][0..dims)].
// One thread per row; with three spatial columns the row goes out as one 16-byte store.
__global__ void __launch_bounds__(256) batch_indexed_rows(const int32_t* __restrict__ coords, int64_t n,
                                                          int dims, BatchStarts starts, int batch_size,
                                                          int32_t* __restrict__ rows) {
  // the offsets arrive with the launch (scalar registers); lanes search them at different places,
  // so they are put into LDS first
  __shared__ int64_t s_start[WCN_VOXEL_MAX_BATCH + 1];
  if (threadIdx.x <= WCN_VOXEL_MAX_BATCH) s_start[threadIdx.x] = starts.start[threadIdx.x];
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int lo = wcn_item_of(s_start, batch_size, i);
  if (dims == 3) {
    const int32_t* c = coords + 3 * i;
    reinterpret_cast<int4*>(rows)[i] = make_int4(lo, c[0], c[1], c[2]);
  } else {
    int32_t* r = rows + i * (dims + 1);
    r[0] = lo;
    for (int d = 0; d < dims; ++d) r[d + 1] = coords[i * dims + d];
  }
}

// ---- bounding box, field widths, bucket boundaries ------------------------------------------------
__device__ __forceinline__ uint32_t scatter_bits(uint32_t x) {  // a bijection of 32-bit words
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  return x ^ (x >> 16);
}

// One row somewhere in each of `samples` equal stretches (rows in a regular order are sampled fairly too);
// `stretch` is their length, 32.32.
__device__ __forceinline__ uint32_t sampled_row(uint32_t k, uint64_t stretch) {
  const uint32_t from = (uint32_t)((uint64_t)k * stretch >> 32), to = (uint32_t)((uint64_t)(k + 1u) * stretch >> 32);
  return from + __umulhi(scatter_bits(k), to - from);
}

// Read-bound: eight rows in flight per thread.  Every workgroup leaves its box in memory (atomics of
// all workgroups on the same eight words are served one after the other) and collects its share of the
// sample: sixteen thousand rows from all over memory took the one compute unit of unique_split 45 us.
template <class Src>
__global__ void __launch_bounds__(1024) unique_box(Src src, int64_t n, int32_t* __restrict__ boxes, int samples,
                                                   uint64_t stretch, int4* __restrict__ sample) {
  for (int k = (int)(blockIdx.x + gridDim.x * threadIdx.x); k < samples; k += (int)(gridDim.x * blockDim.x)) {
    const int64_t i = sampled_row((uint32_t)k, stretch);
    int v[4];
    src.load(i, src.hint(i), v);
    sample[k] = make_int4(v[0], v[1], v[2], v[3]);
  }
  int mn[4] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MAX};
  int mx[4] = {INT32_MIN, INT32_MIN, INT32_MIN, INT32_MIN};
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += 8 * stride) {
    int v[8][4];
#pragma unroll
    for (int u = 0; u < 8; ++u) src.columns_of(i + u * stride < n ? i + u * stride : i, v[u]);
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int d = Src::kFirstBoxColumn; d < 4; ++d) {
        mn[d] = min(mn[d], v[u][d]);
        mx[d] = max(mx[d], v[u][d]);
      }
  }
  if (Src::kFirstBoxColumn > 0) {  // batch items ascend
    mn[0] = src.hint(0).item;
    mx[0] = src.hint(n - 1).item;
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) {
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
      mn[d] = min(mn[d], __shfl_xor(mn[d], s, 64));
      mx[d] = max(mx[d], __shfl_xor(mx[d], s, 64));
    }
  }
  __shared__ int part[16][8];
  if (wcn_lane() == 0) {
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      part[threadIdx.x >> 6][d] = mn[d];
      part[threadIdx.x >> 6][4 + d] = mx[d];
    }
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    const int d = threadIdx.x;
    int a = part[0][d];
    for (int w = 1; w < 16; ++w) a = d < 4 ? min(a, part[w][d]) : max(a, part[w][d]);
    boxes[blockIdx.x * 8 + d] = a;
  }
}

__device__ __forceinline__ KeyLayout key_layout(const int* box, int columns) {
  KeyLayout L;
  uint32_t at = 0;
#pragma unroll
  for (int d = 3; d >= 0; --d) {
    const uint32_t span = d < columns ? (uint32_t)box[4 + d] - (uint32_t)box[d] : 0u;
    L.mn[d] = d < columns ? (uint32_t)box[d] : 0u;
    L.bits[d] = span == 0 ? 0u : 32u - (uint32_t)__builtin_clz(span);
    L.shift[d] = d < columns ? at : 0u;
    at += L.bits[d];
  }
  L.total = at;
  return L;
}

__device__ __forceinline__ unsigned long long pack_key(const KeyLayout& L, const int v[4]) {
  unsigned long long key = 0;
#pragma unroll
  for (int d = 0; d < 4; ++d)
    if (L.bits[d] > 0)  // fields of width 0 stay out (their shift may be 64)
      key |= (unsigned long long)((uint32_t)v[d] - L.mn[d]) << L.shift[d];
  return key;
}

template <typename KeyT>
__device__ __forceinline__ KeyT pack_as(const KeyLayout& L, const int v[4]) {
  if (sizeof(KeyT) == 8) return (KeyT)pack_key(L, v);
  uint32_t key = 0;  // a shift of 32 (of a field of width 0, which is 0) counts as none
#pragma unroll
  for (int d = 0; d < 4; ++d) key |= ((uint32_t)v[d] - L.mn[d]) << (L.shift[d] & 31u);
  return (KeyT)key;
}

__device__ __forceinline__ int key_field(const KeyLayout& L, unsigned long long key, int d) {
  return L.bits[d] == 0 ? 0 : (int)((key >> L.shift[d]) & ((1ull << L.bits[d]) - 1ull));
}

__device__ __forceinline__ void write_row(const KeyLayout& L, unsigned long long key, int columns, int64_t u,
                                          const UniqueOut& out) {
  int32_t field[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) field[d] = (int32_t)((uint32_t)key_field(L, key, d) + L.mn[d]);
  if (out.rows) {
    if (columns == 4) {
      reinterpret_cast<int4*>(out.rows)[u] = make_int4(field[0], field[1], field[2], field[3]);
    } else {
      for (int d = 0; d < columns; ++d) out.rows[u * columns + d] = field[d];
    }
  }
  if (out.coords) {
#pragma unroll
    for (int d = 0; d < 3; ++d) out.coords[3 * u + d] = field[d + 1];
  }
}

// The order of keys in LDS, by a trie: a level takes up to five more of the keys' bits.  Keys with
// the same leading bits share an entry, a 32-bit mask of the values its next five bits take;
// the prefix sum of the masks' populations numbers the entries of the next level, in key order.  The first
// level's entries are the leading log2(ENTRIES) bits themselves, so the 2^18 values a bucket of voxels spans
// are through in one level, and every further level costs the same whatever the keys: no
// comparison sort, no passes over digits that are all alike.
template <int ENTRIES>
struct Trie {
  alignas(16) uint32_t mask[ENTRIES];
  alignas(16) uint16_t before[ENTRIES];
  uint32_t wave[16];
};

// before[e] = sum of mask's populations (POP) or values over the entries below e; returns the total.
// Four entries a thread and turn; the masks are complete up to a multiple of 4 (barrier passed),
// `before` is complete on return.
template <int THREADS, bool POP, int ENTRIES>
__device__ __forceinline__ int trie_scan(Trie<ENTRIES>& T, int entries) {
  const int t = threadIdx.x, w = t >> 6;
  int total = 0;
  for (int e0 = 0; e0 < entries; e0 += 4 * THREADS) {
    const int e = e0 + 4 * t;
    uint4 m = make_uint4(0, 0, 0, 0);
    if (e < entries) m = *reinterpret_cast<const uint4*>(&T.mask[e]);
    const int c0 = POP ? __popc(m.x) : (int)m.x, c1 = POP ? __popc(m.y) : (int)m.y;
    const int c2 = POP ? __popc(m.z) : (int)m.z, c3 = POP ? __popc(m.w) : (int)m.w;
    const int inclusive = wcn_wave_inclusive_sum(c0 + c1 + c2 + c3);
    if (e0 > 0) __syncthreads();  // the last turn's sums have been read
    if (wcn_lane() == 63) T.wave[w] = (uint32_t)inclusive;
    __syncthreads();
    int v = (int)T.wave[wcn_lane() & (THREADS / 64 - 1)];
    v = wcn_lane() < THREADS / 64 ? v : 0;
    const int upto = wcn_wave_inclusive_sum(v);
    const int base = total + (w == 0 ? 0 : __builtin_amdgcn_readlane(upto, w == 0 ? 0 : __builtin_amdgcn_readfirstlane(w) - 1));
    total += __builtin_amdgcn_readlane(upto, THREADS / 64 - 1);
    if (e < entries) {
      const uint32_t b0 = (uint32_t)(base + inclusive - c0 - c1 - c2 - c3);
      const uint32_t b1 = b0 + c0, b2 = b1 + c1, b3 = b2 + c2;
      *reinterpret_cast<uint2*>(&T.before[e]) = make_uint2(b0 | b1 << 16, b2 | b3 << 16);
    }
  }
  __syncthreads();
  return total;
}

// Item j of a thread is the keys' number threadIdx.x + THREADS * j; those at or beyond n are copies of others.
// place[j]: its entry, before and after.
template <int THREADS, int ENTRIES, int PER, typename KeyT>
__device__ __forceinline__ int trie_level(Trie<ENTRIES>& T, int entries, int n, const KeyT (&key)[PER],
                                          int shift, int bits, uint32_t (&place)[PER]) {
  const int t = threadIdx.x;
  const uint32_t low = (1u << bits) - 1u;
  __syncthreads();
  for (int e = 4 * t; e < entries; e += 4 * THREADS) *reinterpret_cast<uint4*>(&T.mask[e]) = make_uint4(0, 0, 0, 0);
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (t + THREADS * j < n) atomicOr(&T.mask[place[j]], 1u << ((uint32_t)(key[j] >> shift) & low));
  __syncthreads();
  const int total = trie_scan<THREADS, true>(T, entries);
  // every lane reads, also for the items it does not have (any entry will do): all reads are in flight together
  uint32_t before[PER], mask[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    before[j] = T.before[place[j]];
    mask[j] = T.mask[place[j]];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t sub = (uint32_t)(key[j] >> shift) & low;
    place[j] = before[j] + (uint32_t)__popc(mask[j] & ((1u << sub) - 1u));
  }
  return total;
}

// place[j] becomes the number of distinct keys below key j; returns the number of distinct keys.
// 2^LOG entries to begin with.
template <int THREADS, int LOG, int ENTRIES, int PER, typename KeyT>
__device__ __forceinline__ int trie_order(Trie<ENTRIES>& T, int n, const KeyT (&key)[PER], int bits,
                                          uint32_t (&place)[PER]) {
  static_assert(ENTRIES >= 1 << LOG && ENTRIES >= THREADS * PER, "entries");
  int shift = bits > LOG ? bits - LOG : 0;
  int entries = 1 << (bits < LOG ? bits : LOG);
#pragma unroll
  for (int j = 0; j < PER; ++j) place[j] = (uint32_t)(key[j] >> shift);
  do {
    const int take = shift < 5 ? shift : 5;
    shift -= take;
    entries = trie_level<THREADS>(T, entries, n, key, shift, take, place);
  } while (shift > 0);
  return entries;
}

template <typename KeyT>
__device__ __forceinline__ int split_rows(const int4* __restrict__ sample, int buckets, const KeyLayout& L,
                                          Trie<kMaxSamples>& T, KeyT* pick, KeyT* __restrict__ bounds) {
  constexpr int PER = kMaxSamples / 1024;
  const int t = threadIdx.x, samples = buckets * kSamplesPerBucket;
  KeyT key[PER];
  uint32_t place[PER];
#pragma unroll
  for (int j0 = 0; j0 < PER; j0 += 8) {
    int4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = sample[t + 1024 * (j0 + j) < samples ? t + 1024 * (j0 + j) : samples - 1];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
      key[j0 + j] = pack_as<KeyT>(L, row);
    }
  }
  const int distinct = trie_order<1024, 14>(T, samples, key, (int)L.total, place);
  // sorted positions: equal keys in any order
  __syncthreads();
  for (int e = 4 * t; e < distinct; e += 4096) *reinterpret_cast<uint4*>(&T.mask[e]) = make_uint4(0, 0, 0, 0);
  __syncthreads();
  uint32_t nth[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (t + 1024 * j < samples) nth[j] = atomicAdd(&T.mask[place[j]], 1u);
  __syncthreads();
  trie_scan<1024, false>(T, distinct);
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (t + 1024 * j < samples) {
      const int at = (int)(T.before[place[j]] + nth[j]);
      if (at > 0 && at % kSamplesPerBucket == 0) pick[at / kSamplesPerBucket - 1] = key[j];
    }
  __syncthreads();
  // A boundary for every distinct pick and, behind a key that was picked twice (it fills a bucket), a second
  // one that closes it: never more boundaries than picks.
  const int picks = buckets - 1;
  const KeyT last = L.total >= 8 * sizeof(KeyT) ? (KeyT)~(KeyT)0 : (KeyT)(((KeyT)1 << L.total) - 1);
  int emits[2], sum = 0;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int i = 2 * t + k;
    const bool first = i < picks && (i == 0 || pick[i] != pick[i - 1]);
    const bool heavy = first && i + 1 < picks && pick[i + 1] == pick[i] && pick[i] != last;
    emits[k] = (first ? 1 : 0) + (heavy ? 1 : 0);
    sum += emits[k];
  }
  const int inclusive = wcn_wave_inclusive_sum(sum);
  if (wcn_lane() == 63) T.wave[t >> 6] = (uint32_t)inclusive;
  __syncthreads();
  int at = inclusive - sum, total = 0;
  for (int i = 0; i < 16; ++i) {
    at += i < (t >> 6) ? (int)T.wave[i] : 0;
    total += (int)T.wave[i];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    if (emits[k] > 0) bounds[at] = pick[2 * t + k];
    if (emits[k] > 1) bounds[at + 1] = pick[2 * t + k] + 1;
    at += emits[k];
  }
  return total + 1;
}

// One workgroup.  Bound by its own latencies: the trie's levels (three for 28-bit keys).
__global__ void __launch_bounds__(1024) unique_split(const int32_t* __restrict__ boxes, int num_boxes,
                                                     const int4* __restrict__ sample, int columns, int buckets,
                                                     UniqueHeader* __restrict__ h,
                                                     uint64_t* __restrict__ bounds) {
  __shared__ Trie<kMaxSamples> T;
  __shared__ uint64_t pick[kMaxBuckets];
  __shared__ int box[8];
  const int t = threadIdx.x, w = t >> 6;
  if (w < 8) {
    int a = w < 4 ? INT32_MAX : INT32_MIN;
    for (int i = wcn_lane(); i < num_boxes; i += 64) a = w < 4 ? min(a, boxes[8 * i + w]) : max(a, boxes[8 * i + w]);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
      const int o = __shfl_xor(a, s, 64);
      a = w < 4 ? min(a, o) : max(a, o);
    }
    if (wcn_lane() == 0) box[w] = a;
  }
  if (t < WCN_VOXEL_MAX_BATCH) h->item_first[t] = INT32_MAX;
  __syncthreads();
  const KeyLayout L = key_layout(box, columns);
  int made = 1;
  if (L.total > 64u)
    made = 0;
  else if (buckets > 1)
    made = L.total <= 32u ? split_rows<uint32_t>(sample, buckets, L, T, (uint32_t*)pick, (uint32_t*)bounds)
                          : split_rows<uint64_t>(sample, buckets, L, T, pick, bounds);
  if (t == 0) {
    h->layout = L;
    h->count = 0;
    h->buckets = made;
    h->overflow = 0;
    h->large = 0;
  }
}

// Successive workgroups go to the eight dies in turn.  A die gets a stretch of successive parts: their
// runs in a bucket are neighbours, and their lines are put together in its own L2.
__device__ __forceinline__ int part_of_block(int block, int parts) {
  const int die = block & 7, each = parts >> 3, extra = parts & 7;
  return die * each + (die < extra ? die : extra) + (block >> 3);
}

// ---- distribution into buckets --------------------------------------------------------------------
// A wave walks 1024 successive rows, 64 at a time.  The wave's own counter of the bucket (LDS) gives the
// rows before them; lanes of one bucket show up when every lane leaves its number at the bucket and reads it
// back, and are ranked one bucket after the other (of 64 rows in no order two meet once in a while; of
// rows in order many do, in few buckets).  So the place is stable, without atomics.  The part's rows then go
// to memory in the order of their buckets, for unique_place to write runs and not single words.
// Bound by the search (11 dependent LDS reads a row, four rows in flight) and its vector instructions.
struct AssignLds {
  union {
    struct {
      uint64_t bounds[kMaxBuckets];
      uint16_t count[8][kMaxBuckets];
      uint8_t lane[8][kMaxBuckets];
    };
    uint32_t staged[kPartRows];
  };
  uint32_t wave[8];
};

// What the wave's lanes wrote to LDS before is there for what they read behind this (no instruction: a wave's LDS
// accesses are in order; the compiler may not hand a lane its own store back, or swap the two).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int STEPS, class Src, typename KeyT>
__device__ __forceinline__ void assign_rows(const Src& src, int64_t n, const KeyLayout& L, int buckets, int stride,
                                            int part, AssignLds& S, const KeyT* __restrict__ bounds,
                                            KeyT* __restrict__ keys, uint32_t* __restrict__ places,
                                            uint32_t* __restrict__ counts) {
  constexpr int ROWS = kPartRows / 512;
  const int t = threadIdx.x, w = t >> 6, lane = wcn_lane();
  const int cuts = buckets - 1;
  KeyT* s_bounds = (KeyT*)S.bounds;
  // the boundaries as a search tree, level after level from entry 1 (in sorted order the upper levels' nodes
  // are multiples of 32 words apart, all in one bank); leaves without a boundary are never passed
  for (int i = t + 1; i < 1 << STEPS; i += 512) {
    const int level = 31 - __builtin_clz((unsigned)i);
    const int at = ((2 * (i - (1 << level)) + 1) << (STEPS - 1 - level)) - 1;
    s_bounds[i] = at < cuts ? bounds[at] : (KeyT)~(KeyT)0;
  }
  for (int i = t; i < 8 * kMaxBuckets / 2; i += 512) reinterpret_cast<uint32_t*>(S.count)[i] = 0;
  __syncthreads();
  const uint32_t last = (uint32_t)n - 1u, part_first = (uint32_t)part * kPartRows;
  const uint32_t wave_first = part_first + (uint32_t)__builtin_amdgcn_readfirstlane(w) * (64 * ROWS);
  const ItemHint from = src.hint(wave_first < last ? wave_first : last);
  const unsigned long long below = (1ull << lane) - 1ull;
  uint16_t* s_count = S.count[w];
  uint8_t* s_lane = S.lane[w];
  uint32_t packed[ROWS];
  KeyT key[ROWS];
#pragma unroll
  for (int r0 = 0; r0 < ROWS; r0 += 4) {
    int v[4][4];
    uint32_t pos[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t i = wave_first + 64u * (r0 + r) + lane;
      src.load(i < last ? i : last, from, v[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      key[r0 + r] = pack_as<KeyT>(L, v[r]);
      pos[r] = 1;
    }
#pragma unroll
    for (int step = 0; step < STEPS; ++step) {
      KeyT b[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = s_bounds[pos[r]];
#pragma unroll
      for (int r = 0; r < 4; ++r) pos[r] = 2u * pos[r] + (b[r] <= key[r0 + r] ? 1u : 0u);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) pos[r] -= 1u << STEPS;  // boundaries at or below the key
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint32_t d = pos[r] < (uint32_t)cuts ? pos[r] : (uint32_t)cuts;
      const bool live = wave_first + 64u * (r0 + r) + lane <= last;
      int rank = 0, together = 1;
      if (live) s_lane[d] = (uint8_t)lane;
      wave_lds_order();
      const uint32_t before = s_count[d];
      unsigned long long met = __ballot(live && s_lane[d] != (uint8_t)lane);
      while (met != 0) {
        const uint32_t shared = __builtin_amdgcn_readlane(d, __ffsll((long long)met) - 1);
        const unsigned long long same = __ballot(live && d == shared);
        if (d == shared) {
          rank = __popcll(same & below);
          together = __popcll(same);
        }
        met &= ~same;
      }
      wave_lds_order();  // every lane has read both words
      if (live && rank == 0) s_count[d] = (uint16_t)(before + (uint32_t)together);
      packed[r0 + r] = d | (before + (uint32_t)rank) << 16;
    }
  }
  __syncthreads();
  // the waves' counts -> the rows of the part before the wave; the buckets' counts -> the part's order
  uint32_t total[4], sum = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int b = 4 * t + k;
    total[k] = 0;
    if (b < buckets) {
      uint32_t run = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) run += S.count[i][b];
      total[k] = run;
      counts[(int64_t)part * stride + b] = run;
    }
    sum += total[k];
  }
  const uint32_t inclusive = (uint32_t)wcn_wave_inclusive_sum((int)sum);
  if (lane == 63) S.wave[w] = inclusive;
  __syncthreads();
  uint32_t at = inclusive - sum;
  for (int i = 0; i < w; ++i) at += S.wave[i];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int b = 4 * t + k;
    if (b < buckets) {
      uint32_t run = at;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t c = S.count[i][b];
        S.count[i][b] = (uint16_t)run;
        run += c;
      }
    }
    at += total[k];
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {  // packed: place in the part's order | bucket << 16
    const uint32_t d = packed[r] & 0xffffu;
    packed[r] = (uint32_t)(s_count[d] + (packed[r] >> 16)) | d << 16;
  }
  const uint32_t live_rows = last - part_first + 1u < (uint32_t)kPartRows ? last - part_first + 1u : (uint32_t)kPartRows;
#pragma unroll
  for (int word = 0; word < 1 + (int)sizeof(KeyT) / 4; ++word) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const uint32_t i = 64u * (ROWS * w + r) + lane;  // in the part
      const uint32_t value = word == 0 ? i | packed[r] >> 16 << 13
                                       : (uint32_t)(word == 1 ? (uint64_t)key[r] : (uint64_t)key[r] >> 32);
      if (i < live_rows) S.staged[packed[r] & 0xffffu] = value;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const uint32_t q = t + 512u * r;
      if (q >= live_rows) continue;
      if (word == 0)
        places[part_first + q] = S.staged[q];
      else
        reinterpret_cast<uint32_t*>(keys)[(uint64_t)(part_first + q) * (sizeof(KeyT) / 4) + (word - 1)] = S.staged[q];
    }
  }
}

template <class Src>
__global__ void __launch_bounds__(512) unique_assign(Src src, int64_t n, const UniqueHeader* __restrict__ h,
                                                     int stride, const uint64_t* __restrict__ bounds,
                                                     void* __restrict__ keys, uint32_t* __restrict__ places,
                                                     uint32_t* __restrict__ counts) {
  __shared__ AssignLds S;
  const int buckets = h->buckets;
  if (buckets == 0) return;
  const int part = part_of_block((int)blockIdx.x, (int)gridDim.x);
  const KeyLayout L = h->layout;
  if (L.total > 32u)
    assign_rows<11, Src, uint64_t>(src, n, L, buckets, stride, part, S, bounds, (uint64_t*)keys, places, counts);
  else if (buckets > 128)
    assign_rows<11, Src, uint32_t>(src, n, L, buckets, stride, part, S, (const uint32_t*)bounds, (uint32_t*)keys,
                                   places, counts);
  else
    assign_rows<7, Src, uint32_t>(src, n, L, buckets, stride, part, S, (const uint32_t*)bounds, (uint32_t*)keys,
                                  places, counts);
}

// counts (parts, stride): every column becomes its exclusive prefix sum, the totals go to sizes.  A
// workgroup takes 32 columns (a line) and deals the parts to its 32 half waves.
__global__ void __launch_bounds__(1024) unique_columns(const UniqueHeader* __restrict__ h, int parts, int stride,
                                                       uint32_t* __restrict__ counts, uint32_t* __restrict__ sizes) {
  __shared__ uint32_t s_sum[32][32];
  const int g = threadIdx.x >> 5, lane = threadIdx.x & 31;
  const int column = (int)blockIdx.x * 32 + lane;
  const bool live = column < h->buckets;
  const int each = (parts + 31) / 32;
  const int begin = g * each < parts ? g * each : parts, end = begin + each < parts ? begin + each : parts;
  uint32_t* at = counts + (live ? column : 0);
  uint32_t sum = 0;
#pragma unroll 8
  for (int p = begin; p < end; ++p) sum += at[(int64_t)p * stride];
  s_sum[g][lane] = sum;
  __syncthreads();
  uint32_t run = 0;
  for (int i = 0; i < g; ++i) run += s_sum[i][lane];
  if (!live) return;
  if (g == 31) sizes[column] = run + sum;
  for (int p0 = begin; p0 < end; p0 += 8) {
    uint32_t c[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) c[k] = at[(int64_t)(p0 + k < end ? p0 + k : end - 1) * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (p0 + k < end) {
        at[(int64_t)(p0 + k) * stride] = run;
        run += c[k];
      }
  }
}

constexpr int kSmallThreads = 512, kSmallPer = 6;  // of unique_bucket

// The least and the greatest key of a bucket.
__device__ __forceinline__ unsigned long long bucket_first(const KeyLayout& L, const uint64_t* bounds, int b) {
  return b == 0 ? 0ull : L.total <= 32u ? reinterpret_cast<const uint32_t*>(bounds)[b - 1] : bounds[b - 1];
}
__device__ __forceinline__ unsigned long long bucket_last(const KeyLayout& L, const uint64_t* bounds, int b, int buckets) {
  if (b < buckets - 1) return bucket_first(L, bounds, b + 1) - 1ull;
  return L.total >= 64u ? ~0ull : (1ull << L.total) - 1ull;
}

// A workgroup per part, on the die that made its keys.  The starts of the buckets and of the part's
// runs are summed up by every workgroup for itself (2048 words each).  Bound by the requests of the
// scattered runs: four rows are 32 successive bytes.
template <typename KeyT>
__device__ __forceinline__ void place_rows(uint32_t first, uint32_t n, const uint32_t* s_base,
                                           const KeyT* __restrict__ keys, const uint32_t* __restrict__ places,
                                           void* __restrict__ keys_out, uint32_t* __restrict__ rows_out) {
  constexpr int PER = kPartRows / 1024;
  uint32_t place[PER];
  KeyT key[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t q = threadIdx.x + 1024u * j, i = first + q < n ? first + q : n - 1u;
    place[j] = places[i];
    key[j] = keys[i];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const uint32_t q = threadIdx.x + 1024u * j;
    if (first + q >= n) continue;
    const uint32_t at = s_base[place[j] >> 13] + q, row = first + (place[j] & 8191u);
    if (sizeof(KeyT) == 4) {
      reinterpret_cast<uint2*>(keys_out)[at] = make_uint2((uint32_t)key[j], row);
    } else {
      reinterpret_cast<KeyT*>(keys_out)[at] = key[j];
      rows_out[at] = row;
    }
  }
}
static_assert(kPartRows == 8192, "13 bits of a place");

// Rows and keys that unique_bucket leaves to unique_bucket_large.
__device__ __forceinline__ bool large_bucket(const UniqueHeader* h, const uint64_t* bounds, int b, int buckets,
                                             uint32_t size) {
  const unsigned long long span = bucket_last(h->layout, bounds, b, buckets) - bucket_first(h->layout, bounds, b);
  return size > 0 && span > 0 && (size > (uint32_t)(kSmallThreads * kSmallPer) || (span >> 32) != 0);
}

__global__ void __launch_bounds__(1024) unique_place(int64_t n, UniqueHeader* __restrict__ h, int stride,
                                                     const uint64_t* __restrict__ bounds,
                                                     uint32_t* __restrict__ large,
                                                     const uint32_t* __restrict__ sizes,
                                                     const uint32_t* __restrict__ counts,
                                                     const void* __restrict__ keys,
                                                     const uint32_t* __restrict__ places,
                                                     uint32_t* __restrict__ starts, void* __restrict__ keys_out,
                                                     uint32_t* __restrict__ rows_out) {
  __shared__ uint32_t s_base[kMaxBuckets];
  __shared__ uint32_t s_wave[16], s_own[16];
  const int buckets = h->buckets;
  if (buckets == 0) return;
  const int parts = (int)gridDim.x, part = part_of_block((int)blockIdx.x, parts);
  const int t = threadIdx.x, w = t >> 6;
  uint32_t size[2], mine[2], own[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int b = 2 * t + k < buckets ? 2 * t + k : buckets - 1;
    size[k] = sizes[b];
    mine[k] = counts[(int64_t)part * stride + b];
    own[k] = counts[(int64_t)(part + 1 < parts ? part + 1 : part) * stride + b];
    own[k] = (part + 1 < parts ? own[k] : size[k]) - mine[k];
    size[k] = 2 * t + k < buckets ? size[k] : 0u;
  }
  const uint32_t inclusive = (uint32_t)wcn_wave_inclusive_sum((int)(size[0] + size[1]));
  const uint32_t own_inclusive = (uint32_t)wcn_wave_inclusive_sum((int)(own[0] + own[1]));
  if (wcn_lane() == 63) {
    s_wave[w] = inclusive;
    s_own[w] = own_inclusive;
  }
  __syncthreads();
  uint32_t run = inclusive - size[0] - size[1], own_run = own_inclusive - own[0] - own[1];
  for (int i = 0; i < w; ++i) {
    run += s_wave[i];
    own_run += s_own[i];
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int b = 2 * t + k;
    if (b < buckets) {
      if (part == 0) {
        starts[b] = run;
        // few (one in ten): listed, because a workgroup each that finds nothing to do took longer than they do
        if (large_bucket(h, bounds, b, buckets, size[k])) large[atomicAdd(&h->large, 1)] = (uint32_t)b;
      }
      s_base[b] = run + mine[k] - own_run;
    }
    run += size[k];
    own_run += own[k];
  }
  if (part == 0 && t == 0) starts[buckets] = (uint32_t)n;
  __syncthreads();
  const uint32_t first = (uint32_t)part * kPartRows;
  if (h->layout.total <= 32u)
    place_rows<uint32_t>(first, (uint32_t)n, s_base, (const uint32_t*)keys, places, keys_out, rows_out);
  else
    place_rows<uint64_t>(first, (uint32_t)n, s_base, (const uint64_t*)keys, places, keys_out, rows_out);
}

// ---- inside the buckets ---------------------------------------------------------------------------
// What a workgroup knows of its bucket.
struct Bucket {
  int index, count;             // which one, of how many
  uint32_t start, size;         // its rows
  unsigned long long lo, last;  // its range of keys
};

template <class Src>
struct BucketArgs {
  Src src;
  int64_t n;
  const uint64_t* bounds;
  const uint32_t* starts;
  const uint32_t* large;  // h->large buckets for unique_bucket_large
  void* keys;  // pairs (key, row) for keys of 32 bits, keys otherwise; with to_orig, left behind: (number of the key, row)
  const uint32_t* rows;
  void* head_key;       // by bucket start + number of the key: the key,
  uint32_t* head_row;   // its first row,
  uint32_t* head_at;    // and where its rows begin in csr_indices
  uint32_t* distinct;   // per bucket
  UniqueHeader* h;
  int64_t* csr_indices;
  bool want_orig;
};

// Word: what the keys' distances from the bucket's least one fit into.  DIRECT: one bucket, its keys made here.
template <class Src, bool DIRECT, bool PAIRS, typename Word, int THREADS, int PER, int LOG, int ENTRIES>
__device__ __forceinline__ void bucket_rows(const BucketArgs<Src>& A, const Bucket& B, const KeyLayout& L,
                                            Trie<ENTRIES>& T) {
  const int t = threadIdx.x, n = (int)B.size;
  auto at = [&](int j) { return t + THREADS * j < n ? t + THREADS * j : n - 1; };
  Word key[PER];
  uint32_t place[PER], number[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (DIRECT) {
      int v[4];
      A.src.load((int64_t)at(j), A.src.hint(at(j)), v);
      key[j] = (Word)pack_key(L, v);
    } else if (PAIRS) {
      key[j] = (Word)(reinterpret_cast<const uint2*>(A.keys)[B.start + at(j)].x - (uint32_t)B.lo);
    } else {
      key[j] = (Word)(reinterpret_cast<const uint64_t*>(A.keys)[B.start + at(j)] - B.lo);
    }
  }
  const unsigned long long span = B.last - B.lo;
  const int distinct = trie_order<THREADS, LOG>(T, n, key, 64 - __builtin_clzll(span), place);
  if (t == 0) A.distinct[B.index] = (uint32_t)distinct;
  // the rows of a key in their order: the trie goes on over the positions in the bucket
  uint32_t row[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    number[j] = place[j];
    row[j] = (uint32_t)at(j);
  }
  int entries = distinct, shift = 32 - __builtin_clz((unsigned)n);
  while (shift > 0 && entries < n) {
    const int take = shift < 5 ? shift : 5;
    shift -= take;
    entries = trie_level<THREADS>(T, entries, n, row, shift, take, place);
  }
#pragma unroll
  for (int j = 0; j < PER; ++j)
    row[j] = DIRECT ? (uint32_t)at(j)
             : PAIRS ? reinterpret_cast<const uint2*>(A.keys)[B.start + at(j)].y
                     : A.rows[B.start + at(j)];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (t + THREADS * j < n) {
      T.mask[place[j]] = row[j];
      T.before[place[j]] = (uint16_t)number[j];
    }
  __syncthreads();
  // from here a thread has the places t + THREADS * j of the sorted order: what it writes lies side by side
  bool head[PER];
  uint32_t previous[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    row[j] = T.mask[at(j)];
    number[j] = T.before[at(j)];
    previous[j] = T.before[at(j) > 0 ? at(j) - 1 : 0];
  }
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int q = t + THREADS * j;
    head[j] = q < n && (q == 0 || previous[j] != number[j]);  // the first row of its key
    if (q < n) {
      if (A.csr_indices) A.csr_indices[B.start + q] = row[j];
      if (A.want_orig) reinterpret_cast<uint2*>(A.keys)[B.start + q] = make_uint2(number[j], row[j]);
    }
    if (head[j]) {
      A.head_row[B.start + number[j]] = row[j];
      A.head_at[B.start + number[j]] = B.start + q;
    }
  }
  Word sorted[PER];
#pragma unroll
  for (int half = 0; half < (int)sizeof(Word) / 4; ++half) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if (t + THREADS * j < n) T.mask[place[j]] = (uint32_t)((uint64_t)key[j] >> (32 * half));
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PER; ++j)
      sorted[j] = (half ? sorted[j] : (Word)0) | (Word)((uint64_t)T.mask[at(j)] << (32 * half));
  }
#pragma unroll
  for (int j = 0; j < PER; ++j)
    if (head[j]) {
      const unsigned long long full = B.lo + (unsigned long long)sorted[j];
      if (PAIRS)
        reinterpret_cast<uint32_t*>(A.head_key)[B.start + number[j]] = (uint32_t)full;
      else
        reinterpret_cast<uint64_t*>(A.head_key)[B.start + number[j]] = full;
    }
}

// Rows that are all alike, any number of them.
template <class Src, bool DIRECT, int THREADS>
__device__ __forceinline__ void bucket_of_one(const BucketArgs<Src>& A, const Bucket& B, const KeyLayout& L) {
  const bool pairs = L.total <= 32u;
  for (uint32_t p = threadIdx.x; p < B.size; p += THREADS) {
    const uint32_t r = DIRECT ? p
                       : pairs ? reinterpret_cast<const uint2*>(A.keys)[B.start + p].y
                               : A.rows[B.start + p];
    if (A.csr_indices) A.csr_indices[B.start + p] = r;
    if (A.want_orig) reinterpret_cast<uint2*>(A.keys)[B.start + p] = make_uint2(0u, r);
    if (p == 0) {
      A.distinct[B.index] = 1;
      A.head_row[B.start] = r;
      A.head_at[B.start] = B.start;
      if (pairs)
        reinterpret_cast<uint32_t*>(A.head_key)[B.start] = (uint32_t)B.lo;
      else
        reinterpret_cast<uint64_t*>(A.head_key)[B.start] = B.lo;
    }
  }
}

template <class Src>
__device__ __forceinline__ bool take_bucket(const BucketArgs<Src>& A, const KeyLayout& L, int index, Bucket* B) {
  B->count = A.h->buckets;
  B->index = index;
  if (B->index >= B->count) return false;
  B->start = B->count == 1 ? 0u : A.starts[B->index];
  B->size = B->count == 1 ? (uint32_t)A.n : A.starts[B->index + 1] - B->start;
  B->lo = bucket_first(L, A.bounds, B->index);
  B->last = bucket_last(L, A.bounds, B->index, B->count);
  return true;
}

// A workgroup per bucket, four to a compute unit (24 KB of LDS, 64 registers).  Bound by the barriers and the
// LDS round trips of the levels, one or two for the keys of a bucket and two or three for its positions: many small
// workgroups hide them in one another.  (One kernel with the numbers of the keys by look-back from
// bucket to bucket waited for its slowest neighbours: 112 us for 4 M rows, against 35 + 18 + 20.)
// Buckets of more rows, and of keys that span more than 32 bits, are the next kernel's.
template <class Src>
__global__ void __launch_bounds__(kSmallThreads, 8) unique_bucket(BucketArgs<Src> A) {
  __shared__ Trie<4096> T;
  const KeyLayout L = A.h->layout;
  Bucket B;
  if (!take_bucket(A, L, (int)blockIdx.x, &B)) return;
  const unsigned long long span = B.last - B.lo;
  if (B.size == 0) {
    if (threadIdx.x == 0) A.distinct[B.index] = 0;
  } else if (span == 0) {
    bucket_of_one<Src, false, kSmallThreads>(A, B, L);
  } else if (B.size <= kSmallThreads * kSmallPer && (span >> 32) == 0) {
    if (L.total <= 32u)
      bucket_rows<Src, false, true, uint32_t, kSmallThreads, kSmallPer, 12>(A, B, L, T);
    else
      bucket_rows<Src, false, false, uint32_t, kSmallThreads, kSmallPer, 12>(A, B, L, T);
  }
}

template <class Src, bool DIRECT>
__global__ void __launch_bounds__(1024) unique_bucket_large(BucketArgs<Src> A) {
  __shared__ Trie<kBucketCap> T;
  const KeyLayout L = A.h->layout;
  const int listed = DIRECT ? 1 : A.h->large;
  for (int i = (int)blockIdx.x; i < listed; i += (int)gridDim.x) {
    Bucket B;
    if (!take_bucket(A, L, DIRECT ? 0 : (int)A.large[i], &B)) return;
    const unsigned long long span = B.last - B.lo;
    if (DIRECT && span == 0) {
      bucket_of_one<Src, true, 1024>(A, B, L);
    } else if (B.size > (uint32_t)kBucketCap) {  // the host sorts in another way then
      if (threadIdx.x == 0) {
        A.h->overflow = 1;
        A.distinct[B.index] = 0;
      }
    } else if (span >> 32) {
      bucket_rows<Src, DIRECT, false, uint64_t, 1024, 8, 13>(A, B, L, T);
    } else if (L.total > 32u) {
      bucket_rows<Src, DIRECT, false, uint32_t, 1024, 8, 13>(A, B, L, T);
    } else if (B.size <= 4096u) {  // nine in ten of these buckets
      bucket_rows<Src, DIRECT, true, uint32_t, 1024, 4, 12>(A, B, L, T);
    } else {
      bucket_rows<Src, DIRECT, true, uint32_t, 1024, 8, 13>(A, B, L, T);
    }
  }
}

// Per bucket: the number of distinct keys in front of it, and the results that need it.
template <class Src>
__global__ void __launch_bounds__(256) unique_finish(BucketArgs<Src> A, int columns, UniqueOut out) {
  __shared__ uint32_t s_sum[4];
  const KeyLayout L = A.h->layout;
  Bucket B;
  if (!take_bucket(A, L, (int)blockIdx.x, &B)) return;
  const int t = threadIdx.x;
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < kMaxBuckets / 256; ++k) {
    const int i = t + 256 * k;
    const uint32_t d = A.distinct[i < B.index ? i : 0];
    sum += i < B.index ? d : 0u;
  }
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readlane(wcn_wave_inclusive_sum((int)sum), 63);
  if (wcn_lane() == 0) s_sum[t >> 6] = wave;
  __syncthreads();
  const int64_t base = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
  const int distinct = (int)A.distinct[B.index];
  if (B.index == B.count - 1 && t == 0) {
    A.h->count = (int32_t)(base + distinct);
    if (out.csr_offsets) out.csr_offsets[base + distinct] = A.n;
  }
  auto head = [&](int u) -> unsigned long long {
    return L.total <= 32u ? reinterpret_cast<const uint32_t*>(A.head_key)[B.start + u]
                          : reinterpret_cast<const uint64_t*>(A.head_key)[B.start + u];
  };
  // the key in front of the bucket's first: two thousand workgroups that all report their first key's
  // item are served one after the other (20 us)
  const int earlier = B.index > 0 ? (int)A.distinct[B.index - 1] : 0;
  const bool known = earlier > 0;
  unsigned long long before = 0;
  if (known) before = head((int)A.starts[B.index - 1] - (int)B.start + earlier - 1);
  for (int u = t; u < distinct; u += 256) {
    const unsigned long long key = head(u), previous = u > 0 ? head(u - 1) : before;
    const int64_t at = base + u;
    if (out.csr_offsets) out.csr_offsets[at] = A.head_at[B.start + u];
    if (out.to_unique) out.to_unique[at] = A.head_row[B.start + u];
    write_row(L, key, columns, at, out);
    if (L.bits[0] <= 6u && ((u == 0 && !known) || key_field(L, key, 0) != key_field(L, previous, 0)))
      atomicMin(&A.h->item_first[key_field(L, key, 0)], (int)at);
  }
  if (out.to_orig)
    for (uint32_t p = t; p < B.size; p += 256) {
      const uint2 r = reinterpret_cast<const uint2*>(A.keys)[B.start + p];
      out.to_orig[r.y] = base + r.x;
    }
}

// ---- the library's sort ---------------------------------------------------------------------------
template <class Src>
__global__ void __launch_bounds__(256) unique_pack(Src src, int64_t n, const UniqueHeader* __restrict__ h,
                                                   void* __restrict__ keys, uint32_t* __restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const KeyLayout L = h->layout;
  int v[4];
  src.load(i, src.hint(i), v);
  const unsigned long long key = pack_key(L, v);
  if (L.total <= 32u)
    reinterpret_cast<uint32_t*>(keys)[i] = (uint32_t)key;
  else
    reinterpret_cast<unsigned long long*>(keys)[i] = key;
  idx[i] = (uint32_t)i;
}

// One pass over the sorted (key, row) pairs.  rank[i] = number of segment heads in [0, i].
template <typename KeyT>
__global__ void __launch_bounds__(256) unique_emit(const KeyT* __restrict__ keys, const uint32_t* __restrict__ idx,
                                                   const uint32_t* __restrict__ rank, int64_t n, int columns,
                                                   UniqueHeader* __restrict__ h, UniqueOut out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const KeyLayout L = h->layout;  // the same for every thread: scalar work
  const KeyT key = keys[i];
  const uint32_t row = idx[i];
  const int64_t u = (int64_t)rank[i] - 1;
  const KeyT previous = i == 0 ? (KeyT)0 : keys[i - 1];
  if (out.csr_indices) out.csr_indices[i] = row;
  if (out.to_orig) out.to_orig[row] = u;
  if (i == 0 || previous != key) {
    if (out.csr_offsets) out.csr_offsets[u] = i;
    // the sort is stable, so the head of a segment is the lowest row of its key
    if (out.to_unique) out.to_unique[u] = row;
    write_row(L, (unsigned long long)key, columns, u, out);
    const int item = key_field(L, (unsigned long long)key, 0);
    if (L.bits[0] <= 6u && (i == 0 || key_field(L, (unsigned long long)previous, 0) != item))
      h->item_first[item] = (int)u;
  }
  if (i == n - 1) {
    if (out.csr_offsets) out.csr_offsets[u + 1] = n;
    h->count = (int32_t)(u + 1);
  }
}

// Sort, rank and emit for one key width.
template <typename KeyT>
int sort_rows(const UniqueView& v, int64_t n, int columns, unsigned key_bits, const UniqueOut& out, hipStream_t s) {
  KeyT* keys_a = reinterpret_cast<KeyT*>(v.keys_a);
  KeyT* keys_b = reinterpret_cast<KeyT*>(v.keys_b);
  size_t temp_bytes = v.temp_bytes;
  if (key_bits > 0) {
    if (rocprim::radix_sort_pairs<SortConfig>(v.temp, temp_bytes, keys_a, keys_b, v.idx_a, v.idx_b, (size_t)n, 0u,
                                  key_bits, s) != hipSuccess)
      return WCN_ERR_LAUNCH;
  }
  const KeyT* keys = key_bits > 0 ? keys_b : keys_a;  // all rows equal: nothing to sort
  const uint32_t* idx = key_bits > 0 ? v.idx_b : v.idx_a;
  HeadIterator<KeyT> heads(rocprim::counting_iterator<uint32_t>(0), HeadFlag<KeyT>{keys});
  temp_bytes = v.temp_bytes;
  if (rocprim::inclusive_scan(v.temp, temp_bytes, heads, v.rank, (size_t)n, rocprim::plus<uint32_t>(), s) !=
      hipSuccess)
    return WCN_ERR_LAUNCH;
  hipLaunchKernelGGL(unique_emit<KeyT>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, keys, idx,
                     (const uint32_t*)v.rank, n, columns, v.hdr, out);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

// The whole pipeline over a row source.  host_item_offsets (batch + 1), when given: the distinct rows
// of every value 0 .. batch - 1 of the first column, whose values are 0 <= v < batch.
template <class Src>
int unique_run(const Src& src, int64_t n, int columns, void* workspace, size_t workspace_bytes,
               const UniqueOut& out, int64_t* num_unique, int64_t* host_item_offsets, int batch, hipStream_t s) {
  if (workspace_bytes < unique_layout(nullptr, n, nullptr)) return WCN_ERR_WORKSPACE;
  UniqueView v;
  unique_layout(workspace, n, &v);
  const int64_t box_parts = (n + 4095) / 4096;
  const int boxes = box_parts < kBoxParts ? (int)box_parts : kBoxParts;
  const bool sampled = n <= kSampleSortRows;
  int64_t wanted = (n + kBucketRows - 1) / kBucketRows;
  wanted = wanted < kMaxBuckets ? wanted : kMaxBuckets;
  const int buckets = !sampled || n <= kBucketCap ? 1 : (int)wanted;
  const int samples = buckets > 1 ? buckets * kSamplesPerBucket : 0;
  int4* sample = reinterpret_cast<int4*>(v.keys_b);
  hipLaunchKernelGGL(unique_box<Src>, dim3((unsigned)boxes), dim3(1024), 0, s, src, n, v.boxes, samples,
                     samples > 0 ? ((uint64_t)n << 32) / (uint64_t)samples : 0ull, sample);
  WCN_LAUNCH_CHECK();
  hipLaunchKernelGGL(unique_split, dim3(1), dim3(1024), 0, s, (const int32_t*)v.boxes, boxes, (const int4*)sample,
                     columns, buckets, v.hdr, v.bounds);
  WCN_LAUNCH_CHECK();
  const BucketArgs<Src> bucket_args{src,      n,      v.bounds, v.starts,   v.large, v.keys_b,        v.idx_b,
                                    v.keys_a, v.rank, v.idx_a,  v.distinct, v.hdr,   out.csr_indices, out.to_orig != nullptr};
  if (sampled && buckets == 1) {
    hipLaunchKernelGGL((unique_bucket_large<Src, true>), dim3(1), dim3(1024), 0, s, bucket_args);
    WCN_LAUNCH_CHECK();
  } else if (sampled) {
    const int parts = (int)((n + kPartRows - 1) / kPartRows);
    hipLaunchKernelGGL(unique_assign<Src>, dim3((unsigned)parts), dim3(512), 0, s, src, n,
                       (const UniqueHeader*)v.hdr, buckets, (const uint64_t*)v.bounds, (void*)v.keys_a, v.idx_a,
                       v.rank);
    WCN_LAUNCH_CHECK();
    hipLaunchKernelGGL(unique_columns, dim3((unsigned)((buckets + 31) / 32)), dim3(1024), 0, s,
                       (const UniqueHeader*)v.hdr, parts, buckets, v.rank, v.sizes);
    WCN_LAUNCH_CHECK();
    hipLaunchKernelGGL(unique_place, dim3((unsigned)parts), dim3(1024), 0, s, n, v.hdr, buckets,
                       (const uint64_t*)v.bounds, v.large, (const uint32_t*)v.sizes, (const uint32_t*)v.rank, (const void*)v.keys_a,
                       (const uint32_t*)v.idx_a, v.starts, (void*)v.keys_b, v.idx_b);
    WCN_LAUNCH_CHECK();
    hipLaunchKernelGGL(unique_bucket<Src>, dim3((unsigned)buckets), dim3(kSmallThreads), 0, s, bucket_args);
    WCN_LAUNCH_CHECK();
    hipLaunchKernelGGL((unique_bucket_large<Src, false>), dim3((unsigned)(buckets < 256 ? buckets : 256)), dim3(1024), 0, s, bucket_args);
    WCN_LAUNCH_CHECK();
  }
  if (sampled) {
    hipLaunchKernelGGL(unique_finish<Src>, dim3((unsigned)buckets), dim3(256), 0, s, bucket_args, columns, out);
    WCN_LAUNCH_CHECK();
  }
  UniqueHeader h;
  constexpr size_t kRead = offsetof(UniqueHeader, pad);
  if (wcn_read_small(&h, v.hdr, kRead, s) != WCN_OK) return WCN_ERR_LAUNCH;
  if (h.layout.total > 64u) return WCN_ERR_COORD_RANGE;
  if (!sampled || h.overflow) {
    hipLaunchKernelGGL(unique_pack<Src>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, n,
                       (const UniqueHeader*)v.hdr, (void*)v.keys_a, v.idx_a);
    WCN_LAUNCH_CHECK();
    const int rc = h.layout.total <= 32u ? sort_rows<uint32_t>(v, n, columns, h.layout.total, out, s)
                                         : sort_rows<unsigned long long>(v, n, columns, h.layout.total, out, s);
    if (rc != WCN_OK) return rc;
    if (wcn_read_small(&h, v.hdr, kRead, s) != WCN_OK) return WCN_ERR_LAUNCH;
  }
  *num_unique = h.count;
  if (host_item_offsets) {
    int64_t at = h.count;
    host_item_offsets[batch] = at;
    for (int b = batch - 1; b >= 0; --b) {
      const int64_t f = (int64_t)b - (int32_t)h.layout.mn[0];
      if (f >= 0 && f < WCN_VOXEL_MAX_BATCH && h.item_first[f] != INT32_MAX) at = h.item_first[f];
      host_item_offsets[b] = at;
    }
  }
  return WCN_OK;
}

// Checks the batch offsets and fills the by-value copy the kernels take.
int make_point_rows(const float* points, int64_t num_points, const int64_t* host_batch_offsets,
                    const int64_t* device_batch_offsets_or_null, int32_t batch_size, double voxel_size,
                    PointRows* src) {
  if (num_points < 0 || num_points >= (1ll << 31) || batch_size < 1 || !host_batch_offsets ||
      !(voxel_size > 0.0))
    return WCN_ERR_INVALID_ARGUMENT;
  if (host_batch_offsets[0] != 0 || host_batch_offsets[batch_size] != num_points)
    return WCN_ERR_INVALID_ARGUMENT;
  for (int b = 0; b < batch_size; ++b)
    if (host_batch_offsets[b + 1] < host_batch_offsets[b]) return WCN_ERR_INVALID_ARGUMENT;
  if (batch_size > WCN_VOXEL_MAX_BATCH && !device_batch_offsets_or_null) return WCN_ERR_INVALID_ARGUMENT;
  if (num_points > 0 && !points) return WCN_ERR_INVALID_ARGUMENT;
  src->points = points;
  src->inv = (float)(1.0 / voxel_size);
  src->batch_size = batch_size;
  src->device_starts = batch_size > WCN_VOXEL_MAX_BATCH ? device_batch_offsets_or_null : nullptr;
  for (int b = 0; b <= WCN_VOXEL_MAX_BATCH; ++b)
    src->starts.start[b] = b <= batch_size && batch_size <= WCN_VOXEL_MAX_BATCH ? host_batch_offsets[b] : 0;
  return WCN_OK;
}

int empty_result(int64_t* csr_offsets, hipStream_t s) {
  if (csr_offsets && hipMemsetAsync(csr_offsets, 0, sizeof(int64_t), s) != hipSuccess) return WCN_ERR_LAUNCH;
  return WCN_OK;
}

}  // namespace

extern "C" {

int wcn_voxel_rows(const float* points, int64_t num_points, const int64_t* host_batch_offsets,
                   const int64_t* device_batch_offsets_or_null, int32_t batch_size, double voxel_size,
                   int32_t* rows, void* stream) {
  PointRows src;
  const int rc = make_point_rows(points, num_points, host_batch_offsets, device_batch_offsets_or_null,
                                 batch_size, voxel_size, &src);
  if (rc != WCN_OK) return rc;
  if (num_points == 0) return WCN_OK;
  if (!rows) return WCN_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(voxel_rows, dim3((unsigned)((num_points + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, src, num_points, (int4*)rows);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_batch_indexed_rows(const int32_t* coords, int64_t num_rows, int32_t dims,
                           const int64_t* host_batch_offsets, int32_t batch_size, int32_t* rows,
                           void* stream) {
  BatchStarts starts;
  if (num_rows < 0 || dims < 1 || !wcn_item_starts(host_batch_offsets, batch_size, num_rows, &starts))
    return WCN_ERR_INVALID_ARGUMENT;
  if (num_rows == 0) return WCN_OK;
  if (!coords || !rows) return WCN_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(batch_indexed_rows, dim3((unsigned)((num_rows + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, coords, num_rows, (int)dims, starts, (int)batch_size, rows);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

size_t wcn_unique_rows_workspace_bytes(int64_t num_rows) {
  if (num_rows < 0 || num_rows >= (1ll << 31)) return 0;
  return unique_layout(nullptr, num_rows, nullptr);
}

int wcn_unique_rows_csr(const int32_t* rows, int64_t num_rows, int32_t columns, void* workspace,
                        size_t workspace_bytes, int32_t* unique_rows, int64_t* to_orig,
                        int64_t* csr_indices, int64_t* csr_offsets, int64_t* to_unique,
                        int64_t* num_unique, void* stream) {
  if (num_rows < 0 || num_rows >= (1ll << 31) || columns < 1 || columns > 4 || !num_unique)
    return WCN_ERR_INVALID_ARGUMENT;
  *num_unique = 0;
  if (num_rows == 0) return empty_result(csr_offsets, (hipStream_t)stream);
  if (!rows || !workspace) return WCN_ERR_INVALID_ARGUMENT;
  const IntRows src{rows, (int)columns};
  const UniqueOut out{unique_rows, nullptr, to_orig, csr_indices, csr_offsets, to_unique};
  return unique_run(src, num_rows, (int)columns, workspace, workspace_bytes, out, num_unique, nullptr, 0,
                    (hipStream_t)stream);
}

int wcn_voxelize_points_csr(const float* points, int64_t num_points, const int64_t* host_batch_offsets,
                            const int64_t* device_batch_offsets_or_null, int32_t batch_size,
                            double voxel_size, void* workspace, size_t workspace_bytes,
                            int32_t* unique_rows, int64_t* to_orig, int64_t* csr_indices,
                            int64_t* csr_offsets, int64_t* to_unique, int64_t* num_unique, void* stream) {
  return wcn_voxelize_points_items(points, num_points, host_batch_offsets, device_batch_offsets_or_null,
                                   batch_size, voxel_size, workspace, workspace_bytes, unique_rows, nullptr,
                                   to_orig, csr_indices, csr_offsets, to_unique, num_unique, nullptr, stream);
}

int wcn_voxelize_points_items(const float* points, int64_t num_points, const int64_t* host_batch_offsets,
                              const int64_t* device_batch_offsets_or_null, int32_t batch_size,
                              double voxel_size, void* workspace, size_t workspace_bytes,
                              int32_t* unique_rows, int32_t* unique_coords, int64_t* to_orig,
                              int64_t* csr_indices, int64_t* csr_offsets, int64_t* to_unique,
                              int64_t* num_unique, int64_t* host_item_offsets, void* stream) {
  if (!num_unique || (host_item_offsets && batch_size > WCN_VOXEL_MAX_BATCH)) return WCN_ERR_INVALID_ARGUMENT;
  *num_unique = 0;
  PointRows src;
  const int rc = make_point_rows(points, num_points, host_batch_offsets, device_batch_offsets_or_null,
                                 batch_size, voxel_size, &src);
  if (rc != WCN_OK) return rc;
  if (num_points == 0) {
    for (int b = 0; host_item_offsets && b <= batch_size; ++b) host_item_offsets[b] = 0;
    return empty_result(csr_offsets, (hipStream_t)stream);
  }
  if (!workspace) return WCN_ERR_INVALID_ARGUMENT;
  const UniqueOut out{unique_rows, unique_coords, to_orig, csr_indices, csr_offsets, to_unique};
  return unique_run(src, num_points, 4, workspace, workspace_bytes, out, num_unique, host_item_offsets,
                    batch_size, (hipStream_t)stream);
}

}  // extern "C"
