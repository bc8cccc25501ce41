// Pooling over a kernel map (gfx950): every output row is the sum / mean / maximum of the input
// rows its pairs name (reference: warpconvnet/nn/functional/sparse_pool.py:25-120, which sorts
// the pairs by output row with torch and reduces the segments with torch_scatter.segment_csr).
//
// The pairs are first put in output-row form (wcn_rows_build, or rows_from_groups below for a builder's map: row_ptr /
// row_in), then one thread per (output row, 16 bytes of channels)
// walks the row's input rows with fp32 accumulators and writes its piece once: no atomics, every
// feature row read in whole 16-byte pieces, the output written once.  HBM-bound:
// s * C * (L + M) + 4 (L + M) bytes.
//
// The gradient runs the same walk over the map with in and out exchanged: the gradient of an
// input row is the sum over its pairs of the output row's gradient (divided by the output row's
// pair count for the mean; only where the input row was the maximum for max).
#include <algorithm>

#include "wcn_rows.h"

namespace {

using namespace wcn_rows;

enum { POOL_SUM = 0, POOL_MEAN = 1, POOL_MAX = 2, POOL_MIN = 3 };

template <typename ARG, int N>
struct __attribute__((aligned(sizeof(ARG) * N > 16 ? 16 : sizeof(ARG) * N))) Args {  // of one piece
  ARG v[N];
};

// out[m] = reduce over the entries of row m; rows without pairs become 0 (sparse_pool.py:92-104).
// For the maximum / minimum, arg[m][c] names the pair that supplied it (the first one in the row's
// order among equals): ARG = int32_t its input row, -1 for rows without pairs; ARG = uint8_t /
// uint16_t its kernel offset, all ones for rows without pairs.
//
// HBM-bound (4.3 TB/s; its gradient 4.6).  Four entries in flight per thread instead of one, and the offset in a byte instead of the
// input row in four (more than the output itself): a 2x2x2 maximum over 500 k rows of 64 fp16 channels 61 -> 24 us.
template <typename T, typename ARG, bool VEC>
__global__ void __launch_bounds__(256) pool_fwd(const T* __restrict__ X, int64_t num_in, int channels,
                                                RowTiling tiling, const uint32_t* __restrict__ row_mask, int words,
                                                const int32_t* __restrict__ row_ptr,
                                                const int32_t* __restrict__ row_in, int64_t num_out,
                                                int mode, T* __restrict__ out,
                                                ARG* __restrict__ arg) {
  constexpr int N = Piece<T>::N, U = 4;
  const int sub = (int)threadIdx.x / tiling.width;
  const int64_t m = (int64_t)blockIdx.x * tiling.rows + sub;
  if (sub >= tiling.rows || m >= num_out) return;
  for (int piece = (int)threadIdx.x % tiling.width; piece < tiling.pieces; piece += tiling.width) {
    const int c0 = piece * N;
    float acc[N];
    int32_t who[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      acc[j] = 0.f;
      who[j] = -1;
    }
    walk_row<U>(row_mask, words, row_ptr, row_in, m, num_in, [&](const int* k, const int32_t* r, const bool* live) {
      Piece<T> x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = load_raw<T, VEC>(X, r[u], channels, c0);
      together(x);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (!live[u]) continue;
        if (mode >= POOL_MAX) {
          const float sign = mode == POOL_MAX ? 1.f : -1.f;  // the minimum is the maximum of -x
          const int32_t tag = sizeof(ARG) == 4 ? r[u] : k[u];
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const float v = to_float(x[u].v[j]);
            const bool better = who[j] < 0 || sign * v > sign * acc[j];
            acc[j] = better ? v : acc[j];
            who[j] = better ? tag : who[j];
          }
        } else {
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(x[u].v[j]);
        }
      }
    });
    if (mode == POOL_MEAN) {
      const int count = row_ptr[m + 1] - row_ptr[m];
      const float inv = count > 0 ? 1.f / (float)count : 0.f;
#pragma unroll
      for (int j = 0; j < N; ++j) acc[j] *= inv;
    }
    store_piece<T, VEC>(out, m, channels, c0, acc);
    if (mode >= POOL_MAX && arg) {
      ARG* dst = arg + m * channels + c0;
      Args<ARG, N> a;
#pragma unroll
      for (int j = 0; j < N; ++j) a.v[j] = (ARG)who[j];
      if (VEC) {
        *reinterpret_cast<Args<ARG, N>*>(dst) = a;
      } else {
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (c0 + j < channels) dst[j] = a.v[j];
      }
    }
  }
}

// dX[n] = sum over the pairs (n, m) of input row n of dY[m] (sum), dY[m] / count[m] (mean), or
// dY[m] where arg[m][c] names the pair (max, min).  `row_mask` / `row_ptr` / `row_in` are the rows form of the
// exchanged map (rows = input rows, entries = output rows); out_ptr is the row_ptr of the forward
// rows form (pair count of every output row), used by the mean.
template <typename T, typename ARG, bool VEC>
__global__ void __launch_bounds__(256) pool_bwd(const T* __restrict__ dY, int64_t num_out, int channels,
                                                RowTiling tiling, const uint32_t* __restrict__ row_mask, int words,
                                                const int32_t* __restrict__ row_ptr,
                                                const int32_t* __restrict__ row_in, int64_t num_in,
                                                int mode, const int32_t* __restrict__ out_ptr,
                                                const ARG* __restrict__ arg, T* __restrict__ dX) {
  constexpr int N = Piece<T>::N, U = 4;
  const int sub = (int)threadIdx.x / tiling.width;
  const int64_t n = (int64_t)blockIdx.x * tiling.rows + sub;
  if (sub >= tiling.rows || n >= num_in) return;
  for (int piece = (int)threadIdx.x % tiling.width; piece < tiling.pieces; piece += tiling.width) {
    const int c0 = piece * N;
    float acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = 0.f;
    walk_row<U>(row_mask, words, row_ptr, row_in, n, num_out, [&](const int* k, const int32_t* r, const bool* live) {
      Piece<T> g[U];
#pragma unroll
      for (int u = 0; u < U; ++u) g[u] = load_raw<T, VEC>(dY, r[u], channels, c0);
      together(g);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t m = r[u];
        if (!live[u]) continue;
        if (mode == POOL_MEAN) {
          const int cnt = out_ptr[m + 1] - out_ptr[m];
          const float inv = cnt > 0 ? 1.f / (float)cnt : 0.f;
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(g[u].v[j]) * inv;
        } else if (mode >= POOL_MAX) {
          const ARG tag = (ARG)(sizeof(ARG) == 4 ? (int32_t)n : k[u]);
#pragma unroll
          for (int j = 0; j < N; ++j)
            if (c0 + j < channels && arg[m * channels + c0 + j] == tag) acc[j] += to_float(g[u].v[j]);
        } else {
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(g[u].v[j]);
        }
      }
    });
    store_piece<T, VEC>(dX, n, channels, c0, acc);
  }
}

// The gradient of a map whose input rows are each in exactly one pair (kernel as large as the stride,
// no voxel twice): every output row hands its gradient to the input rows it was made of.  Nothing is
// added up, so the forward rows form serves and dY and arg are read once and in order: 500 k rows 27 us, where the
// exchanged form took a second build (90 us) and its gathers (82 us).
template <typename T, typename ARG, bool VEC>
__global__ void __launch_bounds__(256) pool_bwd_spread(const T* __restrict__ dY, int64_t num_out, int channels,
                                                       RowTiling tiling, const uint32_t* __restrict__ row_mask,
                                                       int words, const int32_t* __restrict__ row_ptr,
                                                       const int32_t* __restrict__ row_in, int64_t num_in,
                                                       int mode, const ARG* __restrict__ arg,
                                                       T* __restrict__ dX) {
  constexpr int N = Piece<T>::N, U = 4;
  const int sub = (int)threadIdx.x / tiling.width;
  const int64_t m = (int64_t)blockIdx.x * tiling.rows + sub;
  if (sub >= tiling.rows || m >= num_out) return;
  const int count = row_ptr[m + 1] - row_ptr[m];
  const float scale = mode == POOL_MEAN && count > 0 ? 1.f / (float)count : 1.f;
  for (int piece = (int)threadIdx.x % tiling.width; piece < tiling.pieces; piece += tiling.width) {
    const int c0 = piece * N;
    float g[N];
    load_piece<T, VEC>(dY, m, channels, c0, g);
    Args<ARG, N> a{};
    if (mode >= POOL_MAX) {
      const ARG* src = arg + m * channels + c0;
      if (VEC) {
        a = *reinterpret_cast<const Args<ARG, N>*>(src);
      } else {
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (c0 + j < channels) a.v[j] = src[j];
      }
    }
    walk_row<U>(row_mask, words, row_ptr, row_in, m, num_in, [&](const int* k, const int32_t* r, const bool* live) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (!live[u]) continue;
        float v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = mode >= POOL_MAX ? (a.v[j] == (ARG)k[u] ? g[j] : 0.f) : g[j] * scale;
        store_piece<T, VEC>(dX, r[u], channels, c0, v);
      }
    });
  }
}

// ---- rows form of a builder's map ---------------------------------------------------------------
//
// Pairs that ascend in output row inside every offset, once per (offset, row), with their 64-row
// group starts: a wave makes the rows of a group by itself.  The group's first entry is the sum of
// its starts over the offsets (lane = offset).  The runs of its offsets are laid end to end and dealt to the lanes without gaps: every
// offset marks where its run begins, and the running maximum of the marks is a pair's offset.  A row's bits are set in LDS, a
// pair's place follows from the bits below its own.  The numbers of a chunk of pairs stay in registers between the two, and where that is
// all of the group's they go through LDS to their places, in runs.  A group with more asks for everything twice, a chunk after the other, so
// maps of more than five pairs a row are dealt with 1,024 at a time; others with 384 (some 270 on surfaces), in half the registers.  Groups
// that follow one another go to one XCD: their runs follow one another in the lists.  Bound by its chain of two reads and, of full
// groups, by what one wave has to go through.  us, 384 and entries stored one by one / as it is: 3x3x3 over 157,000 rows of 12 pairs 19.7 / 13.8,
// 37,000 of 13 17.7 / 13.2, 163,000 of 9 16.2 / 12.3; of 5 and fewer pairs: 300,000 9.2 / 8.1, 500,000 11.4 / 10.7, 2x2x2 163,000 6.0 / 5.7
// (1,024 at a time, 84 registers: 11.4 and 15.3 over 300,000 and 500,000).
constexpr int GROUPED_WORDS = 4;  // up to 128 offsets

template <bool ONE, int CHUNK>  // ONE: at most 32 offsets; CHUNK: pairs of a group that are held at a time
__global__ void __launch_bounds__(256) rows_from_groups(const int32_t* __restrict__ gathered,
                                                        const int32_t* __restrict__ grouping,
                                                        const int64_t* __restrict__ offsets,
                                                        const int32_t* __restrict__ gs, int K, int words,
                                                        int64_t num_rows, int64_t G, int64_t pairs,
                                                        uint32_t* __restrict__ row_mask,
                                                        int32_t* __restrict__ row_ptr,
                                                        int32_t* __restrict__ row_in,
                                                        int32_t* __restrict__ clear, int clear_words) {
  constexpr int WORDS = ONE ? 1 : GROUPED_WORDS, OFFSETS = 32 * WORDS, ROUNDS = CHUNK / 64;
  __shared__ uint32_t s_mask[4][64][WORDS + (ONE ? 0 : 1)];
  __shared__ int32_t s_first[4][64];
  __shared__ int32_t s_shift[4][OFFSETS];  // the place of an offset's first pair in the lists, less its place among the group's
  __shared__ int32_t s_begin[4][OFFSETS];  // the latter
  __shared__ int32_t s_in[4][CHUNK];         // the group's entries in their places
  __shared__ uint32_t s_mark[4][CHUNK / 4];  // a byte for each of CHUNK of the group's pairs: offset + 1 where a run begins
  const int tid = threadIdx.x, lane = wcn_lane(), wave = tid >> 6;
  if (blockIdx.x == 0)  // counters of whatever follows on the stream
    for (int i = tid; i < clear_words; i += 256) clear[i] = 0;
  const int64_t group = (int64_t)wcn_xcd_tile((int)blockIdx.x, (int)gridDim.x) * 4 + wave, row0 = group * 64;
  if (group >= G) return;
  auto written = [] {  // what this wave has put into LDS is there for all its lanes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
#pragma unroll
  for (int w = 0; w < WORDS; ++w) s_mask[wave][lane][w] = 0u;
  int before = 0, total = 0;
#pragma unroll
  for (int h = 0; h < (ONE ? 1 : 2); ++h) {  // lane k looks after offset k (and 64 + k)
    const int k = lane + 64 * h;
    int n = 0, first = 0;
    if (k < K) {
      const int32_t* g = gs + (int64_t)k * (G + 1) + group;
      const int b = g[0], cnt = g[1] - b;
      const int64_t start = offsets[k] + b;
      before += b;
      n = cnt < 0 || cnt > 64 || start < 0 || start + cnt > pairs ? 0 : cnt;  // inconsistent table: contribute nothing
      first = (int)start;
    }
    const int incl = wcn_wave_inclusive_sum(n);
    if (k < OFFSETS) {
      s_begin[wave][k] = n > 0 ? total + incl - n : -1;
      s_shift[wave][k] = first - (total + incl - n);
    }
    total += __shfl(incl, 63, 64);
  }
  const int base = __shfl(wcn_wave_inclusive_sum(before), 63, 64);
  int carry = 0;  // the offset (+ 1) of the last pair before the chunk
  uint32_t tag[ROUNDS];  // a pair's row in the group and, from bit 8 on, its offset; ~0: none
  int in[ROUNDS];
  auto request = [&](int p0) {  // pairs p0 .. p0 + CHUNK - 1 of the group
    uint8_t* const mark = reinterpret_cast<uint8_t*>(s_mark[wave]);
#pragma unroll
    for (int i = 0; i < CHUNK / 4; i += 64)
      if (p0 + 4 * i < total && i + lane < CHUNK / 4) s_mark[wave][i + lane] = 0u;
    written();
#pragma unroll
    for (int h = 0; h < (ONE ? 1 : 2); ++h) {
      const int o = lane + 64 * h;
      const int at = o < K ? s_begin[wave][o] - p0 : -1;
      if (at >= 0 && at < CHUNK && s_begin[wave][o] >= 0) mark[at] = (uint8_t)(o + 1);
    }
    written();
    int row[ROUNDS];
#pragma unroll
    for (int u = 0; u < ROUNDS; ++u) {
      tag[u] = ~0u;
      if (p0 + u * 64 >= total) continue;
      int v = max((int)mark[u * 64 + lane], lane == 0 ? carry : 0);
      // running maximum over the lanes, as wcn_wave_inclusive_sum
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));
      v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
      carry = __builtin_amdgcn_readlane(v, 63);
      const int p = p0 + u * 64 + lane;
      if (p < total) tag[u] = (uint32_t)(v - 1);
      const int at = p < total ? p + s_shift[wave][v - 1] : 0;
      row[u] = pairs > 0 ? grouping[at] : 0;
      in[u] = pairs > 0 ? gathered[at] : 0;
    }
#pragma unroll
    for (int u = 0; u < ROUNDS; ++u) {
      if (p0 + u * 64 >= total) continue;
      const int64_t r = row[u] - row0;
      tag[u] = tag[u] != ~0u && (uint64_t)r < 64u ? tag[u] << 8 | (uint32_t)r : ~0u;
    }
  };
  for (int p0 = 0; p0 < total; p0 += CHUNK) {
    request(p0);
#pragma unroll
    for (int u = 0; u < ROUNDS; ++u)
      if (tag[u] != ~0u) atomicOr(&s_mask[wave][tag[u] & 63u][ONE ? 0 : tag[u] >> 13], 1u << (tag[u] >> 8 & 31u));
  }
  written();
  int mine = 0;
#pragma unroll
  for (int w = 0; w < WORDS; ++w) mine += __popc(s_mask[wave][lane][w]);
  const int incl = wcn_wave_inclusive_sum(mine);
  s_first[wave][lane] = base + incl - mine;
  if (row0 + lane < num_rows) {
    row_ptr[row0 + lane] = base + incl - mine;
#pragma unroll
    for (int w = 0; w < WORDS; ++w)
      if (w < words) row_mask[(row0 + lane) * words + w] = s_mask[wave][lane][w];
    if (row0 + lane == num_rows - 1) row_ptr[num_rows] = base + incl;
  }
  written();
  const bool again = total > CHUNK;
  carry = 0;
  for (int p0 = 0; p0 < total; p0 += CHUNK) {
    if (again) request(p0);
#pragma unroll
    for (int u = 0; u < ROUNDS; ++u) {
      if (tag[u] == ~0u) continue;
      const int row = (int)(tag[u] & 63u), k = (int)(tag[u] >> 8);
      const uint32_t* const mask = s_mask[wave][row];
      int rank = __popc(mask[ONE ? 0 : k >> 5] & ((1u << (k & 31)) - 1u));
      if (!ONE)
        for (int w = 0; w < (k >> 5); ++w) rank += __popc(mask[w]);
      const int at = s_first[wave][row] - base + rank;
      if (!again) s_in[wave][at] = in[u];
      else if ((int64_t)base + at < pairs) row_in[(int64_t)base + at] = in[u];
    }
  }
  if (again) return;
  written();
  const int held = __shfl(incl, 63, 64);  // of at most CHUNK pairs
  for (int i = lane; i < held; i += 64)
    if ((int64_t)base + i < pairs) row_in[(int64_t)base + i] = s_in[wave][i];
}

// ---- reduction over CSR segments (the point -> voxel pooling) -----------------------------------
//
//   out[u] = reduce over e in [offsets[u], offsets[u+1]) of X[indices ? indices[e] : e]
//
// (reference: warpconvnet/ops/reductions.py:36-72, torch_scatter.segment_csr over features that
// were gathered with features[to_csr_indices] first; here the gather is part of the walk, so the
// gathered copy is never written).  Offsets and indices are 64-bit, as torch.unique and argsort
// return them.  arg[u][c] = the input row that supplied the extremum.
//
// Bound by the gathered rows, and by how many of them are in flight.  A thread walks two segments, four entries
// of each at a time: one after the other, every entry was two memory round trips (its index, its row);
// eight entries of one segment (an average voxel has three) asked for many rows in vain.  4 M rows of 64 bytes
// into 1.3 M segments: 109 us (270 MB read in pieces of 64 bytes, 108 MB written), 115 with four entries of one
// segment, 131 with eight.
template <typename T, bool VEC, bool EXTREME>
__global__ void __launch_bounds__(256) segment_reduce(const T* __restrict__ X, int64_t num_in, int channels,
                                                      RowTiling tiling, const int64_t* __restrict__ offsets,
                                                      const int64_t* __restrict__ indices,
                                                      int64_t num_entries, int64_t num_out, int mode,
                                                      T* __restrict__ out,
                                                      int64_t* __restrict__ arg) {
  constexpr int N = Piece<T>::N, U = 4, S = 2;
  const int sub = (int)threadIdx.x / tiling.width;
  if (sub >= tiling.rows) return;
  int64_t segment[S], begin[S], end[S], longest = 0;
#pragma unroll
  for (int k = 0; k < S; ++k) {
    segment[k] = (int64_t)blockIdx.x * (S * tiling.rows) + k * tiling.rows + sub;
    const int64_t at = segment[k] < num_out ? segment[k] : num_out - 1;
    begin[k] = offsets[at];
    end[k] = offsets[at + 1];
  }
#pragma unroll
  for (int k = 0; k < S; ++k) {
    // offsets that do not fit the entry list are cut to it: nothing is read past its end
    begin[k] = begin[k] < 0 ? 0 : begin[k];
    end[k] = end[k] > num_entries ? num_entries : end[k];
    if (num_in == 0 || segment[k] >= num_out) end[k] = begin[k];
    longest = end[k] - begin[k] > longest ? end[k] - begin[k] : longest;
  }
  const float sign = mode == POOL_MIN ? -1.f : 1.f;  // the minimum is the maximum of -x
  for (int piece = (int)threadIdx.x % tiling.width; piece < tiling.pieces; piece += tiling.width) {
    const int c0 = piece * N;
    float acc[S][N];
    int64_t who[EXTREME ? S : 1][N];
#pragma unroll
    for (int k = 0; k < S; ++k)
#pragma unroll
      for (int j = 0; j < N; ++j) {
        acc[k][j] = 0.f;
        who[EXTREME ? k : 0][j] = -1;
      }
    for (int64_t e = 0; e < longest; e += U) {
      int64_t r[S * U];
      bool live[S * U];
#pragma unroll
      for (int u = 0; u < S * U; ++u) {
        const int k = u / U;
        const int64_t want = begin[k] + e + u % U;
        live[u] = want < end[k];
        // an entry that is there whatever the segment: its own last one, or the list's first
        const int64_t at = live[u] ? want : end[k] > begin[k] ? end[k] - 1 : 0;
        r[u] = at;
      }
      if (indices) {
#pragma unroll
        for (int u = 0; u < S * U; ++u) r[u] = indices[r[u]];
      }
      Piece<T> x[S * U];
#pragma unroll
      for (int u = 0; u < S * U; ++u) {
        live[u] = live[u] && (uint64_t)r[u] < (uint64_t)num_in;
        r[u] = (uint64_t)r[u] < (uint64_t)num_in ? r[u] : 0;
        x[u] = load_raw<T, VEC>(X, r[u], channels, c0);
      }
      together(x);
#pragma unroll
      for (int u = 0; u < S * U; ++u) {
        const int k = u / U;
        if (!live[u]) continue;
        if (EXTREME) {
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const float v = to_float(x[u].v[j]);
            const bool better = who[EXTREME ? k : 0][j] < 0 || sign * v > sign * acc[k][j];
            acc[k][j] = better ? v : acc[k][j];
            who[EXTREME ? k : 0][j] = better ? r[u] : who[EXTREME ? k : 0][j];
          }
        } else {
#pragma unroll
          for (int j = 0; j < N; ++j) acc[k][j] += to_float(x[u].v[j]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < S; ++k) {
      if (segment[k] >= num_out) continue;
      if (mode == POOL_MEAN) {
        const float inv = end[k] > begin[k] ? 1.f / (float)(end[k] - begin[k]) : 1.f;
#pragma unroll
        for (int j = 0; j < N; ++j) acc[k][j] *= inv;
      }
      store_piece<T, VEC>(out, segment[k], channels, c0, acc[k]);
      if (EXTREME && arg) {
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (c0 + j < channels) arg[segment[k] * channels + c0 + j] = who[EXTREME ? k : 0][j];
      }
    }
  }
}

// Every input row lies in at most one segment: dX[n] = dY[u] (sum), dY[u] / count[u] (mean),
// dY[u] where arg[u][c] == n (max, min), with u = segment_of[n]; 0 for rows outside every segment.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256) segment_reduce_bwd(const T* __restrict__ dY, int64_t num_out,
                                                          int channels, const int64_t* __restrict__ offsets,
                                                          const int64_t* __restrict__ segment_of,
                                                          int64_t num_in, int mode,
                                                          const int64_t* __restrict__ arg,
                                                          T* __restrict__ dX) {
  constexpr int N = Piece<T>::N;
  const int pieces = (channels + N - 1) / N;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= num_in * pieces) return;
  const int64_t n = i / pieces;
  const int c0 = (int)(i % pieces) * N;
  float acc[N];
#pragma unroll
  for (int j = 0; j < N; ++j) acc[j] = 0.f;
  const int64_t u = segment_of[n];
  if ((uint64_t)u < (uint64_t)num_out) {
    float g[N];
    load_piece<T, VEC>(dY, u, channels, c0, g);
    if (mode == POOL_MEAN) {
      const int64_t cnt = offsets[u + 1] - offsets[u];
      const float inv = cnt > 0 ? 1.f / (float)cnt : 0.f;
#pragma unroll
      for (int j = 0; j < N; ++j) acc[j] = g[j] * inv;
    } else if (mode >= POOL_MAX) {
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (c0 + j < channels && arg[u * channels + c0 + j] == n) acc[j] = g[j];
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) acc[j] = g[j];
    }
  }
  store_piece<T, VEC>(dX, n, channels, c0, acc);
}

template <typename T, typename ARG>
void launch_pool_fwd(const void* X, int64_t num_in, int channels, int dtype, const WcnRowsView& v, int64_t num_out,
                     int mode, bool vec, void* out, void* arg, hipStream_t s) {
  const RowTiling t = row_tiling(channels, dtype);
  hipLaunchKernelGGL((vec ? pool_fwd<T, ARG, true> : pool_fwd<T, ARG, false>), dim3((unsigned)((num_out + t.rows - 1) / t.rows)), dim3(256), 0, s, (const T*)X,
                     num_in, channels, t, (const uint32_t*)v.row_mask, v.words, (const int32_t*)v.row_ptr,
                     (const int32_t*)v.row_in, num_out, mode, (T*)out, (ARG*)arg);
}

template <typename T, typename ARG>
void launch_pool_bwd(const void* dY, int64_t num_out, int channels, int dtype, const WcnRowsView& v, int64_t num_in,
                     int mode, bool vec, const int32_t* out_ptr, const void* arg, void* dX, hipStream_t s) {
  const RowTiling t = row_tiling(channels, dtype);
  hipLaunchKernelGGL((vec ? pool_bwd<T, ARG, true> : pool_bwd<T, ARG, false>), dim3((unsigned)((num_in + t.rows - 1) / t.rows)), dim3(256), 0, s, (const T*)dY,
                     num_out, channels, t, (const uint32_t*)v.row_mask, v.words, (const int32_t*)v.row_ptr,
                     (const int32_t*)v.row_in, num_in, mode, out_ptr, (const ARG*)arg, (T*)dX);
}

template <typename T, typename ARG>
void launch_pool_spread(const void* dY, int64_t num_out, int channels, int dtype, const WcnRowsView& v, int64_t num_in,
                        int mode, bool vec, const void* arg, void* dX, hipStream_t s) {
  const RowTiling t = row_tiling(channels, dtype);
  hipLaunchKernelGGL((vec ? pool_bwd_spread<T, ARG, true> : pool_bwd_spread<T, ARG, false>), dim3((unsigned)((num_out + t.rows - 1) / t.rows)), dim3(256), 0, s,
                     (const T*)dY, num_out, channels, t, (const uint32_t*)v.row_mask, v.words, (const int32_t*)v.row_ptr,
                     (const int32_t*)v.row_in, num_in, mode, (const ARG*)arg, (T*)dX);
}

// f(T{}, ARG{}) for a feature dtype and an argument width (4: the input row, 1 / 2: the offset)
template <typename F>
void with_types(int dtype, int arg_bytes, const F& f) {
  auto with_arg = [&](auto t) {
    if (arg_bytes == 1) f(t, uint8_t{}); else if (arg_bytes == 2) f(t, uint16_t{}); else f(t, int32_t{});
  };
  if (dtype == WCN_DTYPE_F32) with_arg(float{}); else if (dtype == WCN_DTYPE_F16) with_arg(_Float16{}); else with_arg(__bf16{});
}

int pool_fwd_any(const void* features, int64_t num_in, int32_t channels, int32_t dtype, const void* rows_by_out,
                 int64_t num_out, int32_t num_offsets, int64_t num_pairs, int32_t mode, void* out, void* arg,
                 int arg_bytes, void* stream) {
  if (dtype < 0 || dtype > 2 || mode < POOL_SUM || mode > POOL_MIN || channels < 1 || num_in < 0 ||
      num_out < 0 || num_pairs < 0 || !rows_by_out || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS)
    return WCN_ERR_INVALID_ARGUMENT;
  if (num_out == 0) return WCN_OK;
  if (!out || (num_in > 0 && !features)) return WCN_ERR_INVALID_ARGUMENT;
  WcnRowsView v;
  wcn_rows_layout(const_cast<void*>(rows_by_out), num_out, num_offsets, num_pairs, &v);
  const bool vec = rows_are_vectors(features, channels, dtype) && rows_are_vectors(out, channels, dtype) &&
                   (uintptr_t)arg % 16 == 0;
  if (num_in == 0 && num_pairs > 0) return WCN_ERR_INVALID_ARGUMENT;
  with_types(dtype, arg_bytes, [&](auto t, auto a) {
    launch_pool_fwd<decltype(t), decltype(a)>(features, num_in, channels, dtype, v, num_out, mode, vec, out, arg,
                                              (hipStream_t)stream);
  });
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

// rows_by_in NULL: every input row is in exactly one pair of rows_by_out
int pool_bwd_any(const void* grad_out, int64_t num_out, int32_t channels, int32_t dtype, const void* rows_by_in,
                 const void* rows_by_out, int64_t num_in, int32_t num_offsets, int64_t num_pairs, int32_t mode,
                 const void* arg, int arg_bytes, void* grad_in, void* stream) {
  if (dtype < 0 || dtype > 2 || mode < POOL_SUM || mode > POOL_MIN || channels < 1 || num_in < 0 ||
      num_out < 0 || num_pairs < 0 || (!rows_by_in && !rows_by_out) || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS)
    return WCN_ERR_INVALID_ARGUMENT;
  if ((mode >= POOL_MAX && !arg) || (mode == POOL_MEAN && !rows_by_out)) return WCN_ERR_INVALID_ARGUMENT;
  if (num_in == 0) return WCN_OK;
  if (!grad_in || (num_out > 0 && !grad_out)) return WCN_ERR_INVALID_ARGUMENT;
  WcnRowsView v, vo;
  if (rows_by_in) wcn_rows_layout(const_cast<void*>(rows_by_in), num_in, num_offsets, num_pairs, &v);
  if (rows_by_out) wcn_rows_layout(const_cast<void*>(rows_by_out), num_out, num_offsets, num_pairs, &vo);
  const bool vec = rows_are_vectors(grad_out, channels, dtype) && rows_are_vectors(grad_in, channels, dtype) &&
                   (uintptr_t)arg % 16 == 0;
  if ((!rows_by_in && num_pairs != num_in) || (num_out == 0 && num_pairs > 0)) return WCN_ERR_INVALID_ARGUMENT;
  with_types(dtype, arg_bytes, [&](auto t, auto a) {
    if (rows_by_in)
      launch_pool_bwd<decltype(t), decltype(a)>(grad_out, num_out, channels, dtype, v, num_in, mode, vec,
                                                rows_by_out ? vo.row_ptr : nullptr, arg, grad_in, (hipStream_t)stream);
    else
      launch_pool_spread<decltype(t), decltype(a)>(grad_out, num_out, channels, dtype, vo, num_in, mode, vec, arg, grad_in,
                                                   (hipStream_t)stream);
  });
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

template <typename T>
void launch_segment_reduce(const void* X, int64_t num_in, int channels, int dtype, const int64_t* offsets,
                           const int64_t* indices, int64_t num_entries, int64_t num_out, int mode,
                           bool vec, void* out, int64_t* arg, hipStream_t s) {
  const RowTiling t = row_tiling(channels, dtype);
  hipLaunchKernelGGL((mode >= POOL_MAX ? (vec ? segment_reduce<T, true, true> : segment_reduce<T, false, true>)
                                       : (vec ? segment_reduce<T, true, false> : segment_reduce<T, false, false>)),
                     dim3((unsigned)((num_out + 2 * t.rows - 1) / (2 * t.rows))), dim3(256), 0, s, (const T*)X, num_in, channels, t,
                     offsets, indices, num_entries, num_out, mode, (T*)out, arg);
}

template <typename T>
void launch_segment_reduce_bwd(const void* dY, int64_t num_out, int channels, const int64_t* offsets,
                               const int64_t* segment_of, int64_t num_in, int mode, bool vec,
                               const int64_t* arg, void* dX, hipStream_t s) {
  const int pieces = (channels + Piece<T>::N - 1) / Piece<T>::N;
  const int64_t items = num_in * pieces;
  hipLaunchKernelGGL((vec ? segment_reduce_bwd<T, true> : segment_reduce_bwd<T, false>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s,
                     (const T*)dY, num_out, channels, offsets, segment_of, num_in, mode, arg, (T*)dX);
}

bool map_args_ok(const int64_t* host_offsets, int K, const int32_t* in_maps, const int32_t* out_maps,
                 int64_t* pairs) {
  if (!host_offsets || K < 1 || K > WCN_MAX_OFFSETS || host_offsets[0] != 0) return false;
  for (int k = 0; k < K; ++k)
    if (host_offsets[k + 1] < host_offsets[k]) return false;
  *pairs = host_offsets[K];
  if (*pairs > INT32_MAX) return false;
  return *pairs == 0 || (in_maps && out_maps);
}

}  // namespace

extern "C" {

size_t wcn_map_rows_workspace_bytes(int64_t num_rows, int32_t num_offsets, int64_t num_pairs) {
  if (num_rows < 0 || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || num_pairs < 0) return 0;
  return wcn_rows_layout(nullptr, num_rows, num_offsets, num_pairs, nullptr);
}

int wcn_map_rows_build(const int32_t* gathered_rows, const int32_t* grouping_rows,
                       const int64_t* host_offsets, int32_t num_offsets, int64_t num_rows,
                       void* workspace, size_t workspace_bytes, void* stream) {
  int64_t pairs = 0;
  if (!map_args_ok(host_offsets, num_offsets, gathered_rows, grouping_rows, &pairs) || num_rows < 0 ||
      num_rows >= (1ll << 31) || !workspace)
    return WCN_ERR_INVALID_ARGUMENT;
  if (workspace_bytes < wcn_map_rows_workspace_bytes(num_rows, num_offsets, pairs))
    return WCN_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  WcnRowsView v;
  wcn_rows_layout(workspace, num_rows, num_offsets, pairs, &v);
  if (hipMemcpyAsync(v.offsets, host_offsets, sizeof(int64_t) * (size_t)(num_offsets + 1),
                     hipMemcpyHostToDevice, s) != hipSuccess)
    return WCN_ERR_LAUNCH;
  if (num_rows == 0) return WCN_OK;
  return wcn_rows_build(gathered_rows, grouping_rows, num_offsets, num_rows, pairs, v, s);
}

}  // extern "C"

int wcn_rows_from_groups(const int32_t* gathered_rows, const int32_t* grouping_rows, const int64_t* device_offsets,
                         const int32_t* group_start, int num_offsets, int64_t num_rows, int64_t num_pairs,
                         void* workspace, size_t workspace_bytes, int32_t* clear, int clear_words, hipStream_t s) {
  if (num_offsets < 1 || num_offsets > 32 * GROUPED_WORDS || num_rows < 0 || num_rows >= (1ll << 31) || num_pairs < 0 ||
      num_pairs > INT32_MAX || !workspace || !device_offsets || !group_start ||
      (num_pairs > 0 && (!gathered_rows || !grouping_rows)))
    return WCN_ERR_INVALID_ARGUMENT;
  if (workspace_bytes < wcn_map_rows_workspace_bytes(num_rows, num_offsets, num_pairs)) return WCN_ERR_WORKSPACE;
  if (num_rows == 0) return WCN_OK;
  WcnRowsView v;
  wcn_rows_layout(workspace, num_rows, num_offsets, num_pairs, &v);
  const bool many = num_pairs > 5 * num_rows;
  hipLaunchKernelGGL((num_offsets <= 32 ? (many ? rows_from_groups<true, 1024> : rows_from_groups<true, 384>)
                                       : many ? rows_from_groups<false, 1024> : rows_from_groups<false, 384>), dim3((unsigned)((v.G + 3) / 4)), dim3(256), 0, s, gathered_rows,
                     grouping_rows, device_offsets, group_start, num_offsets, v.words, num_rows, v.G, num_pairs, v.row_mask,
                     v.row_ptr, v.row_in, clear, clear_words);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

extern "C" {

int wcn_map_rows_build_grouped(const int32_t* gathered_rows, const int32_t* grouping_rows,
                               const int64_t* device_offsets, const int32_t* group_start, int32_t num_offsets,
                               int64_t num_rows, int64_t num_pairs, void* workspace, size_t workspace_bytes,
                               void* stream) {
  return wcn_rows_from_groups(gathered_rows, grouping_rows, device_offsets, group_start, num_offsets, num_rows, num_pairs,
                              workspace, workspace_bytes, nullptr, 0, (hipStream_t)stream);
}

int wcn_sparse_pool_fwd(const void* features, int64_t num_in, int32_t channels, int32_t dtype,
                        const void* rows_by_out, int64_t num_out, int32_t num_offsets,
                        int64_t num_pairs, int32_t mode, void* out, int32_t* argmax_or_null,
                        void* stream) {
  return pool_fwd_any(features, num_in, channels, dtype, rows_by_out, num_out, num_offsets, num_pairs, mode, out,
                      argmax_or_null, 4, stream);
}

int wcn_sparse_pool_bwd(const void* grad_out, int64_t num_out, int32_t channels, int32_t dtype,
                        const void* rows_by_in, const void* rows_by_out, int64_t num_in,
                        int32_t num_offsets, int64_t num_pairs, int32_t mode,
                        const int32_t* argmax_or_null, void* grad_in, void* stream) {
  if (!rows_by_in) return WCN_ERR_INVALID_ARGUMENT;
  return pool_bwd_any(grad_out, num_out, channels, dtype, rows_by_in, rows_by_out, num_in, num_offsets, num_pairs, mode,
                      argmax_or_null, 4, grad_in, stream);
}

/* The offset of an extremum is kept in one byte where every offset fits (255 marks rows without pairs). */
int32_t wcn_pool_offset_bytes(int32_t num_offsets) { return num_offsets <= 255 ? 1 : 2; }

int wcn_sparse_pool_fwd_offsets(const void* features, int64_t num_in, int32_t channels, int32_t dtype,
                                const void* rows_by_out, int64_t num_out, int32_t num_offsets, int64_t num_pairs,
                                int32_t mode, void* out, void* arg_offsets_or_null, void* stream) {
  return pool_fwd_any(features, num_in, channels, dtype, rows_by_out, num_out, num_offsets, num_pairs, mode, out,
                      arg_offsets_or_null, wcn_pool_offset_bytes(num_offsets), stream);
}

int wcn_sparse_pool_bwd_offsets(const void* grad_out, int64_t num_out, int32_t channels, int32_t dtype,
                                const void* rows_by_in_or_null, const void* rows_by_out, int64_t num_in,
                                int32_t num_offsets, int64_t num_pairs, int32_t mode, const void* arg_offsets_or_null,
                                void* grad_in, void* stream) {
  return pool_bwd_any(grad_out, num_out, channels, dtype, rows_by_in_or_null, rows_by_out, num_in, num_offsets, num_pairs,
                      mode, arg_offsets_or_null, wcn_pool_offset_bytes(num_offsets), grad_in, stream);
}

int wcn_segment_reduce(const void* features, int64_t num_in, int32_t channels, int32_t dtype,
                       const int64_t* segment_offsets, const int64_t* indices_or_null,
                       int64_t num_entries, int64_t num_segments, int32_t mode, void* out,
                       int64_t* argmax_or_null, void* stream) {
  if (dtype < 0 || dtype > 2 || mode < POOL_SUM || mode > POOL_MIN || channels < 1 || num_in < 0 ||
      num_segments < 0 || channels > (1 << 20) || num_entries < 0)
    return WCN_ERR_INVALID_ARGUMENT;
  if (num_segments == 0) return WCN_OK;
  if (!out || !segment_offsets || (num_in > 0 && !features)) return WCN_ERR_INVALID_ARGUMENT;
  const bool vec = rows_are_vectors(features, channels, dtype) && rows_are_vectors(out, channels, dtype);
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case WCN_DTYPE_F32:
      launch_segment_reduce<float>(features, num_in, channels, dtype, segment_offsets, indices_or_null,
                                   num_entries, num_segments, mode, vec, out, argmax_or_null, s);
      break;
    case WCN_DTYPE_F16:
      launch_segment_reduce<_Float16>(features, num_in, channels, dtype, segment_offsets, indices_or_null,
                                      num_entries, num_segments, mode, vec, out, argmax_or_null, s);
      break;
    default:
      launch_segment_reduce<__bf16>(features, num_in, channels, dtype, segment_offsets, indices_or_null,
                                    num_entries, num_segments, mode, vec, out, argmax_or_null, s);
      break;
  }
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_segment_reduce_bwd(const void* grad_out, int64_t num_segments, int32_t channels, int32_t dtype,
                           const int64_t* segment_offsets, const int64_t* segment_of_row, int64_t num_in,
                           int32_t mode, const int64_t* argmax_or_null, void* grad_in, void* stream) {
  if (dtype < 0 || dtype > 2 || mode < POOL_SUM || mode > POOL_MIN || channels < 1 || num_in < 0 ||
      num_segments < 0 || channels > (1 << 20))
    return WCN_ERR_INVALID_ARGUMENT;
  if (mode >= POOL_MAX && !argmax_or_null) return WCN_ERR_INVALID_ARGUMENT;
  if (num_in == 0) return WCN_OK;
  if (!grad_in || !segment_of_row || !segment_offsets || (num_segments > 0 && !grad_out))
    return WCN_ERR_INVALID_ARGUMENT;
  const bool vec = rows_are_vectors(grad_out, channels, dtype) && rows_are_vectors(grad_in, channels, dtype);
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case WCN_DTYPE_F32:
      launch_segment_reduce_bwd<float>(grad_out, num_segments, channels, segment_offsets, segment_of_row,
                                       num_in, mode, vec, argmax_or_null, grad_in, s);
      break;
    case WCN_DTYPE_F16:
      launch_segment_reduce_bwd<_Float16>(grad_out, num_segments, channels, segment_offsets,
                                          segment_of_row, num_in, mode, vec, argmax_or_null, grad_in, s);
      break;
    default:
      launch_segment_reduce_bwd<__bf16>(grad_out, num_segments, channels, segment_offsets, segment_of_row,
                                        num_in, mode, vec, argmax_or_null, grad_in, s);
      break;
  }
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

}  // extern "C"
