// Depthwise convolution over a kernel map (gfx950):
//
//   out[m][c] = sum over the pairs (n, m) of offset k of X[n][c] * W[k][c]
//
// (reference: warpconvnet/nn/functional/sparse_conv_depth.py:151-231).  A multiplication per gathered
// value: memory traffic is all there is, and the forward pass and the input gradient are one walk
// over a rows form of the map, a thread per (row, 16 bytes of channels), fp32 sums, one store.
#include <algorithm>

#include "wcn_conv_args.h"
#include "wcn_rows.h"

namespace {

using namespace wcn_rows;

// The set bits of row_mask[m] name the offsets of the row's entries in order, which selects the weight
// row; `reverse`: the rows form is that of the forward map and offset k stands for K - 1 - k (the input
// gradient over a map that is its own exchange: no second rows form).  With an identity offset that offset
// is X[m] * W[identity] for every m < num_in and its pairs are ignored (sparse_conv_depth.py:163-165).
// The bias is added to the rounded sum, as a separate addition behind the call would.
//
// Bound by the rate of the gathered rows (a gather alone of these rows: 40 us) and by the LDS that
// the weights come from.  (A piece's eight weights side by side, its two 16-byte reads 32 bytes from its neighbour's: two thirds of
// the LDS's cycles, most of them bank conflicts, and 71.6 us below; the halves apart: 64.2.  Rows padded by 16, 32, 64
// bytes on top: the same.)  LDS_W: the
// weight, as fp32, in LDS for the life of the workgroup, which takes many rows; read from memory instead, the
// rows of a wave asked for eight different weight rows per entry, two 16-byte loads each beside the one of the
// feature row.  Eight entries in flight and the next row's mask on its way: 500 k rows of 64 fp16
// channels, 4.2 entries a row, 258 -> 75 us at the time (four entries: 77; with a branch around each load: 107).
template <typename T, typename WT, bool LDS_W, bool VEC>
__global__ void __launch_bounds__(256) depthwise_rows(const T* __restrict__ X, int64_t num_in, int channels,
                                                      RowTiling tiling, const WT* __restrict__ W, int K, int identity,
                                                      bool reverse, const uint32_t* __restrict__ row_mask, int words,
                                                      const int32_t* __restrict__ row_ptr,
                                                      const int32_t* __restrict__ row_in, int64_t num_out,
                                                      const T* __restrict__ bias, T* __restrict__ out) {
  constexpr int N = Piece<T>::N, U = 8;
  // The first four channels of every piece, then the last four: in either, K rows of 16 bytes per piece, so that the
  // pieces of a row lie side by side.
  extern __shared__ __attribute__((aligned(16))) float s_w[];
  const int pitch = tiling.pieces * 4;
  if (LDS_W) {
    const int padded = tiling.pieces * N;
    for (int i = threadIdx.x; i < K * padded; i += 256) {
      const int k = i / padded, c = i % padded;
      s_w[(c % N / 4 * K + k) * pitch + c / N * 4 + c % 4] = c < channels ? to_float(W[(int64_t)k * channels + c]) : 0.f;
    }
    __syncthreads();
  }
  const int sub = (int)threadIdx.x / tiling.width;
  if (sub >= tiling.rows) return;
  for (int piece = (int)threadIdx.x % tiling.width; piece < tiling.pieces; piece += tiling.width) {
    const int c0 = piece * N;
    float b[N];
#pragma unroll
    for (int j = 0; j < N; ++j) b[j] = bias && c0 + j < channels ? to_float(bias[c0 + j]) : 0.f;
    int next_first = 0;  // the next row's first entry and mask word are on their way while a row is worked on
    uint32_t next_word = 0;
    if ((int64_t)blockIdx.x * tiling.rows + sub < num_out) {
      next_first = row_ptr[(int64_t)blockIdx.x * tiling.rows + sub];
      next_word = row_mask[((int64_t)blockIdx.x * tiling.rows + sub) * words];
    }
    for (int64_t m = (int64_t)blockIdx.x * tiling.rows + sub; m < num_out; m += (int64_t)gridDim.x * tiling.rows) {
      float acc[N];
#pragma unroll
      for (int j = 0; j < N; ++j) acc[j] = 0.f;
      auto add = [&](const Piece<T>& x, int k) {
        if (LDS_W) {
          float w[N];
#pragma unroll
          for (int h = 0; h < N / 4; ++h)
            *reinterpret_cast<f32x4*>(w + 4 * h) = *reinterpret_cast<const f32x4*>(s_w + (h * K + k) * pitch + piece * 4);
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(x.v[j]) * w[j];
        } else {
          const WT* w = W + (int64_t)k * channels + c0;
#pragma unroll
          for (int j = 0; j < N; ++j)
            if (c0 + j < channels) acc[j] += to_float(x.v[j]) * to_float(w[j]);
        }
      };
      // the identity's own row is requested with the first entries and added before them
      bool own = identity >= 0 && m < num_in;
      const Piece<T> x_own = load_raw<T, VEC>(X, own ? m : 0, channels, c0);
      int first = next_first;
      uint32_t word = next_word;
      const int64_t m_next = m + (int64_t)gridDim.x * tiling.rows;
      if (m_next < num_out) {
        next_first = row_ptr[m_next];
        next_word = row_mask[m_next * words];
      }
      for (int v = 0; v < words; ++v) {
        if (v > 0) word = row_mask[m * words + v];
        walk_word<U>(word, v * 32, first, row_in, num_in, [&](const int* k, const int32_t* r, const bool* live) {
          Piece<T> x[U];
#pragma unroll
          for (int u = 0; u < U; ++u) x[u] = load_raw<T, VEC>(X, r[u], channels, c0);
          together(x);
          if (own) add(x_own, identity);
          own = false;
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (live[u] && k[u] != identity) add(x[u], reverse ? K - 1 - k[u] : k[u]);
        });
        first += __popc(word);
      }
      if (own) add(x_own, identity);
      if (bias) {
#pragma unroll
        for (int j = 0; j < N; ++j) acc[j] = to_float(from_float<T>(acc[j])) + b[j];
      }
      store_piece<T, VEC>(out, m, channels, c0, acc);
    }
  }
}

// dW[k][c] = sum over the pairs of offset k of X[in][c] * dY[out][c].  A workgroup owns the pairs of one
// offset in one range and writes one partial row; the ranges of an offset are added in order.  With the
// map's group starts a range is one of output rows, the same for all offsets, and the workgroups of
// a range follow one another on one XCD: its dY rows (at most 8192, 1 MB of 64 fp16 channels) then come
// out of that XCD's L2 for all offsets but the first.  Without them a range is a share of the offset's pairs.
// Four pairs in flight per thread: 2.1 M pairs of 64 fp16 channels 117 + 57 (reduction) -> 88 + 10 us.
// The column sums of dY (a bias's gradient) ride on this launch and the reduction's: over 500 k rows of 64 fp16 channels 85.0 + 12.7 and
// 10.4 + 4.1 us one after the other, 90.7 and 10.7 together; a layer and a pooling forward and backward 531 -> 505 to 514 us.
struct WgradRanges {
  const int32_t* gs;  // (K, G + 1) or null
  int64_t G;
  int32_t ranges;
  int64_t groups_per_range;
};
// The identity offset has a pair for every row, several times as many as another: its part of a range is
// cut into this many, each a place of its own among the range's partial rows.
constexpr int OWN_PARTS = 8;
__host__ __device__ inline int wgrad_places(int K, int identity) { return K + (identity >= 0 ? OWN_PARTS - 1 : 0); }

template <typename T, bool VEC>
__global__ void __launch_bounds__(256) depthwise_wgrad(const T* __restrict__ X, int64_t num_in,
                                                       const T* __restrict__ dY, int64_t num_out,
                                                       int channels, const int32_t* __restrict__ in_maps,
                                                       const int32_t* __restrict__ out_maps,
                                                       const int64_t* __restrict__ offsets, WgradRanges q, int K,
                                                       int identity, int64_t identity_rows,
                                                       float* __restrict__ partial, int grid, ColumnPart columns) {
  constexpr int N = Piece<T>::N, U = 4;
  __shared__ float s_sum[256][N + 1];
  if ((int)blockIdx.x >= grid) {  // the column sums of dY: workgroups of their own behind the others
    column_part<T, VEC>(columns, (int)blockIdx.x - grid, &s_sum[0][0]);
    return;
  }
  // blockIdx % 8 is the XCD: range = 8 * (b / 8 / K) + b % 8
  const int places = wgrad_places(K, identity);
  const int t = blockIdx.x >> 3, place = t % places, range = (t / places) * 8 + (blockIdx.x & 7);
  if (range >= q.ranges) return;
  const bool ident = identity >= 0 && place >= identity && place < identity + OWN_PARTS;
  const int k = ident ? identity : identity >= 0 && place >= identity ? place - (OWN_PARTS - 1) : place;
  int64_t first, last;  // pairs of the offset, or rows of the identity
  const int64_t n_k = ident ? identity_rows : offsets[k + 1] - offsets[k];
  if (q.gs) {
    const int64_t g0 = range * q.groups_per_range, g1 = g0 + q.groups_per_range < q.G ? g0 + q.groups_per_range : q.G;
    const int32_t* row = q.gs + (int64_t)k * (q.G + 1);
    first = ident ? g0 * 64 : row[g0];
    last = ident ? g1 * 64 : row[g1];
  } else {
    const int64_t share = (n_k + q.ranges - 1) / q.ranges;
    first = range * share;
    last = first + share;
  }
  if (last > n_k) last = n_k;
  if (ident && last > first) {
    const int64_t share = (last - first + OWN_PARTS - 1) / OWN_PARTS;
    first += (place - identity) * share;
    last = first + share < last ? first + share : last;
  }
  const int count = last > first ? (int)(last - first) : 0;
  const int64_t pbase = offsets[k] + first;
  const int pieces = (channels + N - 1) / N;
  float* sums = partial + ((int64_t)range * places + place) * channels;
  // the 256 threads are `lanes` pairs wide and `width` channel pieces deep
  for (int p0 = 0; p0 < pieces; p0 += 256) {
    const int width = pieces - p0 < 256 ? pieces - p0 : 256;  // pieces handled in this pass
    const int lanes = 256 / width;
    const int piece = p0 + (int)threadIdx.x % width, lane = (int)threadIdx.x / width;
    const int c0 = piece * N;
    float acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = 0.f;
    if (lane < lanes) {
      // the next pairs' rows are known before this one's data are waited for; past the end the last pair is read again
      int64_t rin[U], rout[U];
      auto request = [&](int p) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int pu = p + u * lanes < count ? p + u * lanes : count - 1;
          rin[u] = ident ? first + pu : (int64_t)in_maps[pbase + pu];
          rout[u] = ident ? first + pu : (int64_t)out_maps[pbase + pu];
        }
      };
      if (count > 0) request(lane);
      for (int p = lane; p < count; p += U * lanes) {
        Piece<T> x[U], g[U];
        bool live[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool there = (uint64_t)rin[u] < (uint64_t)num_in && (uint64_t)rout[u] < (uint64_t)num_out;
          live[u] = there && p + u * lanes < count;
          x[u] = load_raw<T, VEC>(X, there ? rin[u] : 0, channels, c0);
          g[u] = load_raw<T, VEC>(dY, there ? rout[u] : 0, channels, c0);
        }
        request(p + U * lanes);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (!live[u]) x[u] = g[u] = Piece<T>{};
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(x[u].v[j]) * to_float(g[u].v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) s_sum[threadIdx.x][j] = acc[j];
    __syncthreads();
    if (lane == 0) {  // one thread per piece adds the lanes in order
      for (int l = 1; l < lanes; ++l)
#pragma unroll
        for (int j = 0; j < N; ++j) acc[j] += s_sum[l * width + (int)threadIdx.x % width][j];
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (c0 + j < channels) sums[c0 + j] = acc[j];
    }
    __syncthreads();
  }
}

// dW[k][c] = the ranges' partial rows added up: 16 stretches side by side, then those in order.  From blockIdx.x = K on: the
// second pass of the column sums, 16 channels each.
template <typename WT>
__global__ void __launch_bounds__(1024) depthwise_wgrad_reduce(const float* __restrict__ partial, int ranges,
                                                               int K, int identity, int channels, WT* __restrict__ dW,
                                                               WcnColumnSums columns) {
  __shared__ float s_sum[16][64];
  if ((int)blockIdx.x >= K) {
    const int c0 = (int)blockIdx.y * 64 + ((int)blockIdx.x - K) * 16;
    if (columns.out_dtype == WCN_DTYPE_F32) wcn_column_sums_finish<float>(columns, c0, (float*)columns.out);
    else if (columns.out_dtype == WCN_DTYPE_F16) wcn_column_sums_finish<_Float16>(columns, c0, (_Float16*)columns.out);
    else wcn_column_sums_finish<__bf16>(columns, c0, (__bf16*)columns.out);
    return;
  }
  const int k = blockIdx.x, lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int c = blockIdx.y * 64 + lane;
  float sum = 0.f;
  if (c < channels) {
    const int places = wgrad_places(K, identity), own = k == identity ? OWN_PARTS : 1;
    const float* src = partial + (int64_t)(identity >= 0 && k > identity ? k + OWN_PARTS - 1 : k) * channels + c;
    const int rows = ranges * own;
    for (int i = part; i < rows; i += 16 * 8) {  // eight loads in flight per thread
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int at = i + 16 * u < rows ? i + 16 * u : i;
        v[u] = src[((int64_t)(at / own) * places + at % own) * channels];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += i + 16 * u < rows ? v[u] : 0.f;
    }
  }
  s_sum[part][lane] = sum;
  __syncthreads();
  if (part != 0 || c >= channels) return;
  for (int p = 1; p < 16; ++p) sum += s_sum[p][lane];
  dW[(int64_t)k * channels + c] = from_float<WT>(sum);
}

// Ranges of the weight gradient: about 4096 workgroups over all offsets (16 per CU), not less than
// 512 rows each (a partial row and its reduction per range) nor more than 8192 (dY rows that an L2 keeps).
inline int64_t wgrad_rows_per_range(int64_t rows, int K) {
  const int64_t want = (rows * K / 4096 + 63) / 64 * 64;
  return want < 512 ? 512 : want > 8192 ? 8192 : want;
}
inline int64_t wgrad_ranges(int64_t rows, int K) {
  const int64_t per = wgrad_rows_per_range(rows, K);
  return rows < 1 ? 1 : (rows + per - 1) / per;
}

// f(T{}, WT{})
template <typename F>
void with_types(int dtype, int weight_dtype, const F& f) {
  if (dtype == WCN_DTYPE_F32) f(float{}, float{});
  else if (dtype == WCN_DTYPE_F16) { if (weight_dtype == WCN_DTYPE_F32) f(_Float16{}, float{}); else f(_Float16{}, _Float16{}); }
  else { if (weight_dtype == WCN_DTYPE_F32) f(__bf16{}, float{}); else f(__bf16{}, __bf16{}); }
}

bool types_ok(int dtype, int weight_dtype) {
  return dtype >= 0 && dtype <= 2 && (weight_dtype == dtype || weight_dtype == WCN_DTYPE_F32);
}

}  // namespace

extern "C" {

int wcn_sparse_depthwise_fwd_fused(const void* features, int64_t num_in, int32_t channels, int32_t dtype,
                                   const void* weight, int32_t weight_dtype, const void* rows_by_out,
                                   int64_t num_out, int32_t num_offsets, int64_t num_pairs,
                                   int32_t identity_offset, int32_t reverse_offsets, const void* bias_or_null,
                                   void* out, void* stream) {
  if (!types_ok(dtype, weight_dtype) || channels < 1 || num_in < 0 || num_out < 0 || num_pairs < 0 || !rows_by_out ||
      !weight || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || identity_offset >= num_offsets)
    return WCN_ERR_INVALID_ARGUMENT;
  if (num_out == 0) return WCN_OK;
  if (!out || num_in == 0 || !features) return WCN_ERR_INVALID_ARGUMENT;
  WcnRowsView v;
  wcn_rows_layout(const_cast<void*>(rows_by_out), num_out, num_offsets, num_pairs, &v);
  const bool vec = rows_are_vectors(features, channels, dtype) && rows_are_vectors(out, channels, dtype);
  const RowTiling t = row_tiling(channels, dtype);
  const size_t lds = sizeof(float) * (size_t)num_offsets * (t.pieces * 4) * (dtype == WCN_DTYPE_F32 ? 1 : 2);
  // up to 32 KB a CU still holds five workgroups; more of them than one pass over the chip only make more copies
  const bool lds_w = lds <= 32768;
  const int64_t need = (num_out + t.rows - 1) / t.rows;
  const unsigned grid = (unsigned)(lds_w ? std::min<int64_t>(need, 2048) : need);
  with_types(dtype, weight_dtype, [&](auto a, auto b) {
    using T = decltype(a);
    using WT = decltype(b);
    auto kernel = lds_w ? (vec ? depthwise_rows<T, WT, true, true> : depthwise_rows<T, WT, true, false>)
                        : (vec ? depthwise_rows<T, WT, false, true> : depthwise_rows<T, WT, false, false>);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds_w ? lds : 0, (hipStream_t)stream, (const T*)features, num_in,
                       channels, t, (const WT*)weight, num_offsets, identity_offset, reverse_offsets != 0,
                       (const uint32_t*)v.row_mask, v.words, (const int32_t*)v.row_ptr, (const int32_t*)v.row_in, num_out,
                       (const T*)bias_or_null, (T*)out);
  });
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_sparse_depthwise_fwd(const void* features, int64_t num_in, int32_t channels, int32_t dtype,
                             const void* weight, int32_t weight_dtype, const void* rows_by_out,
                             int64_t num_out, int32_t num_offsets, int64_t num_pairs,
                             int32_t identity_offset, void* out, void* stream) {
  return wcn_sparse_depthwise_fwd_fused(features, num_in, channels, dtype, weight, weight_dtype, rows_by_out, num_out,
                                        num_offsets, num_pairs, identity_offset, 0, nullptr, out, stream);
}

size_t wcn_depthwise_wgrad_workspace_bytes(int32_t num_offsets, int32_t channels, int64_t num_pairs,
                                           int64_t identity_rows) {
  if (num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || channels < 1 || num_pairs < 0 || identity_rows < 0) return 0;
  return wcn_align256(sizeof(int64_t) * (size_t)(num_offsets + 1)) +
         wcn_align256(sizeof(float) * (size_t)wgrad_ranges(num_pairs + identity_rows, num_offsets) *
                      (size_t)wgrad_places(num_offsets, 0) * (size_t)channels);
}

size_t wcn_depthwise_wgrad_grouped_workspace_bytes(int32_t num_offsets, int32_t channels, int64_t num_out) {
  if (num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || channels < 1 || num_out < 0) return 0;
  return wcn_align256(sizeof(float) * (size_t)wgrad_ranges(num_out, num_offsets) * (size_t)wgrad_places(num_offsets, 0) *
                      (size_t)channels);
}

static int depthwise_wgrad_launch(const void* features, int64_t num_in, const void* grad_out, int64_t num_out,
                                  int32_t channels, int32_t dtype, const int32_t* in_maps, const int32_t* out_maps,
                                  const int64_t* offsets, const WgradRanges& q, int32_t K, int32_t identity,
                                  void* grad_weight, int32_t weight_dtype, float* partial, hipStream_t s,
                                  const WcnColumnSums& columns = WcnColumnSums{}) {
  const int64_t identity_rows = identity >= 0 ? std::min(num_in, num_out) : 0;
  const bool vec = rows_are_vectors(features, channels, dtype) && rows_are_vectors(grad_out, channels, dtype);
  const int ranges = num_in == 0 || num_out == 0 ? 0 : q.ranges;  // 0: the sums are zeros
  const unsigned grid = (unsigned)((ranges + 7) / 8 * 8) * (unsigned)wgrad_places(K, identity);
  const unsigned parts = (unsigned)columns.parts;
  const ColumnPart part = column_part_of(grad_out, num_out, dtype, columns);
  with_types(dtype, weight_dtype, [&](auto a, auto b) {
    using T = decltype(a);
    using WT = decltype(b);
    if (grid + parts > 0)
      hipLaunchKernelGGL((vec ? depthwise_wgrad<T, true> : depthwise_wgrad<T, false>), dim3(grid + parts), dim3(256), 0, s, (const T*)features, num_in, (const T*)grad_out,
                       num_out, channels, in_maps, out_maps, offsets, q, K, identity, identity_rows, partial, (int)grid, part);
    hipLaunchKernelGGL(depthwise_wgrad_reduce<WT>, dim3((unsigned)K + (columns.channels > 0 ? 4u : 0u), (unsigned)((channels + 63) / 64)), dim3(1024), 0, s,
                       (const float*)partial, ranges, K, identity, channels, (WT*)grad_weight, columns);
  });
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_sparse_depthwise_wgrad(const void* features, int64_t num_in, const void* grad_out,
                               int64_t num_out, int32_t channels, int32_t dtype,
                               const int32_t* in_maps, const int32_t* out_maps,
                               const int64_t* host_offsets, int32_t num_offsets,
                               int32_t identity_offset, void* grad_weight, int32_t weight_dtype,
                               void* workspace, size_t workspace_bytes, void* stream) {
  if (!types_ok(dtype, weight_dtype) || channels < 1 || num_in < 0 || num_out < 0 || !grad_weight || !workspace ||
      !host_offsets || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || host_offsets[0] != 0 ||
      identity_offset >= num_offsets)
    return WCN_ERR_INVALID_ARGUMENT;
  for (int k = 0; k < num_offsets; ++k)
    if (host_offsets[k + 1] < host_offsets[k]) return WCN_ERR_INVALID_ARGUMENT;
  const int64_t pairs = host_offsets[num_offsets];
  if (pairs > INT32_MAX || (pairs > 0 && (!in_maps || !out_maps))) return WCN_ERR_INVALID_ARGUMENT;
  if ((num_in > 0 && !features) || (num_out > 0 && !grad_out)) return WCN_ERR_INVALID_ARGUMENT;
  const int64_t identity_rows = identity_offset >= 0 ? std::min(num_in, num_out) : 0;
  if (workspace_bytes < wcn_depthwise_wgrad_workspace_bytes(num_offsets, channels, pairs, identity_rows))
    return WCN_ERR_WORKSPACE;
  int64_t* offsets = (int64_t*)workspace;
  float* partial = (float*)((char*)workspace + wcn_align256(sizeof(int64_t) * (size_t)(num_offsets + 1)));
  hipStream_t s = (hipStream_t)stream;
  if (hipMemcpyAsync(offsets, host_offsets, sizeof(int64_t) * (size_t)(num_offsets + 1),
                     hipMemcpyHostToDevice, s) != hipSuccess)
    return WCN_ERR_LAUNCH;
  const WgradRanges q{nullptr, 0, (int32_t)wgrad_ranges(pairs + identity_rows, num_offsets), 0};
  return depthwise_wgrad_launch(features, num_in, grad_out, num_out, channels, dtype, in_maps, out_maps, offsets, q,
                                num_offsets, identity_offset, grad_weight, weight_dtype, partial, s);
}

static int wgrad_grouped(const void* features, int64_t num_in, const void* grad_out, int64_t num_out,
                         int32_t channels, int32_t dtype, const int32_t* in_maps, const int32_t* out_maps,
                         const int64_t* device_offsets, const int32_t* group_start, int32_t num_offsets,
                         int32_t identity_offset, void* grad_weight, int32_t weight_dtype,
                         void* workspace, size_t workspace_bytes, const WcnColumnSums& columns, void* stream) {
  if (!types_ok(dtype, weight_dtype) || channels < 1 || num_in < 0 || num_out < 0 || !grad_weight || !workspace ||
      !device_offsets || !group_start || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || identity_offset >= num_offsets ||
      (num_in > 0 && !features) || (num_out > 0 && !grad_out) || num_out > INT32_MAX)
    return WCN_ERR_INVALID_ARGUMENT;
  if (workspace_bytes < wcn_depthwise_wgrad_grouped_workspace_bytes(num_offsets, channels, num_out))
    return WCN_ERR_WORKSPACE;
  const WgradRanges q{group_start, (num_out + 63) / 64, (int32_t)wgrad_ranges(num_out, num_offsets),
                      wgrad_rows_per_range(num_out, num_offsets) / 64};
  return depthwise_wgrad_launch(features, num_in, grad_out, num_out, channels, dtype, in_maps, out_maps, device_offsets, q,
                                num_offsets, identity_offset, grad_weight, weight_dtype, (float*)workspace,
                                (hipStream_t)stream, columns);
}

int wcn_sparse_depthwise_wgrad_grouped(const void* features, int64_t num_in, const void* grad_out, int64_t num_out,
                                       int32_t channels, int32_t dtype, const int32_t* in_maps, const int32_t* out_maps,
                                       const int64_t* device_offsets, const int32_t* group_start, int32_t num_offsets,
                                       int32_t identity_offset, void* grad_weight, int32_t weight_dtype,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  return wgrad_grouped(features, num_in, grad_out, num_out, channels, dtype, in_maps, out_maps, device_offsets, group_start,
                       num_offsets, identity_offset, grad_weight, weight_dtype, workspace, workspace_bytes, WcnColumnSums{}, stream);
}

int wcn_sparse_depthwise_wgrad_grouped_bias(const void* features, int64_t num_in, const void* grad_out, int64_t num_out,
                                            int32_t channels, int32_t dtype, const int32_t* in_maps, const int32_t* out_maps,
                                            const int64_t* device_offsets, const int32_t* group_start, int32_t num_offsets,
                                            int32_t identity_offset, void* grad_weight, int32_t weight_dtype,
                                            void* workspace, size_t workspace_bytes, void* grad_bias, int32_t bias_dtype,
                                            void* bias_workspace, size_t bias_workspace_bytes, void* stream) {
  if (!types_ok(dtype, weight_dtype) || channels < 1 || num_out < 0 || bias_dtype < 0 || bias_dtype > 2 || !grad_bias || !bias_workspace)
    return WCN_ERR_INVALID_ARGUMENT;
  if (bias_workspace_bytes < wcn_column_sums_workspace_bytes(channels)) return WCN_ERR_WORKSPACE;
  WcnColumnSums columns = {(float*)bias_workspace, 0, channels, grad_bias, bias_dtype};
  wcn_column_sums_parts(num_out, dtype, &columns);
  return wgrad_grouped(features, num_in, grad_out, num_out, channels, dtype, in_maps, out_maps, device_offsets, group_start,
                       num_offsets, identity_offset, grad_weight, weight_dtype, workspace, workspace_bytes, columns, stream);
}

}  // extern "C"
