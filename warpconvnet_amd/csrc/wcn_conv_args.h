// Arguments shared by the contraction kernels of wcn_conv.hip and wcn_conv_pack.hip.
#ifndef WCN_CONV_ARGS_H_
#define WCN_CONV_ARGS_H_
#include "wcn_common.h"

#include <type_traits>

struct ConvArgs {
  const void* X;
  const void* Wt;              // weight tiles Wt[k][n][c], see conv_prep_weight
  const void* Wf;              // the same values in the order of the kernel for small maps, or null
  const void* zeros;           // 1 KiB of zeros (source of loads that have nothing to fetch)
  const void* bias;            // same dtype as X, or null
  const int32_t* in_maps;      // pair lists; inside every offset out_maps ascends
  const int32_t* out_maps;
  const int64_t* offsets;      // (K + 1), device
  const int32_t* group_start;  // (K, G + 1): pairs of offset k below output row 64 * g
  void* out;
  int64_t num_in, num_out, G;
  int64_t num_pairs;           // all offsets together (known on the host)
  int64_t list_capacity;       // > 0: the lists of a builder that the host has not waited for (num_pairs: its guess), see lists_absent
  int32_t K, c_in, c_out, c_in_pad, c_out_pad, identity;
  int32_t vec_in;   // feature rows are 16-byte aligned and a whole number of 16-byte vectors
  int32_t vec_out;  // same for output rows
  int32_t flat_in;  // c_in is a multiple of the staged row and the feature matrix is below 4 GiB
  // Few output tiles and several slices of input channels (small maps with wide features): the
  // slices go to different workgroups (blockIdx.z), each writes its fp32 sums to
  // partial[slice][row][c_out_pad] and conv_split_reduce adds them in slice order.
  int32_t split;
  float* partial;
  // What the epilogue does besides bias and rounding (wcn_sparse_conv_fwd_fused): add a row of
  // `residual` (num_out x c_out, the element type of the features) and / or clamp at zero, both
  // on the fp32 sums before the one rounding.
  const void* residual;
  int32_t relu;
  int32_t bias_rounded;  // the bias is added to the rounded sums (not in the kernels for small maps and wide rows and the ring)
  int32_t vec_res;  // rows of `residual` are 16-byte aligned and a whole number of 16-byte vectors

  // Lists that the host has not waited for hold what they should if offsets[K], the pairs, is at most their capacity and
  // offsets[K + 1], the builder's status, 0.  Otherwise the kernel returns at once and the host launches again.
  __device__ __forceinline__ bool lists_absent() const {
    return list_capacity > 0 && (offsets[K] > list_capacity || offsets[K + 1] != 0);
  }
};


// The pair-packed contraction (wcn_conv_pack*.hip): whether it takes a problem, and its launch.
constexpr int WCN_PACK_MAX_BIAS = 1024;  // output channels (padded) whose bias fits the kernel's LDS copy
bool wcn_conv_pack_takes(const ConvArgs& a, int dtype);
int wcn_conv_pack_launch(const ConvArgs& a, int dtype, hipStream_t stream);

// The output-stationary contraction for wide rows (wcn_conv_dense.hip): whether it takes a problem,
// and its launch.
bool wcn_conv_dense_takes(const ConvArgs& a, int dtype);
int wcn_conv_dense_launch(const ConvArgs& a, int dtype, hipStream_t stream);

// The contraction for small maps (wcn_conv_split.hip): whether it takes a problem, and its launch.
bool wcn_conv_split_takes(const ConvArgs& a, int dtype);
int wcn_conv_split_launch(const ConvArgs& a, int dtype, hipStream_t stream);

// The contraction over a tile plan (wcn_conv_tiles.hip): whether it takes a problem's shape, and its launch
// (X, Wt, bias, residual, relu, out and the sizes are read from `a`).
bool wcn_conv_tiles_takes(int dtype, int num_offsets, int c_in, int c_out);
bool wcn_conv_tiles_rows(int num_offsets, int c_in, int c_out, int64_t num_out);  // enough rows for a plan, whatever the pairs
int wcn_conv_tiles_worth(int num_offsets, int c_in, int c_out, int64_t num_out, const int64_t* host_offsets, int identity,
                         int calls);
int wcn_conv_tiles_launch(const ConvArgs& a, int dtype, const WcnTilePlan& plan, hipStream_t stream);

// The contraction for maps with exactly one pair per output row (wcn_conv_single.hip): whether it
// takes a problem's shape, and its launch over pair lists in any order (`host_offsets`: the K + 1
// offsets; X, Wt, bias, residual, relu, out, the lists and the sizes are read from `a`).
constexpr int WCN_SINGLE_MAX_OFFSETS = 64;
struct WcnSingleTiles {  // tiles of 64 to 256 pairs of one offset, in offset order
  int32_t first_tile[WCN_SINGLE_MAX_OFFSETS + 1];
  int32_t first_pair[WCN_SINGLE_MAX_OFFSETS + 1];
  int32_t total;
};
bool wcn_conv_single_takes(int dtype, int c_in, int c_out, int num_offsets);
int wcn_conv_single_launch(const ConvArgs& a, int dtype, const int64_t* host_offsets, hipStream_t stream);

// Column sums of a (rows, channels) array: the first pass, `parts` fp32 partial sums per channel, and what the second is to do
// with them (wcn_colsum.hip; the gradient of a bias).
struct WcnColumnSums {
  float* partial;  // (parts, channels)
  int32_t parts, channels;
  void* out;
  int32_t out_dtype;
};
void wcn_column_sums_parts(int64_t num_rows, int dtype, WcnColumnSums* c);  // sets parts
int wcn_column_sums_first(const void* rows, int64_t num_rows, int dtype, const WcnColumnSums& c, hipStream_t stream);
int wcn_column_sums_second(const WcnColumnSums& c, hipStream_t stream);

#ifdef __HIPCC__
// The second pass by a workgroup's first 256 threads for 16 channels from c0 on: parts p, p + 16, ... to thread p / 16, eight in flight, their
// sixteen sums added in order.
template <typename OT>
__device__ __forceinline__ void wcn_column_sums_finish(const WcnColumnSums& s, int c0, OT* out) {
  __shared__ float s_sum[16][16];
  constexpr int AHEAD = 8;
  const bool there = threadIdx.x < 256;
  const int at = threadIdx.x & 15, stretch = threadIdx.x >> 4, c = c0 + at;
  float sum = 0.f;
  if (there && c < s.channels) {
    for (int p = stretch; p < s.parts; p += 16 * AHEAD) {
      float v[AHEAD];
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) v[i] = p + 16 * i < s.parts ? s.partial[(int64_t)(p + 16 * i) * s.channels + c] : 0.f;
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) sum += v[i];
    }
  }
  if (there) s_sum[stretch][at] = sum;
  __syncthreads();
  if (stretch != 0 || c >= s.channels) return;
  for (int p = 1; p < 16; ++p) sum += s_sum[p][at];
  out[c] = (OT)sum;
}
#endif

// The weight gradient of 16-bit rows of whole vectors (wcn_conv_wgrad.hip): whether it takes a problem, the bytes of its
// partial sums (pairs with the identity's rows), and its launch (with the column sums of grad_out, both passes).
bool wcn_wgrad_tiles_takes(int dtype, int c_in, int c_out, const void* features, const void* grad_out);
size_t wcn_wgrad_tiles_partial_bytes(int num_offsets, int c_in, int c_out, int64_t pairs);
int wcn_wgrad_tiles_launch(const void* features, int64_t num_in, int c_in, const void* grad_out, int64_t num_out, int c_out,
                           int dtype, const int32_t* in_maps, const int32_t* out_maps, const int64_t* host_offsets,
                           const int64_t* device_offsets, int num_offsets, int identity, void* grad_weight,
                           int weight_dtype, float* partial, const WcnColumnSums* columns_or_null, hipStream_t stream);

#endif  // WCN_CONV_ARGS_H_

// The contraction for narrow layers (wcn_conv_group.hip): a wave per group of 64 output rows.
bool wcn_conv_group_shape(int dtype, int num_offsets, int c_in, int c_out);  // what it asks of the layer alone
bool wcn_conv_group_takes(const ConvArgs& a, int dtype);
int wcn_conv_group_launch(const ConvArgs& a, int dtype, hipStream_t stream);

// The contraction kernel a launcher has just enqueued, as the profiler would print its name
// ("conv_fwd_pack<f16, 512, 11, 4, 2, true, false, false>"): kept per host thread for
// wcn_conv_last_kernel (a measurement aid: reports name what ran, not what was expected to run).
void wcn_conv_note_kernel(const char* format, ...);
template <typename T>
inline const char* wcn_type_text() {
  return sizeof(T) == 4 ? "float" : (std::is_same<T, _Float16>::value ? "f16" : "bf16");
}
