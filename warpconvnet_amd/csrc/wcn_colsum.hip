// Column sums of a (rows, channels) array in fp32 (gfx950): the gradient of a layer's bias.
#include <algorithm>

#include "wcn_conv_args.h"
#include "wcn_rows.h"

namespace {

using namespace wcn_rows;

constexpr int PARTS = 512;  // workgroups of the first pass: two per CU

// A workgroup sums a stretch of rows, a thread per 16 bytes of channels, four rows in flight.  HBM-bound (5 TB/s): 500 k
// rows of 64 fp16 channels (64 MB) in 12 + 4 us, where a generic column reduction took 34.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256) column_sums(const T* __restrict__ X, int64_t n, int channels, RowTiling tiling,
                                                   int64_t per, float* __restrict__ partial) {
  constexpr int N = Piece<T>::N, U = 4;
  __shared__ float s_sum[256][N + 1];
  const int sub = (int)threadIdx.x / tiling.width, at = (int)threadIdx.x % tiling.width;
  const int64_t begin = blockIdx.x * per, end = begin + per < n ? begin + per : n;
  for (int p0 = 0; p0 < tiling.pieces; p0 += tiling.width) {
    const int c0 = (p0 + at) * N;
    float acc[N];
#pragma unroll
    for (int j = 0; j < N; ++j) acc[j] = 0.f;
    if (sub < tiling.rows && p0 + at < tiling.pieces) {
      for (int64_t m = begin + sub; m < end; m += U * tiling.rows) {
        Piece<T> x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int64_t r = m + u * tiling.rows;
          x[u] = load_raw<T, VEC>(X, r < end ? r : end - 1, channels, c0);
          if (r >= end) x[u] = Piece<T>{};
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(x[u].v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) s_sum[threadIdx.x][j] = acc[j];
    __syncthreads();
    if (sub == 0 && p0 + at < tiling.pieces) {
      for (int l = 1; l < tiling.rows; ++l)
#pragma unroll
        for (int j = 0; j < N; ++j) acc[j] += s_sum[l * tiling.width + at][j];
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (c0 + j < channels) partial[(int64_t)blockIdx.x * channels + c0 + j] = acc[j];
    }
    __syncthreads();
  }
}

template <typename OT>
__global__ void __launch_bounds__(256) column_sums_finish(WcnColumnSums s) {
  wcn_column_sums_finish<OT>(s, (int)blockIdx.x * 16, (OT*)s.out);
}

inline int column_parts(int64_t n, int rows) {  // at least four rows per thread in a part
  return (int)std::max<int64_t>(1, std::min<int64_t>(PARTS, n / (4 * rows)));
}

}  // namespace

int wcn_column_sums_first(const void* rows, int64_t num_rows, int dtype, WcnColumnSums* c, hipStream_t s) {
  const RowTiling t = row_tiling(c->channels, dtype);
  const bool vec = rows_are_vectors(rows, c->channels, dtype);
  c->parts = column_parts(num_rows, t.rows);
  const int64_t per = (num_rows + c->parts - 1) / c->parts;
  auto first = [&](auto v) {
    using T = decltype(v);
    hipLaunchKernelGGL((vec ? column_sums<T, true> : column_sums<T, false>), dim3((unsigned)c->parts), dim3(256), 0, s,
                       (const T*)rows, num_rows, c->channels, t, per, c->partial);
  };
  if (dtype == WCN_DTYPE_F32) first(float{}); else if (dtype == WCN_DTYPE_F16) first(_Float16{}); else first(__bf16{});
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

int wcn_column_sums_second(const WcnColumnSums& c, hipStream_t s) {
  const dim3 grid((unsigned)((c.channels + 15) / 16)), block(256);
  if (c.out_dtype == WCN_DTYPE_F32) hipLaunchKernelGGL(column_sums_finish<float>, grid, block, 0, s, c);
  else if (c.out_dtype == WCN_DTYPE_F16) hipLaunchKernelGGL(column_sums_finish<_Float16>, grid, block, 0, s, c);
  else hipLaunchKernelGGL(column_sums_finish<__bf16>, grid, block, 0, s, c);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}

extern "C" {

size_t wcn_column_sums_workspace_bytes(int32_t channels) {
  return channels < 1 ? 0 : wcn_align256(sizeof(float) * (size_t)PARTS * (size_t)channels);
}

int wcn_column_sums(const void* rows, int64_t num_rows, int32_t channels, int32_t dtype, void* out, int32_t out_dtype,
                    void* workspace, size_t workspace_bytes, void* stream) {
  if (dtype < 0 || dtype > 2 || out_dtype < 0 || out_dtype > 2 || channels < 1 || num_rows < 0 || !out || !workspace ||
      (num_rows > 0 && !rows))
    return WCN_ERR_INVALID_ARGUMENT;
  if (workspace_bytes < wcn_column_sums_workspace_bytes(channels)) return WCN_ERR_WORKSPACE;
  WcnColumnSums c = {(float*)workspace, 0, channels, out, out_dtype};
  const int st = wcn_column_sums_first(rows, num_rows, dtype, &c, (hipStream_t)stream);
  return st != WCN_OK ? st : wcn_column_sums_second(c, (hipStream_t)stream);
}

}  // extern "C"
