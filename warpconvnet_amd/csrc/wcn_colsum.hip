// Column sums of a (rows, channels) array in fp32 (gfx950): the gradient of a layer's bias.
#include <algorithm>

#include "wcn_conv_args.h"
#include "wcn_rows.h"

namespace {

using namespace wcn_rows;

constexpr int PARTS = 512;  // workgroups of the first pass: two per CU

// HBM-bound (5 TB/s): 500 k rows of 64 fp16 channels (64 MB) in 12 + 4 us, where a generic column reduction took 34.
template <typename T, bool VEC>
__global__ void __launch_bounds__(256) column_sums(ColumnPart c) {
  __shared__ float s_sum[256 * (Piece<T>::N + 1)];
  column_part<T, VEC>(c, (int)blockIdx.x, s_sum);
}

template <typename OT>
__global__ void __launch_bounds__(256) column_sums_finish(WcnColumnSums s) {
  wcn_column_sums_finish<OT>(s, (int)blockIdx.x * 16, (OT*)s.out);
}

inline int column_parts(int64_t n, int rows) {  // at least four rows per thread in a part
  return (int)std::max<int64_t>(1, std::min<int64_t>(PARTS, n / (4 * rows)));
}

}  // namespace

void wcn_column_sums_parts(int64_t num_rows, int dtype, WcnColumnSums* c) {
  c->parts = column_parts(num_rows, row_tiling(c->channels, dtype).rows);
}

int wcn_column_sums_first(const void* rows, int64_t num_rows, int dtype, const WcnColumnSums& c, hipStream_t s) {
  const bool vec = rows_are_vectors(rows, c.channels, dtype);
  const ColumnPart part = column_part_of(rows, num_rows, dtype, c);
  auto first = [&](auto v) {
    using T = decltype(v);
    hipLaunchKernelGGL((vec ? column_sums<T, true> : column_sums<T, false>), dim3((unsigned)c.parts), dim3(256), 0, s, part);
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
  wcn_column_sums_parts(num_rows, dtype, &c);
  const int st = wcn_column_sums_first(rows, num_rows, dtype, c, (hipStream_t)stream);
  return st != WCN_OK ? st : wcn_column_sums_second(c, (hipStream_t)stream);
}

}  // extern "C"
