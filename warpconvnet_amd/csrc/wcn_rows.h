// Feature rows in 16-byte pieces and the walk over a map's rows form, shared by the pooling and the
// depthwise kernels (gfx950).
#ifndef WCN_ROWS_H_
#define WCN_ROWS_H_
#include "wcn_common.h"
#include "wcn_mma.h"

namespace wcn_rows {

using namespace wcn_mma;

template <typename T>
struct Piece {  // 16 bytes of channels
  static constexpr int N = 16 / sizeof(T);
  typedef T Vec __attribute__((ext_vector_type(N)));
  Vec v;
};

// Holds the compiler to loads that have been asked for together: left alone it moves each one (or the
// first conversion of its data) into the branch that uses it, and a wave then waits for one row at a time.
template <typename T, int U>
__device__ __forceinline__ void together(Piece<T> (&x)[U]) {
#pragma unroll
  for (int u = 0; u < U; ++u) asm volatile("" : "+v"(x[u].v));
}

// One 16-byte piece of row `row`, channels c0 .. c0 + N - 1 (zeros past the last channel).  VEC: rows whose
// byte length is a multiple of 16; others are read element by element.  It is a template parameter
// and not a flag: with a branch between them the loads of several rows were no longer in flight together.
template <typename T, bool VEC>
__device__ __forceinline__ Piece<T> load_raw(const T* __restrict__ base, int64_t row, int channels, int c0) {
  Piece<T> p;
  const T* src = base + row * channels + c0;
  if (VEC) {
    p.v = *reinterpret_cast<const typename Piece<T>::Vec*>(src);
  } else {
#pragma unroll
    for (int j = 0; j < Piece<T>::N; ++j) p.v[j] = c0 + j < channels ? src[j] : (T)0.f;
  }
  return p;
}

template <typename T, bool VEC>
__device__ __forceinline__ void load_piece(const T* __restrict__ base, int64_t row, int channels, int c0, float* out) {
  const Piece<T> p = load_raw<T, VEC>(base, row, channels, c0);
#pragma unroll
  for (int j = 0; j < Piece<T>::N; ++j) out[j] = to_float(p.v[j]);
}

template <typename T, bool VEC>
__device__ __forceinline__ void store_piece(T* __restrict__ base, int64_t row, int channels, int c0, const float* val) {
  constexpr int N = Piece<T>::N;
  T* dst = base + row * channels + c0;
  if (VEC) {
    Piece<T> p;
#pragma unroll
    for (int j = 0; j < N; ++j) p.v[j] = from_float<T>(val[j]);
    *reinterpret_cast<typename Piece<T>::Vec*>(dst) = p.v;
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (c0 + j < channels) dst[j] = from_float<T>(val[j]);
  }
}

inline bool rows_are_vectors(const void* p, int channels, int dtype) {
  const size_t es = dtype == WCN_DTYPE_F32 ? 4 : 2;
  return ((size_t)channels * es) % 16 == 0 && ((uintptr_t)p % 16) == 0;
}

// A workgroup of 256 threads takes `rows` whole rows at a time, a thread per 16-byte piece (rows of
// more than 256 pieces: one row, 256 pieces after the other).  No division inside the row loop: the
// 64-bit quotient of a flat index cost as much as a piece's arithmetic.
struct RowTiling {
  int pieces;  // per row
  int width;   // pieces side by side
  int rows;    // rows side by side
};
inline RowTiling row_tiling(int channels, int dtype) {
  const int per = dtype == WCN_DTYPE_F32 ? 4 : 8;
  RowTiling t;
  t.pieces = (channels + per - 1) / per;
  t.width = t.pieces < 256 ? t.pieces : 256;
  t.rows = 256 / t.width;
  return t;
}

// The first pass of column sums (WcnColumnSums) as a kernel reads it.  A workgroup of 256 threads sums a stretch of `per` rows,
// a thread per 16 bytes of channels, four rows in flight.  s_sum: 256 (Piece<T>::N + 1) floats.
struct ColumnPart {
  const void* rows;
  float* partial;
  int64_t n, per;
  RowTiling tiling;
  int32_t channels;
};
template <class Sums>
inline ColumnPart column_part_of(const void* rows, int64_t n, int dtype, const Sums& c) {
  return {rows, c.partial, n, c.parts > 0 ? (n + c.parts - 1) / c.parts : 0, row_tiling(c.channels > 0 ? c.channels : 1, dtype), c.channels};
}
template <typename T, bool VEC>
__device__ __forceinline__ void column_part(const ColumnPart& c, int part, float* s_sum) {
  constexpr int N = Piece<T>::N, U = 4;
  const T* const X = (const T*)c.rows;
  const RowTiling tiling = c.tiling;
  const int sub = (int)threadIdx.x / tiling.width, at = (int)threadIdx.x % tiling.width;
  const int64_t begin = part * c.per, end = begin + c.per < c.n ? begin + c.per : c.n;
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
          x[u] = load_raw<T, VEC>(X, r < end ? r : end - 1, c.channels, c0);
          if (r >= end) x[u] = Piece<T>{};
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < N; ++j) acc[j] += to_float(x[u].v[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) s_sum[threadIdx.x * (N + 1) + j] = acc[j];
    __syncthreads();
    if (sub == 0 && p0 + at < tiling.pieces) {
      for (int l = 1; l < tiling.rows; ++l)
#pragma unroll
        for (int j = 0; j < N; ++j) acc[j] += s_sum[(l * tiling.width + at) * (N + 1) + j];
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (c0 + j < c.channels) c.partial[(int64_t)part * c.channels + c0 + j] = acc[j];
    }
    __syncthreads();
  }
}

// Entries of one row of a rows form, U at a time in ascending offset: f(k[U], r[U], live[U]).  Where there are
// fewer than U, or an entry is no row of the `limit` there are, live is false and r names a row that can be
// read all the same (limit >= 1): the U row numbers are loaded without a branch between them, and so are the U feature
// rows the caller asks for.
template <int U, typename F>
__device__ __forceinline__ void walk_word(uint32_t word, int k0, int first, const int32_t* __restrict__ row_in,
                                          int64_t limit, F&& f) {
  const int last = first + __popc(word) - 1;
  int e = first;
  for (uint32_t bits = word; bits; e += U) {
    int k[U];
    int32_t r[U];
    bool live[U];
#pragma unroll
    for (int u = 0; u < U; ++u) r[u] = row_in[e + u < last ? e + u : last];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      k[u] = k0 + (__ffs(bits) - 1);
      live[u] = bits != 0 && (uint32_t)r[u] < (uint64_t)limit;
      r[u] = (uint32_t)r[u] < (uint64_t)limit ? r[u] : 0;
      bits &= bits - 1u;
    }
    f(k, r, live);
  }
}

template <int U, typename F>
__device__ __forceinline__ void walk_row(const uint32_t* __restrict__ row_mask, int words,
                                         const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ row_in,
                                         int64_t m, int64_t limit, F&& f) {
  int first = row_ptr[m];  // of the word's entries
  for (int w = 0; w < words; ++w) {
    const uint32_t word = row_mask[m * words + w];
    walk_word<U>(word, w * 32, first, row_in, limit, f);
    first += __popc(word);
  }
}

}  // namespace wcn_rows
#endif  // WCN_ROWS_H_
