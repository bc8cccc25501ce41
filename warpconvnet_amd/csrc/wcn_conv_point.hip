// Contraction of a layer with one offset and one voxel (gfx950, MFMA): the kernel behind wcn_pointwise_fwd.
//
//   out[m, :] = bias + X[m, :] @ W
//
// (the 1x1x1 convolution of a residual block whose width changes, and of a head; 16-bit rows; in place of a library
// product where gradients are not asked for).  Rows this narrow are moved, not computed:
// 64 -> 32 channels are 64 operations per byte, and the chip does 230.  So:
//
//   * workgroups of four waves, as many as fit, walk tiles of 64 to 256 rows with W^T in LDS, brought there once;
//   * a wave's rows go from memory into registers in operand layout (lane = row, 16 bytes) and are asked for a
//     tile ahead; a row is read once, whatever c_out is;
//   * the product is transposed (W^T is the A operand), so a lane ends up with four channels of a row in each of two 16-channel
//     blocks; lanes of two neighbouring quarters exchange halves (v_permlane16_swap) and store 16 bytes, a wave 64 bytes in a
//     row of its output (four channels a lane and 32 bytes in a row: 32 -> 64 over 1,000,000 rows 55 us, 39 this way).
//
// Measured (bf16, 1,000,000 rows; before: the library's matrix product): 64 -> 32 78 -> 32 us, at 6 TB/s; 64 -> 64 105 -> 54; 32 -> 32
// 135 -> 21; 128 -> 64 144 -> 84, 4.5 TB/s.  What bounds it: memory; the wide ones the stores, 64 bytes of a line at a time.
#include <algorithm>
#include <mutex>

#include "wcn_common.h"
#include "wcn_conv_args.h"
#include "wcn_mma.h"

namespace {

using namespace wcn_mma;

struct PointArgs {
  const void *X, *W, *bias;
  void* out;
  int64_t rows;
  int32_t c_out, tiles;
};

constexpr int POINT_WAVES = 4;
constexpr int POINT_LDS = 80 * 1024;

// KS: 32-channel steps of a row (c_in = 32 KS); BPW: 16-row blocks of a wave
template <typename T, int KS, int BPW>
__global__ void __launch_bounds__(POINT_WAVES * 64, 4) pointwise_fwd(PointArgs a) {
  typedef typename Mma<T>::V V;
  extern __shared__ __attribute__((aligned(16))) unsigned char point_smem[];
  constexpr int C_IN = KS * 32;
  constexpr int ROW_BYTES = KS * 64 + 16;  // a row of W^T plus 16 bytes: 16 consecutive rows are read from distinct banks
  constexpr int TILE = POINT_WAVES * BPW * 16;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane & 15, kg = lane >> 4;
  const int npairs = (a.c_out + 31) / 32;  // pairs of 16-channel blocks of output channels
  const T* __restrict__ X = (const T*)a.X;
  T* __restrict__ out = (T*)a.out;
  const int64_t last = a.rows - 1;
  auto fetch = [&](int tile, V (&B)[BPW][KS]) {
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
      const int64_t m = (int64_t)tile * TILE + (wave * BPW + b) * 16 + p;
      const T* row = X + (m < last ? m : last) * C_IN + kg * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) B[b][ks] = *reinterpret_cast<const V*>(row + ks * 32);
    }
  };
  V B[BPW][KS];
  int tile = blockIdx.x;
  fetch(tile, B);
  {  // W (c_in x c_out) into rows of W^T: a lane takes two rows of eight channels, neighbours neighbouring rows
    const T* __restrict__ W = (const T*)a.W;
    const int have = a.c_out / 8;
    for (int i = tid; i < C_IN / 2 * npairs * 4; i += POINT_WAVES * 64) {
      const int k = i % (C_IN / 2) * 2, n8 = i / (C_IN / 2);
      V w0 = Mma<T>::zero(), w1 = Mma<T>::zero();
      if (n8 < have) {
        w0 = *reinterpret_cast<const V*>(W + (int64_t)k * a.c_out + n8 * 8);
        w1 = *reinterpret_cast<const V*>(W + (int64_t)(k + 1) * a.c_out + n8 * 8);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const T both[2] = {w0[e], w1[e]};
        *reinterpret_cast<uint32_t*>(point_smem + (n8 * 8 + e) * ROW_BYTES + k * 2) = *reinterpret_cast<const uint32_t*>(both);
      }
    }
    __syncthreads();
  }
  while (tile < a.tiles) {
    const int next = tile + (int)gridDim.x;
    V C[BPW][KS];
    fetch(next < a.tiles ? next : tile, C);
    for (int cp = 0; cp < npairs; ++cp) {
      f32x4 acc[2][BPW];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int b = 0; b < BPW; ++b) acc[h][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const V A = *reinterpret_cast<const V*>(point_smem + (cp * 32 + h * 16 + p) * ROW_BYTES + (ks * 32 + kg * 8) * 2);
#pragma unroll
          for (int b = 0; b < BPW; ++b) acc[h][b] = Mma<T>::mma(A, B[b][ks], acc[h][b]);
        }
      }
      // Lane (p, kg) holds channels 4 kg .. + 3 of row p of both blocks; lanes kg and kg ^ 1 exchange four, so that each
      // has eight in a row of one block: stores of 16 bytes, 64 in a row of a wave.
      const int col = cp * 32 + (kg & 1) * 16 + (kg >> 1) * 8;
      float bias[2][4] = {};
      if (a.bias) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (cp * 32 + h * 16 + 4 * kg < a.c_out) load_floats<T, 4>((const T*)a.bias + cp * 32 + h * 16 + 4 * kg, bias[h]);
      }
#pragma unroll
      for (int b = 0; b < BPW; ++b) {
        uint32_t half[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          T t[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) t[e] = from_float<T>(acc[h][b][e] + bias[h][e]);
          const uint2 two = *reinterpret_cast<const uint2*>(t);
          half[h][0] = two.x;
          half[h][1] = two.y;
        }
        u32x4 eight;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto s2 = __builtin_amdgcn_permlane16_swap(half[0][i], half[1][i], false, false);
          eight[i] = s2[0];
          eight[2 + i] = s2[1];
        }
        const int64_t m = (int64_t)tile * TILE + (wave * BPW + b) * 16 + p;
        if (m <= last && col < a.c_out) *reinterpret_cast<u32x4*>(out + m * a.c_out + col) = eight;
      }
    }
    tile = next;
#pragma unroll
    for (int b = 0; b < BPW; ++b)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) B[b][ks] = C[b][ks];
  }
}

inline int point_cus() {
  static std::mutex mu;
  static int cus[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 256;
  std::lock_guard<std::mutex> hold(mu);
  if (cus[device] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || n < 1) n = 256;
    cus[device] = n;
  }
  return cus[device];
}

// rows of W^T in LDS, up to a whole pair of 16-channel blocks
int point_lds(int ks, int c_out) { return (c_out + 31) / 32 * 32 * (ks * 64 + 16); }

template <typename T, int KS, int BPW>
int launch_point(PointArgs a, hipStream_t s) {
  const int lds = point_lds(KS, a.c_out);
  const int64_t tiles = (a.rows + POINT_WAVES * BPW * 16 - 1) / (POINT_WAVES * BPW * 16);
  if (tiles > INT32_MAX || lds > POINT_LDS) return WCN_ERR_INVALID_ARGUMENT;
  {  // more than 64 KiB of dynamic LDS has to be allowed once per device and kernel
    static std::mutex mu;
    static bool allowed[64] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return WCN_ERR_LAUNCH;
    std::lock_guard<std::mutex> hold(mu);
    if (!allowed[device]) {
      if (hipFuncSetAttribute((const void*)pointwise_fwd<T, KS, BPW>, hipFuncAttributeMaxDynamicSharedMemorySize, POINT_LDS) !=
          hipSuccess)
        return WCN_ERR_LAUNCH;
      allowed[device] = true;
    }
  }
  a.tiles = (int32_t)tiles;
  const int per_cu = std::max(1, std::min(4, (160 * 1024) / lds));
  const unsigned grid = (unsigned)std::min<int64_t>(tiles, (int64_t)point_cus() * per_cu);
  hipLaunchKernelGGL((pointwise_fwd<T, KS, BPW>), dim3(grid), dim3(POINT_WAVES * 64), lds, s, a);
  wcn_conv_note_kernel("pointwise_fwd<%s, %d, %d>", wcn_type_text<T>(), KS, BPW);
  return hipGetLastError() == hipSuccess ? WCN_OK : WCN_ERR_LAUNCH;
}

template <typename T>
int launch_point_typed(const PointArgs& a, int c_in, hipStream_t s) {
  switch (c_in / 32) {
    case 1: return launch_point<T, 1, 4>(a, s);
    case 2: return launch_point<T, 2, 2>(a, s);
    case 3: return launch_point<T, 3, 2>(a, s);
    case 4: return launch_point<T, 4, 2>(a, s);
    case 6: return launch_point<T, 6, 1>(a, s);
    case 8: return launch_point<T, 8, 1>(a, s);
    default: return WCN_ERR_INVALID_ARGUMENT;
  }
}

}  // namespace

extern "C" {

// 16-bit rows, whole 16-byte vectors on both sides, of 32 to 96 channels, 128, 192 or 256, whose weight fits twice into the LDS of
// a CU.  Up to 96 channels on both sides whatever the number of rows, wider ones up to 32,768 rows and from 100,000 on.  Between
// the two a weight of 16 KB and more is as long on its way into every workgroup's LDS as the library takes for all of it, and where the
// GPU is what a network waits for the library's product is the one that is 1 to 6 us shorter.  Where the host is, this one is, at any
// size: a library product is called through Python.  us of a layer with a bias called alone, bf16, here / by the library's product:
//     rows            1,000        30,000       60,000       90,000
//     128 -> 64      20 / 36      20 / 38      22 / 38      26 / 47
//     128 -> 128     21 / 36      22 / 37      26 / 40      30 / 51
//     256 -> 128     21 / 36      27 / 38      32 / 42      37 / 56
// (A U-Net over 60,000 voxels, with two such layers of fewer than 32,768 rows: 1,267 / 1,385 us,
// of which two runs of one side differ by 9 %.)  us on the GPU here / the library's matrix product, bf16:
//     rows      32->32      64->32      64->64      96->96      128->64     128->128    192->96     256->128
//      1,000    3 /   4     3 /  4      4 /   4     5 /   5     5 /   4     7 /   5     6 /   6     8 /   6
//     30,000    4 /  22     4 /  6      5 /  19     6 /  27     6 /   8     8 /   7     9 /  12    13 /   9
//     60,000    4 /   9     5 /  6      6 /   7     8 /  12     9 /   8    12 /  10    16 /  14    19 /  13
//    100,000    5 /  23     7 / 14     10 /  20    13 /  29    15 /  24    21 /  22    22 /  37    27 /  28
//    300,000    8 /  58    13 / 26     19 /  51    26 /  75    27 /  62    39 /  40    39 /  93    55 /  55
//  1,000,000   21 / 135    32 / 78     54 / 105    94 / 192    84 / 144   134 / 167   140 / 232   195 / 234
int32_t wcn_pointwise_takes(int64_t num_rows, int32_t c_in, int32_t c_out, int32_t dtype) {
  if (dtype != WCN_DTYPE_F16 && dtype != WCN_DTYPE_BF16) return 0;
  if (num_rows < 1 || num_rows > INT32_MAX || c_in < 32 || c_in > 256 || c_in % 32 != 0 || c_out % 8 != 0 || c_out < 8 || c_out > 1024)
    return 0;
  const int ks = c_in / 32;
  if ((ks > 4 && ks != 6 && ks != 8) || point_lds(ks, c_out) > POINT_LDS) return 0;
  return (c_in <= 96 && c_out <= 96) || num_rows <= 32768 || num_rows >= 100000;
}

int wcn_pointwise_fwd(const void* rows, int64_t num_rows, int32_t c_in, int32_t dtype, const void* weight, int32_t c_out,
                      const void* bias, void* out, void* stream) {
  if (!rows || !weight || !out || !wcn_pointwise_takes(num_rows, c_in, c_out, dtype)) return WCN_ERR_INVALID_ARGUMENT;
  if (((uintptr_t)rows | (uintptr_t)weight | (uintptr_t)out | (uintptr_t)bias) & 15) return WCN_ERR_INVALID_ARGUMENT;
  const PointArgs a = {rows, weight, bias, out, num_rows, c_out, 0};
  return dtype == WCN_DTYPE_F16 ? launch_point_typed<_Float16>(a, c_in, (hipStream_t)stream)
                                : launch_point_typed<__bf16>(a, c_in, (hipStream_t)stream);
}

}  // extern "C"
