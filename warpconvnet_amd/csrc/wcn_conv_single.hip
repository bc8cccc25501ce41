// Feature contraction for maps in which every output row has exactly one pair (gfx950, MFMA): the
// transposed convolution that undoes a strided one whose kernel is as large as its stride (the
// decoder's up-sampling of a U-Net: every fine voxel has one parent and lies at one offset from it).
//
//   out[out_k[p], :] = act(bias + X[in_k[p], :] @ W[k] + residual[out_k[p], :])     for every pair p
//
// Nothing is accumulated across pairs, so there are no sums to keep anywhere, no phases and no order
// the pairs of an offset have to be in: the lists are taken as they are (a forward map with its
// lists exchanged is not re-ordered first), cut into tiles of 64 to 256 pairs of one offset.  A workgroup
// of four waves walks a contiguous stretch of tiles with W[k]^T of the current offset in LDS (loaded
// again when the offset changes); a wave takes one to four blocks of 16 pairs, whose list entries it has asked for a tile
// ahead.  The product is transposed: W[k]^T is the A operand (rows = output channels, read from LDS), the gathered rows
// are the B operand and go from memory straight into registers in operand layout (lane = pair,
// 8 channels), so a lane ends up with 4 consecutive output channels of one pair in each of two 16-channel blocks;
// neighbouring quarters of the wave exchange halves and store 16 bytes.  Output channels are walked 32 at a time with the
// gathered rows kept.
// What bounds it: the way of a wave's rows and stores through memory, so the number of waves in flight: 128 registers and fewer
// leave four a SIMD (64 channels at a time with four blocks of rows took 130 to 244: one to three).  bf16, kernel and stride 2, us:
// 32 -> 32 over 1,000,000 fine rows 52 -> 41, 64 -> 32 over 550,000 40 -> 25, 128 -> 64 over 130,000 24 -> 18; over the
// levels of one scan of 60,000 voxels (where smaller tiles make more workgroups) 256 -> 128 23 -> 13, 128 -> 64 12 -> 8.
// Replaces the same reference path as the other kernels (sparse_conv.py:495-544 + the native GEMMs
// it calls) for this kind of map.
#include <algorithm>
#include <mutex>

#include "wcn_common.h"
#include "wcn_conv_args.h"
#include "wcn_mma.h"

namespace {

using namespace wcn_mma;

constexpr int SINGLE_WAVES = 4;
// 16-pair blocks of a wave: what leaves four waves a SIMD (128 registers)
constexpr int single_bpw(int ks) { return ks <= 2 ? 4 : ks <= 4 ? 2 : 1; }
constexpr int single_tile(int ks) { return SINGLE_WAVES * single_bpw(ks) * 16; }  // pairs per tile

// KS: 32-channel steps of the gathered rows (c_in = 32 KS)
template <typename T, int KS>
__global__ void __launch_bounds__(SINGLE_WAVES * 64, 4) conv_fwd_single(ConvArgs a, WcnSingleTiles tt) {
  typedef typename Mma<T>::V V;
  extern __shared__ __attribute__((aligned(16))) unsigned char single_smem[];
  constexpr int BPW = single_bpw(KS), TILE = single_tile(KS);
  constexpr int ROW_BYTES = KS * 64 + 16;  // a row of W[k]^T (c_in values) plus 16 bytes: the operand reads of
                                           // 16 consecutive rows then fall into distinct banks
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int p = lane & 15, kg = lane >> 4;
  const int ncb = (a.c_out + 15) / 16;     // 16-channel blocks of output channels
  const int npairs = (ncb + 1) / 2;        // pairs of them
  const T* __restrict__ X = (const T*)a.X;
  const T* __restrict__ Wt = (const T*)a.Wt;
  T* __restrict__ out = (T*)a.out;
  const int per_wg = (tt.total + (int)gridDim.x - 1) / (int)gridDim.x;
  const int t_begin = (int)blockIdx.x * per_wg;
  const int t_end = t_begin + per_wg < tt.total ? t_begin + per_wg : tt.total;
  if (t_begin >= t_end) return;  // (the whole workgroup)
  // the entries of this lane's pairs of a tile in offset `of`; a place without a pair: -1
  auto entries = [&](int tile, int of, int32_t (&irow)[BPW], int32_t (&orow)[BPW]) {
    const int run_end = tt.first_pair[of + 1];
    const int p0 = tt.first_pair[of] + (tile - tt.first_tile[of]) * TILE + wave * (BPW * 16) + p;
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
      const bool live = p0 + b * 16 < run_end;
      irow[b] = live ? a.in_maps[p0 + b * 16] : -1;
      orow[b] = live ? a.out_maps[p0 + b * 16] : -1;
    }
  };
  int k = 0, loaded = -1;
  while (k + 1 < a.K && t_begin >= tt.first_tile[k + 1]) ++k;  // tiles ascend in offset
  int32_t irow[BPW], orow[BPW];
  entries(t_begin, k, irow, orow);
  for (int tile = t_begin; tile < t_end; ++tile) {
    // the wave's rows, in MFMA operand layout
    V B[BPW][KS];
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
      const bool ok = (uint32_t)irow[b] < (uint64_t)a.num_in && (uint32_t)orow[b] < (uint64_t)a.num_out;
      if (!ok) orow[b] = -1;
      const T* row = X + (int64_t)(ok ? irow[b] : 0) * a.c_in + kg * 8;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) B[b][ks] = *reinterpret_cast<const V*>(row + ks * 32);
    }
    if (k != loaded) {
      __syncthreads();  // everybody has finished with the previous offset's tile
      const u32x4* src = reinterpret_cast<const u32x4*>(Wt + (int64_t)k * a.c_out_pad * a.c_in_pad);
      const int pieces = ncb * 16 * KS * 4;  // 16-byte pieces: KS * 4 per row (the tiles are zero padded beyond c_out)
      for (int i = tid; i < pieces; i += SINGLE_WAVES * 64) {
        const int row = i / (KS * 4), part = i % (KS * 4);
        *reinterpret_cast<u32x4*>(single_smem + row * ROW_BYTES + part * 16) =
            src[(int64_t)row * (a.c_in_pad / 8) + part];
      }
      __syncthreads();
      loaded = k;
    }
    int32_t next_irow[BPW], next_orow[BPW];  // asked for a tile ahead
    if (tile + 1 < t_end) {
      while (k + 1 < a.K && tile + 1 >= tt.first_tile[k + 1]) ++k;
      entries(tile + 1, k, next_irow, next_orow);
    }
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
          if (h == 0 || cp * 2 + 1 < ncb) {  // uniform
            const V A = *reinterpret_cast<const V*>(single_smem + (cp * 32 + h * 16 + p) * ROW_BYTES + (ks * 32 + kg * 8) * 2);
#pragma unroll
            for (int b = 0; b < BPW; ++b) acc[h][b] = Mma<T>::mma(A, B[b][ks], acc[h][b]);
          }
        }
      }
      // Lane (p, kg) holds channels 4 kg .. + 3 of pair p in both blocks; lanes kg and kg ^ 1 exchange four, so that each has
      // eight of one block and stores 16 bytes.
      float bias[2][4] = {};
      if (a.bias) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (cp * 32 + h * 16 + 4 * kg < a.c_out) load_floats<T, 4>((const T*)a.bias + cp * 32 + h * 16 + 4 * kg, bias[h]);
      }
      const int col = cp * 32 + (kg & 1) * 16 + (kg >> 1) * 8;
#pragma unroll
      for (int b = 0; b < BPW; ++b) {
        uint32_t half[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float r[4] = {0.f, 0.f, 0.f, 0.f};
          if (a.residual && orow[b] >= 0 && cp * 32 + h * 16 + 4 * kg < a.c_out)
            load_floats<T, 4>((const T*)a.residual + (int64_t)orow[b] * a.c_out + cp * 32 + h * 16 + 4 * kg, r);
          T t[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float f = acc[h][b][e];
            if (a.bias_rounded) f = to_float(from_float<T>(f));
            f = f + bias[h][e] + r[e];
            if (a.relu) f = f < 0.f ? 0.f : f;
            t[e] = from_float<T>(f);
          }
          const uint2 two = *reinterpret_cast<const uint2*>(t);
          half[h][0] = two.x;
          half[h][1] = two.y;
        }
        u32x4 eight;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const auto swapped = __builtin_amdgcn_permlane16_swap(half[0][i], half[1][i], false, false);
          eight[i] = swapped[0];
          eight[2 + i] = swapped[1];
        }
        if (orow[b] >= 0 && col < a.c_out)  // c_out is a multiple of 8: all eight or none
          *reinterpret_cast<u32x4*>(out + (int64_t)orow[b] * a.c_out + col) = eight;
      }
    }
#pragma unroll
    for (int b = 0; b < BPW; ++b) {
      irow[b] = next_irow[b];
      orow[b] = next_orow[b];
    }
  }
}

inline int single_cus() {
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

template <typename T, int KS>
int launch_single(const ConvArgs& a, const WcnSingleTiles& tt, hipStream_t s) {
  const int ncb = (a.c_out + 15) / 16;
  const int lds = ncb * 16 * (KS * 64 + 16);
  if (lds > 160 * 1024) return WCN_ERR_INVALID_ARGUMENT;
  const void* fn = (const void*)conv_fwd_single<T, KS>;
  // more than 64 KiB of dynamic LDS has to be allowed once per device and kernel (the largest is asked for)
  static std::mutex mu;
  static bool allowed[64] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return WCN_ERR_LAUNCH;
  {
    std::lock_guard<std::mutex> hold(mu);
    if (!allowed[device]) {
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess)
        return WCN_ERR_LAUNCH;
      allowed[device] = true;
    }
  }
  // workgroups per CU: four waves a SIMD, and what LDS holds
  const int per_cu = std::max(1, std::min(4, (160 * 1024) / lds));
  const unsigned grid = (unsigned)std::min<int64_t>(tt.total, (int64_t)single_cus() * per_cu);
  hipLaunchKernelGGL((conv_fwd_single<T, KS>), dim3(grid), dim3(SINGLE_WAVES * 64), lds, s, a, tt);
  wcn_conv_note_kernel("conv_fwd_single<%s, %d>", wcn_type_text<T>(), KS);
  return hipGetLastError() == hipSuccess ? WCN_OK : WCN_ERR_LAUNCH;
}

template <typename T>
int launch_single_typed(const ConvArgs& a, const WcnSingleTiles& tt, hipStream_t s) {
  switch (a.c_in / 32) {
    case 1: return launch_single<T, 1>(a, tt, s);
    case 2: return launch_single<T, 2>(a, tt, s);
    case 3: return launch_single<T, 3>(a, tt, s);
    case 4: return launch_single<T, 4>(a, tt, s);
    case 6: return launch_single<T, 6>(a, tt, s);
    case 8: return launch_single<T, 8>(a, tt, s);
    default: return WCN_ERR_INVALID_ARGUMENT;
  }
}

}  // namespace

// 16-bit rows of 32, 64, 96, 128, 192 or 256 input channels that are whole 16-byte vectors on both
// sides, at most 64 offsets, at most 256 output channels.
bool wcn_conv_single_takes(int dtype, int c_in, int c_out, int num_offsets) {
  if (dtype != WCN_DTYPE_F16 && dtype != WCN_DTYPE_BF16) return false;
  if (c_in % 32 != 0 || c_out % 8 != 0 || c_out < 8 || c_out > 256 || num_offsets < 1 || num_offsets > WCN_SINGLE_MAX_OFFSETS)
    return false;
  const int ks = c_in / 32;
  return ks == 1 || ks == 2 || ks == 3 || ks == 4 || ks == 6 || ks == 8;
}

int wcn_conv_single_launch(const ConvArgs& a, int dtype, const int64_t* host_offsets, hipStream_t s) {
  WcnSingleTiles tt;
  const int tile = single_tile(a.c_in / 32);
  int64_t tiles = 0;
  for (int k = 0; k < a.K; ++k) {
    tt.first_tile[k] = (int32_t)tiles;
    tt.first_pair[k] = (int32_t)host_offsets[k];
    tiles += (host_offsets[k + 1] - host_offsets[k] + tile - 1) / tile;
  }
  if (tiles > INT32_MAX || host_offsets[a.K] > INT32_MAX) return WCN_ERR_INVALID_ARGUMENT;
  for (int k = a.K; k <= WCN_SINGLE_MAX_OFFSETS; ++k) {
    tt.first_tile[k] = (int32_t)tiles;
    tt.first_pair[k] = (int32_t)host_offsets[a.K];
  }
  tt.total = (int32_t)tiles;
  if (tiles == 0) return WCN_OK;
  return dtype == WCN_DTYPE_F16 ? launch_single_typed<_Float16>(a, tt, s) : launch_single_typed<__bf16>(a, tt, s);
}
