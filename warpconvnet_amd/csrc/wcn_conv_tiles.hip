// Feature contraction over a tile plan (gfx950, MFMA): 16-bit rows, tiles of 128 output rows whose pairs lie in
// few offsets (wcn_tiles.hip).
//
//   out[m, :] = bias + sum_k X[in_k(m), :] @ W[k]        (in_k(m): the input row paired with output
//                                                          row m in offset k, if there is one)
//
// A workgroup of four waves owns 128 output rows x TN output channels (TN = 32 NBW), a wave 64 rows x TN / 2
// channels, with the fp32 sums in registers from the tile's first offset to its last.  A step is one offset and KC input
// channels: the 128 gathered rows' slices and the TN rows of W[k]^T, both fetched from memory straight into LDS
// (global_load_lds, 16 bytes per lane, neighbouring lanes a row: whole cache lines), D - 1 steps before they are
// multiplied.  One barrier per step, which waits for what is due and leaves the newest loads in flight.  A place
// of the tile without a pair in the offset reads a block of zeros.  The sums of a row come in ascending offset and
// channel, whatever the tile: results are bitwise reproducible, and the same as those of the pair-packed kernel.
//
// LDS: D buffers of both operands and the tile's input rows (at most 16 KB), so that two or three workgroups
// share a CU and one's start and end pass beside the other's multiplications.  Rows of an LDS buffer lie without
// padding; the 16-byte piece p of row r sits at p ^ (bits of r), which is arranged on the source side: a lane
// fetches the piece that belongs where its data lands.
//
// What bounds it: the way of both operands out of the L2 into LDS (256 -> 256 over 39 k rows 10 TB/s with the matrix pipes 36 %
// busy, 64 -> 64 over 157 k 16 TB/s; behind the L2 it moves 2 to 5), and for few rows the longest tile.  Tried: 256-row
// tiles of eight waves (a quarter to a half less weight traffic, one workgroup per CU: 10 to 30 % slower), deeper buffers with fewer workgroups
// (the same or slower).  Tiles in descending length (the plan's order) instead of ascending: 128 -> 128 over 170 k rows
// 116 -> 84 us, 256 -> 256 over 39 k rows 138 -> 89.
#include <algorithm>
#include <mutex>

#include "wcn_common.h"
#include "wcn_conv_args.h"
#include "wcn_mma.h"

namespace {

using namespace wcn_mma;

constexpr int TM = WCN_TILE_ROWS;


// 16 bytes per lane from g to LDS at lds_off + 16 * lane (counted by vmcnt)
__device__ __forceinline__ void to_lds(const char* g, uint32_t lds_off) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_off) : "memory");
}
template <typename T, int NBW, int KC, int D>
struct TileCfg {
  static constexpr int TN = 32 * NBW, WAVES = 4;
  static constexpr int LPR = KC / 8;        // lanes (16-byte pieces) of a row's slice
  static constexpr int RPI = 64 / LPR;      // rows of one load
  static constexpr int A_BYTES = TM * KC * 2, B_BYTES = TN * KC * 2;
  static constexpr int NA = 32 / RPI;                     // row loads of a wave and step
  static constexpr int B_LOADS = TN / RPI;                // weight loads of a step
  static constexpr int NB = (B_LOADS + WAVES - 1) / WAVES;            // ... of a wave
  static constexpr int SUM_STRIDE = TN * 4 + 16;          // bytes of a row of sums in LDS
  static constexpr int RING_BYTES = D * (A_BYTES + B_BYTES), SUM_BYTES = 64 * SUM_STRIDE;
  static constexpr int NAN_AT = RING_BYTES - 16;          // a word per wave: whether it has a NaN among its sums
  static_assert(SUM_BYTES <= NAN_AT, "the sums are put in rows beside these words");
  static int lds(int K) { return std::max(RING_BYTES + (K + 1) / 2 * 1024, SUM_BYTES); }
};

template <typename T, int NBW, int KC, int D>
__global__ void __launch_bounds__(256, 2) conv_fwd_tiles(ConvArgs a, WcnTilePlan plan, int col_groups) {
  typedef TileCfg<T, NBW, KC, D> C;
  typedef typename Mma<T>::V V;
  extern __shared__ __attribute__((aligned(16))) char tiles_smem[];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tiles_smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int c = lane & 15, g = lane >> 4;
  // workgroups of a tile's column groups follow one another on one XCD (blockIdx % 8): they gather the same rows
  const int b8 = (int)blockIdx.x >> 3;
  const int64_t tile = (int64_t)(b8 / col_groups) * 8 + ((int)blockIdx.x & 7);
  const int col0 = (b8 % col_groups) * C::TN;
  if (tile >= plan.tiles) return;
  const int K = a.K;
  const uint32_t row_bytes = (uint32_t)a.c_in * 2u;
  const int NCH = (a.c_in + KC - 1) / KC;  // chunks of a row
  const uint32_t all = __builtin_amdgcn_readfirstlane(plan.mask[tile]);
  const int n_off = __popc(all), S = n_off * NCH;
  int32_t* const table = reinterpret_cast<int32_t*>(tiles_smem + C::RING_BYTES);  // n_off x TM input rows
  const char* const zeros = (const char*)plan.zeros + lane * 16;
  // this lane's place in a load: row lane / LPR of RPI, and the piece that belongs at its 16 bytes
  const int l_row = lane / C::LPR, l_slot = lane % C::LPR;
  auto piece_of = [&](int row) { return KC == 64 ? l_slot ^ ((row >> 1) & 7) : l_slot ^ ((row >> 2) & 3); };
  uint32_t a_piece[C::NA];
#pragma unroll
  for (int i = 0; i < C::NA; ++i) {
    a_piece[i] = (uint32_t)piece_of(i * C::RPI + l_row) * 16u;  // the wave's first row is a multiple of 32
  }
  const char* b_src[C::NB];
  uint32_t b_dst[C::NB];
#pragma unroll
  for (int i = 0; i < C::NB; ++i) {
    const int load = (i * C::WAVES + wave) % C::B_LOADS;  // past the last: one of the first again
    const int row = load * C::RPI + l_row;
    const int n = col0 + row < a.c_out_pad ? col0 + row : a.c_out_pad - 1;  // past the last channel: its sums are not stored
    b_src[i] = (const char*)a.Wt + ((size_t)n * a.c_in_pad) * 2 + piece_of(row) * 16;
    b_dst[i] = lds0 + D * C::A_BYTES + load * 1024;
  }
  const size_t w_tile_bytes = (size_t)a.c_out_pad * a.c_in_pad * 2;

  struct Cursor {  // step: the j-th offset of the tile and the chunk
    int j, chunk;
  };
  auto next = [&](Cursor& q) {
    if (++q.chunk == NCH) {
      q.chunk = 0;
      ++q.j;
    }
  };
  auto fetch_rows = [&](const Cursor& q, int buf) {
    const uint32_t at = (uint32_t)q.chunk * (KC * 2), limit = q.j < n_off ? row_bytes : 0u;
    int32_t in[C::NA];
#pragma unroll
    for (int i = 0; i < C::NA; ++i) in[i] = table[(q.j < n_off ? q.j : 0) * TM + wave * 32 + i * C::RPI + l_row];
#pragma unroll
    for (int i = 0; i < C::NA; ++i) {
      // both addresses are made and one is chosen: no branches between the loads
      const char* row = (const char*)a.X + (size_t)(uint32_t)(in[i] < 0 ? 0 : in[i]) * row_bytes + (at + a_piece[i]);
      asm("" : "+v"(row));
      const bool there = (in[i] >= 0) & (at + a_piece[i] < limit);
      to_lds(there ? row : zeros, lds0 + buf * C::A_BYTES + wave * (32 * KC * 2) + i * 1024);
    }
  };
  auto fetch_weights = [&](int k, int chunk, int buf) {
    const size_t at = (size_t)k * w_tile_bytes + (size_t)chunk * (KC * 2);
#pragma unroll
    for (int i = 0; i < C::NB; ++i) to_lds(b_src[i] + at, b_dst[i] + buf * C::B_BYTES);
  };

  f32x4 acc[4][NBW];
  auto clear = [&]() {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < NBW; ++cb) acc[rb][cb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  // the operands of 32 channels of a step out of a buffer
  auto operands = [&](int buf, int ks, V (&x)[4], V (&w)[NBW]) {
    const char* const A = tiles_smem + buf * C::A_BYTES + wr * (64 * KC * 2);
    const char* const B = tiles_smem + D * C::A_BYTES + buf * C::B_BYTES + wc * (16 * NBW * KC * 2);
    auto at = [&](int row) {
      const int p = ks * 4 + g;
      return row * (KC * 2) + (KC == 64 ? p ^ ((row >> 1) & 7) : p ^ ((row >> 2) & 3)) * 16;
    };
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) x[rb] = *reinterpret_cast<const V*>(A + at(rb * 16 + c));
#pragma unroll
    for (int cb = 0; cb < NBW; ++cb) w[cb] = *reinterpret_cast<const V*>(B + at(cb * 16 + c));
  };
  clear();

  if (S > 0) {
    // the rows' numbers, offset by offset, as they lie in the plan: 1 KiB per load, two offsets (the plan has room behind
    // its last)
    const char* const nbr = (const char*)(plan.nbr + tile * K * TM) + lane * 16;
    for (int i = wave; i < (n_off + 1) / 2; i += C::WAVES) to_lds(nbr + i * 1024, lds0 + C::RING_BYTES + i * 1024);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // step s multiplies what buffer s % D holds; it was asked for D - 1 steps before
    Cursor qa{0, 0}, qb{0, 0};
    uint32_t rest = all;  // offsets from qb's on
    int kb = __builtin_ctz(rest), steps_b = 0;
    auto fetch = [&](int buf) {
      fetch_weights(kb, qb.chunk, buf);
      fetch_rows(qa, buf);
      next(qa);
      if (++steps_b < S && ++qb.chunk == NCH) {  // past the last step: the last weights again
        qb.chunk = 0;
        rest &= rest - 1u;
        kb = __builtin_ctz(rest);
      }
    };
#pragma unroll
    for (int i = 0; i < D - 1; ++i) fetch(i);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * (C::NA + C::NB)) : "memory");
    int buf = 0;
    for (int s = 0; s < S; ++s) {
      fetch(buf == 0 ? D - 1 : buf - 1);
#pragma unroll
      for (int ks = 0; ks < KC / 32; ++ks) {
        V x[4], w[NBW];
        operands(buf, ks, x, w);
#pragma unroll
        for (int cb = 0; cb < NBW; ++cb)
#pragma unroll
          for (int rb = 0; rb < 4; ++rb) acc[rb][cb] = Mma<T>::mma(w[cb], x[rb], acc[rb][cb]);
      }
      buf = buf == D - 1 ? 0 : buf + 1;
      // what the next step multiplies has landed, here and, behind the barrier, everywhere
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * (C::NA + C::NB)) : "memory");
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");

    // A place without a pair has multiplied zeros, and zero times an infinite or NaN weight is NaN: a tile with one among its
    // sums is gone through again, a step at a time, with such products left out.
    bool nan = false;
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < NBW; ++cb)
#pragma unroll
        for (int e = 0; e < 4; ++e) nan |= acc[rb][cb][e] != acc[rb][cb][e];
    uint32_t* const words = reinterpret_cast<uint32_t*>(tiles_smem + C::NAN_AT);
    const bool any = __ballot(nan) != 0ull;
    if (lane == 0) words[wave] = any ? 1u : 0u;
    __syncthreads();
    const u32x4 found = *reinterpret_cast<const u32x4*>(words);
    if (__builtin_amdgcn_readfirstlane(found[0] | found[1] | found[2] | found[3]) != 0u) {
      clear();
      Cursor q{0, 0};
      rest = all;
#pragma nounroll
      for (int s = 0; s < S; ++s) {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the buffer (and the words above) have been read
        fetch_weights(__builtin_ctz(rest), q.chunk, 0);
        fetch_rows(q, 0);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        bool pair[4];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb) pair[rb] = table[q.j * TM + wr * 64 + rb * 16 + c] >= 0;
#pragma unroll
        for (int ks = 0; ks < KC / 32; ++ks) {
          V x[4], w[NBW];
          operands(0, ks, x, w);
#pragma unroll
          for (int cb = 0; cb < NBW; ++cb)
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
              const f32x4 with = Mma<T>::mma(w[cb], x[rb], acc[rb][cb]);
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[rb][cb][e] = pair[rb] ? with[e] : acc[rb][cb][e];
            }
        }
        next(q);
        if (q.chunk == 0) rest &= rest - 1u;
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }

  // ---- the sums in rows through LDS, 64 rows at a time, then bias, residual, clamp, one rounding, whole 16-byte stores ----
  constexpr int PIECES = C::TN / 8, PASS = C::WAVES * 64 / PIECES, RT = (64 + PASS - 1) / PASS;  // PASS rows side by side, RT of them per thread
  const int piece = tid % PIECES, col = col0 + piece * 8;
  const bool writes = tid < PASS * PIECES && col < a.c_out;
  float b[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (a.bias && writes) {
#pragma unroll
    for (int e = 0; e < 8; ++e) b[e] = to_float(((const T*)a.bias)[col + e]);
  }
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    int32_t place[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int row = tid / PIECES + i * PASS;
      place[i] = plan.order[tile * TM + half * 64 + (row < 64 ? row : 63)];
    }
    if (half > 0) __syncthreads();
    if (wr == half) {
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int cb = 0; cb < NBW; ++cb) {
          const int row = rb * 16 + c, at = (wc * NBW + cb) * 16 + 4 * g;
          *reinterpret_cast<f32x4*>(tiles_smem + row * C::SUM_STRIDE + at * 4) = acc[rb][cb];
        }
    }
    __syncthreads();
    if (!writes) continue;
    u32x4 res[RT];
    if (a.residual) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
        res[i] = *reinterpret_cast<const u32x4*>(static_cast<const T*>(a.residual) + (int64_t)(place[i] < 0 ? 0 : place[i]) * a.c_out + col);
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int row = tid / PIECES + i * PASS;
      if (row >= 64 || place[i] < 0) continue;
      const f32x4* src = reinterpret_cast<const f32x4*>(tiles_smem + row * C::SUM_STRIDE + piece * 32);
      const f32x4 lo = src[0], hi = src[1];
      T r[8], t[8];
      if (a.residual) *reinterpret_cast<u32x4*>(r) = res[i];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float f = e < 4 ? lo[e & 3] : hi[e & 3];
        if (a.bias_rounded) f = to_float(from_float<T>(f));
        f += b[e];
        if (a.residual) f += to_float(r[e]);
        if (a.relu) f = f < 0.f ? 0.f : f;
        t[e] = from_float<T>(f);
      }
      *reinterpret_cast<u32x4*>((T*)a.out + (int64_t)place[i] * a.c_out + col) = *reinterpret_cast<const u32x4*>(t);
    }
  }
}

template <typename T, int NBW, int KC, int D>
int launch_tiles(const ConvArgs& a, const WcnTilePlan& plan, hipStream_t s) {
  typedef TileCfg<T, NBW, KC, D> C;
  const void* fn = (const void*)conv_fwd_tiles<T, NBW, KC, D>;
  {  // more than 64 KiB of dynamic LDS has to be allowed once per device and kernel
    static std::mutex mu;
    static bool allowed[64] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return WCN_ERR_LAUNCH;
    std::lock_guard<std::mutex> hold(mu);
    if (!allowed[device]) {
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, C::lds(WCN_TILE_MAX_OFFSETS)) != hipSuccess)
        return WCN_ERR_LAUNCH;
      allowed[device] = true;
    }
  }
  const int cols = (a.c_out + C::TN - 1) / C::TN;
  const int64_t grid = (plan.tiles + 7) / 8 * 8 * cols;
  if (grid > INT32_MAX) return WCN_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL((conv_fwd_tiles<T, NBW, KC, D>), dim3((unsigned)grid), dim3(C::WAVES * 64), C::lds(a.K), s, a, plan, cols);
  wcn_conv_note_kernel("conv_fwd_tiles<%s, %d, %d, %d>", wcn_type_text<T>(), NBW, KC, D);
  return hipGetLastError() == hipSuccess ? WCN_OK : WCN_ERR_LAUNCH;
}

template <typename T>
int launch_typed(const ConvArgs& a, const WcnTilePlan& plan, hipStream_t s) {
  // Slices of 64 channels (a barrier per 64, two workgroups per CU), or of 32 with one more buffer (smaller LDS: three
  // workgroups per CU, for narrow outputs).  Rows of an odd number of 32-channel slices would leave half of the last of
  // 64 empty; up to 64 output channels the third workgroup pays as soon as there are tiles for it (fp16 64 -> 64, us:
  // 39 k rows 22 and 24, 170 k 38 and 37, 300 k 46 and 41, 1 M 132 and 117).
  const bool odd = (a.c_in + 31) / 32 % 2, many = plan.tiles > 1024;
  if (a.c_out <= 32) return launch_tiles<T, 1, 32, 3>(a, plan, s);
  if (a.c_out <= 64)
    return odd || many ? launch_tiles<T, 2, 32, 3>(a, plan, s) : launch_tiles<T, 2, 64, 2>(a, plan, s);
  if (a.c_out <= 96)
    return odd || many ? launch_tiles<T, 3, 32, 3>(a, plan, s) : launch_tiles<T, 3, 64, 2>(a, plan, s);
  return odd ? launch_tiles<T, 4, 32, 3>(a, plan, s) : launch_tiles<T, 4, 64, 2>(a, plan, s);
}

}  // namespace

bool wcn_conv_tiles_takes(int dtype, int num_offsets, int c_in, int c_out) {
  return dtype != WCN_DTYPE_F32 && num_offsets <= WCN_TILE_MAX_OFFSETS && c_in % 8 == 0 && c_out % 8 == 0;
}

// Whether this kernel is the one to take (wcn_conv_tiles_supported).  The lines, from timings over 12,000 to 1 M
// rows of 32 to 256 bf16 channels on surfaces of 37 to 95 % (other kernel -> this one, us, the plan apart):
//   rows        64->64       96->96       128->128     256->256
//     24,000    19 ->  18    42 ->  38     49 ->  41   136 ->  78
//     39,000    30 ->  22    90 ->  39     64 ->  44   164 ->  89
//    170,000    73 ->  37   213 ->  71    188 ->  84   517 -> 273
//    300,000    82 ->  41   255 ->  80    294 ->  91   854 -> 279
//  1,000,000   203 -> 117
// Few rows: the longest tile (all offsets, 0.7 us each per 64 channels) is the time, and the kernel for small maps deals
// its offsets to several waves.  Narrow rows (32 -> 32: 30 -> 24 at 170 k) gain less than a plan costs, and their kernel adds
// the identity's product first: taken over a plan that a wider layer has left, a layer's last bits would tell what ran
// before it (over 4 x 250 k voxels, ten such layers in a network's pass: 1 %).  Pairs spread evenly over the offsets (volume-filling noise): a tile has pairs in two thirds of them,
// whatever the order of the rows, and such maps stay with the other kernels.  A plan takes about 20 us and 0.07 per thousand
// rows; a call saves about 40 ps per pair and 64 x 128 channels (60 with the few offsets of a strided kernel: 96 -> 128,
// 2x2x2, 300 k -> 162 k rows 65 -> 29 us), and `calls` calls over the map are expected.
int wcn_conv_tiles_worth(int K, int c_in, int c_out, int64_t num_out, const int64_t* host_offsets, int identity, int calls) {
  double sum = 0.0, squares = 0.0;
  for (int k = 0; k < K; ++k) {
    if (k == identity) continue;
    const double n = (double)(host_offsets[k + 1] - host_offsets[k]);
    sum += n;
    squares += n * n;
  }
  // effective number of offsets: 26 of 26 for noise, 25 for spheres, 17 to 22 for rooms
  if (squares <= 0.0 || (K > 12 && sum * sum / squares > 0.98 * (K - (identity >= 0 ? 1 : 0)))) return 0;
  if (!wcn_conv_tiles_rows(K, c_in, c_out, num_out)) return 0;
  const double saved = (double)host_offsets[K] * (K <= 12 ? 60e-6 : 40e-6) * ((double)c_in * c_out / 8192.0);
  return saved * calls > 20.0 + 70e-6 * num_out ? 3 : 2;
}

bool wcn_conv_tiles_rows(int K, int c_in, int c_out, int64_t num_out) {
  return num_out >= (K <= 12 || (c_in >= 64 && c_out > 64) ? 16384 : 32768) && !(c_in <= 32 && c_out <= 32);
}

int wcn_conv_tiles_launch(const ConvArgs& a, int dtype, const WcnTilePlan& plan, hipStream_t s) {
  return dtype == WCN_DTYPE_F16 ? launch_typed<_Float16>(a, plan, s)
                                : launch_typed<__bf16>(a, plan, s);
}
