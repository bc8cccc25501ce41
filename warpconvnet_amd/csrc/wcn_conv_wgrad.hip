// Weight gradient of the sparse convolution for 16-bit rows of whole 16-byte vectors (gfx950, MFMA):
//
//   dW[k][ci][co] = sum over the pairs p of offset k of  X[in_maps[p]][ci] * dY[out_maps[p]][co]
//
// (the identity offset of a same-size map: over all rows m of X[m] dY[m]; the other element types and ragged rows:
// wcn_conv_bwd.hip).  The pairs of every offset are cut into chunks; a workgroup of four waves owns one chunk
// and one tile of up to 128 x 128 (ci, co), a wave a quarter of it, with the fp32 sums in MFMA accumulators, and writes
// it once; a second kernel adds the chunks of an offset in a fixed order (bitwise reproducible).
//
// A step is 64 pairs.  Their rows of X and of dY go from memory straight into LDS as they are (global_load_lds, 16
// bytes per lane), one step ahead of the multiplications.  The MFMA operands want consecutive PAIRS of one
// channel: ds_read_b64_tr_b16 turns 4 rows x 16 channels into that on the way out of LDS.  (Turned on the way in,
// element by element, a step of 64 x 64 channels took 128 two-byte LDS writes per wave beside 8 MFMAs, and a row was gathered
// once for every 64 channels of the other side.)  Piece p (16 bytes) of row r sits at p ^ f(r), f even, so that the sixteen
// 32-byte runs of a transposing read lie in different banks; the source side arranges it.
//
// What bounds it: the gathered rows (5.4 to 6.4 TB/s behind the L2, which hits 24 to 44 %; matrix pipes 8 to 25 %) and, for a few thousand pairs per offset, the partial sums (64 KB per chunk).
// A stage of 3x3x3 96 -> 96 over 300 k rows and 128 -> 128 over 170 k with its 2x2x2 layers, bf16, all four weight gradients:
// 667 -> 285 us (91, 107, 30 and 29, reductions 27); with the rows of dY shared in the XCDs' L2s (wgrad_first_chunk) 232 (74, 80, 25 and
// 28), where every row of dY came from behind the L2 for every offset.
// The column sums of dY (a bias's gradient) are workgroups of the same launch, behind the others, where the last of those leave CUs
// idle: these four and their column sums 206 + 39 us one after the other, 234 together; of a stage on 24,000 voxels of 32 and 64
// channels, where most of a launch is its start and end, 28 + 22 and 31.
#include <algorithm>
#include <mutex>

#include "wcn_common.h"
#include "wcn_conv_args.h"
#include "wcn_mma.h"
#include "wcn_rows.h"

namespace {

using namespace wcn_mma;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

__device__ __align__(256) uint32_t wgrad_zeros[256];  // source of what is not there; never written

constexpr int KP = 64;            // pairs of a step
constexpr int SEGMENT = 2048;     // pairs whose rows' numbers are in LDS at a time

struct WgradTileArgs {
  const void *X, *dY;
  const int32_t *in_maps, *out_maps;
  const int64_t* offsets;  // (K + 1), device
  float* partial;          // (chunks, c_in_pad, c_out_pad)
  int64_t num_in, num_out, identity_rows;
  int32_t K, c_in, c_out, c_in_pad, c_out_pad, identity, pairs_per_chunk, chunks, tiles_in, tiles_out;  // chunks: most on an XCD
  int32_t grid;  // workgroups of the tiles
};

__device__ __forceinline__ void to_lds(const char* g, uint32_t lds_off) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_off) : "memory");
}

// Which chunks of an offset (W of them, in the order of its pairs) an XCD works on: those of about an eighth of the pairs, the
// same eighth for all offsets, so that the rows of dY (which ascend inside every offset) that its workgroups read at a time are the
// same few thousand and come out of its L2 for all offsets but the first.  The rounding differs from offset to offset, so
// that no XCD gets the odd chunk of all of them.
__host__ __device__ inline int wgrad_first_chunk(int xcd, int chunks, int k) {
  const int64_t at = (int64_t)xcd * chunks - (5 * k & 7);
  return at <= 0 ? 0 : (int)((at + 7) / 8);
}

struct WgradChunk {
  int k, chunk, chunks, before;  // offset, number among its chunks, how many it has, and those of the offsets before it
};
// The q-th chunk of an XCD: a lane per offset, 64 offsets at a time.
__device__ __forceinline__ WgradChunk chunk_of(const int64_t* __restrict__ offsets, int K, int identity, int64_t identity_rows,
                                               int per, int xcd, int q) {
  int here = 0, all = 0;
  for (int k0 = 0; k0 < K; k0 += 64) {
    const int k = k0 + wcn_lane();
    int64_t n = k < K ? offsets[k + 1] - offsets[k] : 0;
    if (k == identity) n = identity_rows;
    const int W = (int)((n + per - 1) / per);
    const int j0 = wgrad_first_chunk(xcd, W, k), mine = wgrad_first_chunk(xcd + 1, W, k) - j0;
    const int incl = wcn_wave_inclusive_sum(mine), incl_all = wcn_wave_inclusive_sum(W);
    const int past = __popcll(__ballot(here + incl <= q));  // offsets whose chunks here end at or before this one
    if (past < 64) {
      WgradChunk c;
      c.k = k0 + past;
      c.chunk = __shfl(j0, past, 64) + q - (here + __shfl(incl - mine, past, 64));
      c.chunks = __shfl(W, past, 64);
      c.before = all + __shfl(incl_all - W, past, 64);
      return c;
    }
    here += __shfl(incl, 63, 64);
    all += __shfl(incl_all, 63, 64);
  }
  return {K, 0, 1, all};
}

template <int N>
struct Side {  // one operand: a tile of 32 N channels in rows of S
  static constexpr int T = 32 * N, S = N == 3 ? 128 : T;
  static constexpr int LPR = S / 8, RPI = 64 / LPR, LOADS = KP / RPI / 4;  // lanes of a row, rows of a load, loads of a wave
  static constexpr int BYTES = KP * S * 2;
  static_assert(LOADS >= 1, "every wave loads");
  static __device__ __forceinline__ int f(int r) {
    return S == 128 ? 2 * ((r & 3) | ((r >> 1) & 4)) : S == 64 ? 2 * (((r >> 1) & 1) | ((r >> 2) & 2)) : 2 * ((r >> 3) & 1);
  }
};

template <typename T, int NI, int NO>
__global__ void __launch_bounds__(256, 2) conv_wgrad_tiles(WgradTileArgs a, wcn_rows::ColumnPart columns) {
  typedef typename Mma<T>::V V;
  typedef Side<NI> I;
  typedef Side<NO> O;
  constexpr int STAGE = I::BYTES + O::BYTES;
  extern __shared__ __attribute__((aligned(16))) char wgrad_smem[];
  if ((int)blockIdx.x >= a.grid) {  // the column sums of dY: workgroups of their own behind the others
    wcn_rows::column_part<T, true>(columns, (int)blockIdx.x - a.grid, reinterpret_cast<float*>(wgrad_smem));
    return;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)wgrad_smem;
  int32_t* const s_in = reinterpret_cast<int32_t*>(wgrad_smem + 2 * STAGE);
  int32_t* const s_out = s_in + SEGMENT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tiles of a chunk follow one another on one XCD (blockIdx % 8): they gather the same rows
  const int tiles = a.tiles_in * a.tiles_out, b8 = (int)blockIdx.x >> 3;
  const int xcd = (int)blockIdx.x & 7, tile = b8 % tiles;
  const int ci0 = tile / a.tiles_out * I::T, co0 = tile % a.tiles_out * O::T;
  const WgradChunk at_chunk = chunk_of(a.offsets, a.K, a.identity, a.identity_rows, a.pairs_per_chunk, xcd, b8 / tiles);
  const int k = __builtin_amdgcn_readfirstlane(at_chunk.k);
  if (k >= a.K) return;
  const int W = __builtin_amdgcn_readfirstlane(at_chunk.chunks), j = __builtin_amdgcn_readfirstlane(at_chunk.chunk);
  const int chunk = __builtin_amdgcn_readfirstlane(at_chunk.before) + j;
  const bool ident = k == a.identity;
  const int64_t n_k = ident ? a.identity_rows : a.offsets[k + 1] - a.offsets[k];
  // The steps of an XCD's chunks of the offset are dealt to them in turn: all its workgroups move through their eighth together.
  const int j0 = wgrad_first_chunk(xcd, W, k), abreast = wgrad_first_chunk(xcd + 1, W, k) - j0;
  const uint32_t all_steps = (uint32_t)((n_k + KP - 1) / KP), each = all_steps / (uint32_t)W, odd = all_steps - each * (uint32_t)W;
  auto steps_before = [&](uint32_t c) { return (int64_t)each * c + odd * c / (uint32_t)W; };  // of chunk c; W < 65,536
  const int64_t step0 = steps_before((uint32_t)j0) + (j - j0), step1 = steps_before((uint32_t)(j0 + abreast));
  const int my_steps = step1 > step0 ? (int)((step1 - step0 + abreast - 1) / abreast) : 0;
  const int64_t pbase = a.offsets[k];
  const uint32_t in_bytes = (uint32_t)a.c_in * 2u, out_bytes = (uint32_t)a.c_out * 2u;
  const char* const zeros = (const char*)wgrad_zeros + lane * 16;

  // this lane's part of a load: row and piece
  uint32_t i_at[I::LOADS], o_at[O::LOADS];  // bytes from the row's start
#pragma unroll
  for (int j = 0; j < I::LOADS; ++j) {
    const int r = (wave * I::LOADS + j) * I::RPI + lane / I::LPR;
    i_at[j] = (uint32_t)ci0 * 2u + (uint32_t)((lane % I::LPR) ^ I::f(r)) * 16u;
    if (NI == 3 && ((lane % I::LPR) ^ I::f(r)) >= I::T / 8) i_at[j] = 0xffffffffu;  // beyond the tile: zeros
  }
#pragma unroll
  for (int j = 0; j < O::LOADS; ++j) {
    const int r = (wave * O::LOADS + j) * O::RPI + lane / O::LPR;
    o_at[j] = (uint32_t)co0 * 2u + (uint32_t)((lane % O::LPR) ^ O::f(r)) * 16u;
    if (NO == 3 && ((lane % O::LPR) ^ O::f(r)) >= O::T / 8) o_at[j] = 0xffffffffu;
  }
  auto fetch_side = [&](auto side, const int32_t* idx, const void* base, uint32_t bytes, const auto& at, uint32_t dst) {
    typedef decltype(side) Sd;
    int32_t row[Sd::LOADS];
#pragma unroll
    for (int j = 0; j < Sd::LOADS; ++j) row[j] = idx[(wave * Sd::LOADS + j) * Sd::RPI + lane / Sd::LPR];
#pragma unroll
    for (int j = 0; j < Sd::LOADS; ++j) {
      const char* p = (const char*)base + (size_t)(uint32_t)(row[j] < 0 ? 0 : row[j]) * bytes + (at[j] < bytes ? at[j] : 0u);
      asm("" : "+v"(p));
      to_lds(((row[j] >= 0) & (at[j] < bytes)) ? p : zeros, dst + (wave * Sd::LOADS + j) * 1024);
    }
  };
  auto fetch = [&](int s, int buf) {  // step s of the segment
    fetch_side(I{}, s_in + s * KP, a.X, in_bytes, i_at, lds0 + buf * STAGE);
    fetch_side(O{}, s_out + s * KP, a.dY, out_bytes, o_at, lds0 + buf * STAGE + I::BYTES);
  };

  // this wave's quarter, and the lane's place in the transposing reads: row 8 g + i / 4 (+ 4, + 32), channels 4 (i % 4)
  const int wi = (wave >> 1) * NI, wo = (wave & 1) * NO;  // 16-channel blocks
  const int i = lane & 15, g = lane >> 4, r0 = 8 * g + i / 4;
  const int i_base = r0 * (I::S * 2) + (i & 1) * 8, o_base = r0 * (O::S * 2) + (i & 1) * 8;
  int i_piece[NI], o_piece[NO];
#pragma unroll
  for (int b = 0; b < NI; ++b) i_piece[b] = i_base + (((wi + b) * 2 + (i & 3) / 2) ^ I::f(r0)) * 16;
#pragma unroll
  for (int b = 0; b < NO; ++b) o_piece[b] = o_base + (((wo + b) * 2 + (i & 3) / 2) ^ O::f(r0)) * 16;
  auto operand = [&](const char* at, int stride) -> V {
    typedef __attribute__((address_space(3))) s16x4* P;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)(__attribute__((address_space(3))) char*)at);
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)(__attribute__((address_space(3))) char*)(at + 4 * stride));
    const s16x8 both = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(V, both);
  };

  f32x4 acc[NI][NO];
#pragma unroll
  for (int x = 0; x < NI; ++x)
#pragma unroll
    for (int y = 0; y < NO; ++y) acc[x][y] = (f32x4){0.f, 0.f, 0.f, 0.f};

  constexpr int SEG_STEPS = SEGMENT / KP;
  for (int seg = 0; seg < my_steps; seg += SEG_STEPS) {
    const int steps = my_steps - seg < SEG_STEPS ? my_steps - seg : SEG_STEPS;
    // the rows' numbers; a pair that is not there, or names rows that are not, adds nothing
    for (int p = tid; p < (steps + 1) * KP && p < SEGMENT; p += 256) {
      int32_t rin = -1, rout = -1;
      const int64_t pair = (step0 + (int64_t)(seg + p / KP) * abreast) * KP + p % KP;
      if (p < steps * KP && pair < n_k) {
        rin = ident ? (int32_t)pair : a.in_maps[pbase + pair];
        rout = ident ? (int32_t)pair : a.out_maps[pbase + pair];
      }
      const bool there = (uint32_t)rin < (uint64_t)a.num_in && (uint32_t)rout < (uint64_t)a.num_out;
      s_in[p] = there ? rin : -1;
      s_out[p] = there ? rout : -1;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    fetch(0, 0);
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int s = 0; s < steps; ++s) {
      const int buf = s & 1;
      if (s + 1 < steps) fetch(s + 1, buf ^ 1);
      const char* const A = wgrad_smem + buf * STAGE;
      const char* const B = A + I::BYTES;
#pragma unroll
      for (int ks = 0; ks < KP / 32; ++ks) {
        V x[NI], y[NO];
#pragma unroll
        for (int b = 0; b < NI; ++b) x[b] = operand(A + i_piece[b] + ks * 32 * I::S * 2, I::S * 2);
#pragma unroll
        for (int b = 0; b < NO; ++b) y[b] = operand(B + o_piece[b] + ks * 32 * O::S * 2, O::S * 2);
#pragma unroll
        for (int xb = 0; xb < NI; ++xb)
#pragma unroll
          for (int yb = 0; yb < NO; ++yb) acc[xb][yb] = Mma<T>::mma(x[xb], y[yb], acc[xb][yb]);
      }
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }

  // a lane holds column i = channel of dY, rows 4 g .. + 3 = channels of X
  float* const out = a.partial + (int64_t)chunk * a.c_in_pad * a.c_out_pad;
#pragma unroll
  for (int xb = 0; xb < NI; ++xb)
#pragma unroll
    for (int yb = 0; yb < NO; ++yb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        out[(int64_t)(ci0 + (wi + xb) * 16 + 4 * g + r) * a.c_out_pad + co0 + (wo + yb) * 16 + i] = acc[xb][yb][r];
}

// dW[k] = the offset's chunks added up, rounded once: a workgroup owns 256 consecutive values of the padded plane, its
// waves the chunks c = j, j + 4, ..., eight loads in flight, combined as (0 + 1) + (2 + 3).
// Workgroups behind those (`columns.parts` > 0) finish the bias's gradient, which would be a launch of its own (4.6 us over 96
// channels).
template <typename WT>
__global__ void __launch_bounds__(256) wgrad_tiles_reduce(WgradTileArgs a, WT* __restrict__ dW, int planes, WcnColumnSums columns) {
  __shared__ f32x4 part[4][64];
  if ((int)blockIdx.x >= planes) {
    const int c0 = ((int)blockIdx.x - planes) * 16;
    if (columns.out_dtype == WCN_DTYPE_F32) wcn_column_sums_finish(columns, c0, (float*)columns.out);
    else if (columns.out_dtype == WCN_DTYPE_F16) wcn_column_sums_finish(columns, c0, (_Float16*)columns.out);
    else wcn_column_sums_finish(columns, c0, (__bf16*)columns.out);
    return;
  }
  const int plane = a.c_in_pad * a.c_out_pad, slices = plane / 256;
  const int k = blockIdx.x / slices, slice = blockIdx.x % slices;
  const int j = threadIdx.x >> 6, e = threadIdx.x & 63;
  const int elem = slice * 256 + e * 4;
  int c0 = 0;  // chunks of the offsets before k, and of k
  for (int k0 = 0; k0 < k; k0 += 64) {
    const int kk = k0 + e;
    int64_t n = kk < k ? a.offsets[kk + 1] - a.offsets[kk] : 0;
    if (kk < k && kk == a.identity) n = a.identity_rows;
    c0 += __shfl(wcn_wave_inclusive_sum((int)((n + a.pairs_per_chunk - 1) / a.pairs_per_chunk)), 63, 64);
  }
  const int64_t n_k = k == a.identity ? a.identity_rows : a.offsets[k + 1] - a.offsets[k];
  const int chunks = (int)((n_k + a.pairs_per_chunk - 1) / a.pairs_per_chunk);
  const float* const src = a.partial + (int64_t)c0 * plane + elem;
  f32x4 sum = (f32x4){0.f, 0.f, 0.f, 0.f};
  constexpr int U = 8;
  for (int c = j; c < chunks; c += 4 * U) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const f32x4*>(src + (int64_t)(c + 4 * u < chunks ? c + 4 * u : c) * plane);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c + 4 * u < chunks) sum += v[u];
  }
  part[j][e] = sum;
  __syncthreads();
  if (j != 0) return;
  const f32x4 total = (part[0][e] + part[1][e]) + (part[2][e] + part[3][e]);
  const int ci = elem / a.c_out_pad, co = elem % a.c_out_pad;
  if (ci >= a.c_in) return;
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (co + r < a.c_out) dW[((int64_t)k * a.c_in + ci) * a.c_out + co + r] = from_float<WT>(total[r]);
}

inline int blocks_of(int c) { return c <= 32 ? 1 : c <= 64 ? 2 : c <= 96 ? 3 : 4; }  // 32-channel blocks of a tile
inline int padded(int c) { return (c + 32 * blocks_of(c) - 1) / (32 * blocks_of(c)) * (32 * blocks_of(c)); }

// Workgroups that the chip holds at once: two per CU with tiles of more than 64 channels on both sides, else three.
inline int64_t wgrad_slots(int c_in, int c_out) { return blocks_of(c_in) > 2 && blocks_of(c_out) > 2 ? 512 : 768; }
// Pairs per chunk: as many workgroups as that, so that none is left for a second round; a multiple of a step and not
// fewer than 256.
inline int64_t wgrad_pairs_per_chunk(int64_t pairs, int K, int c_in, int c_out) {
  const int64_t tiles = (int64_t)(padded(c_in) / (32 * blocks_of(c_in))) * (padded(c_out) / (32 * blocks_of(c_out)));
  const int64_t slots = wgrad_slots(c_in, c_out) / tiles;
  const int64_t want = std::max<int64_t>(64, std::max(slots / 2, slots - K / 2));  // half a chunk is lost per offset
  const int64_t p = std::max<int64_t>(256, (pairs + want - 1) / want);
  return std::min<int64_t>((p + KP - 1) / KP * KP, 1 << 30);
}

struct WgradChunking {
  int64_t per, most;  // pairs per chunk; chunks of the XCD that has most of them (-1: too many to number)
};

// Where some XCD has more chunks than it holds at once, chunks get longer until none has, if a round of those takes less time
// than the rounds that it replaces take with the chunks' mean length (an offset's last chunk is short).  Wide rows leave few workgroups
// for a chunk's place: there a chunk per offset may be too many already.  us, 3x3x3 on rooms, bf16, first length / longer:
//     256 -> 256  24,000 rows   66 /  52 (1.06 times as long)    3,000 rows   34 /  31 (1.2)
//     256 -> 512  24,000       118 / 128 (1.95; two rounds of mean length are 1.7)     100,000   359 / 423 (1.98)
//     512 -> 512  24,000       194 / 236 (none has fitted at 2.2)                      300,000   1,980 / 2,490
//     384 -> 384  24,000       130 / 137
// (1024 -> 1024 over 20,000 rows, whose partial sums are 270 MB, 690 / 610: a third less of them.)
WgradChunking wgrad_chunking(const int64_t* host_offsets, int K, int identity, int64_t identity_rows, int c_in, int c_out) {
  int64_t pairs = 0, chunks = 0;  // of all offsets
  auto most_of = [&](int64_t per) -> int64_t {
    int64_t here[8] = {}, most = 0;
    pairs = chunks = 0;
    for (int k = 0; k < K; ++k) {
      const int64_t n = k == identity ? identity_rows : host_offsets[k + 1] - host_offsets[k];
      const int64_t W = (n + per - 1) / per;
      if (W >= 65536) return -1;  // see conv_wgrad_tiles
      pairs += n;
      chunks += W;
      for (int x = 0; x < 8; ++x) here[x] += wgrad_first_chunk(x + 1, (int)W, k) - wgrad_first_chunk(x, (int)W, k);
    }
    for (int x = 0; x < 8; ++x) most = std::max(most, here[x]);
    return most > INT32_MAX / 8 ? -1 : most;
  };
  const int64_t tiles = (int64_t)(padded(c_in) / (32 * blocks_of(c_in))) * (padded(c_out) / (32 * blocks_of(c_out)));
  const int64_t room = wgrad_slots(c_in, c_out) / 8 / tiles;
  WgradChunking first;
  first.per = wgrad_pairs_per_chunk(host_offsets[K] + identity_rows, K, c_in, c_out);
  first.most = most_of(first.per);
  if (first.most <= room || room < 1) return first;
  const int64_t limit = (first.most + room - 1) / room * pairs / chunks;
  if (most_of(1 << 30) > room) return first;
  int64_t per = first.per;
  for (int turn = 0; turn < 16; ++turn) {
    per = std::min<int64_t>((per + per / 24) / KP * KP + KP, 1 << 30);
    if (per >= limit) break;
    const int64_t most = most_of(per);
    if (most <= room) return {per, most};
  }
  return first;
}

template <typename T, int NI, int NO>
int launch_wgrad_tiles(WgradTileArgs a, const wcn_rows::ColumnPart& columns, int parts, hipStream_t s) {
  constexpr int lds = 2 * (Side<NI>::BYTES + Side<NO>::BYTES) + 2 * SEGMENT * 4;
  static_assert(lds >= 256 * 9 * 4, "room for the column sums");
  const void* fn = (const void*)conv_wgrad_tiles<T, NI, NO>;
  {  // more than 64 KiB of dynamic LDS has to be allowed once per device and kernel
    static std::mutex mu;
    static bool allowed[64] = {};
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return WCN_ERR_LAUNCH;
    std::lock_guard<std::mutex> hold(mu);
    if (!allowed[device]) {
      if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return WCN_ERR_LAUNCH;
      allowed[device] = true;
    }
  }
  const int64_t grid = (int64_t)a.chunks * 8 * a.tiles_in * a.tiles_out;
  if (grid + parts > INT32_MAX) return WCN_ERR_INVALID_ARGUMENT;
  a.grid = (int32_t)grid;
  if (grid + parts > 0) hipLaunchKernelGGL((conv_wgrad_tiles<T, NI, NO>), dim3((unsigned)(grid + parts)), dim3(256), lds, s, a, columns);
  return WCN_OK;
}

template <typename T, int NI>
int launch_out(const WgradTileArgs& a, const wcn_rows::ColumnPart& c, int parts, hipStream_t s) {
  switch (blocks_of(a.c_out)) {
    case 1: return launch_wgrad_tiles<T, NI, 1>(a, c, parts, s);
    case 2: return launch_wgrad_tiles<T, NI, 2>(a, c, parts, s);
    case 3: return launch_wgrad_tiles<T, NI, 3>(a, c, parts, s);
    default: return launch_wgrad_tiles<T, NI, 4>(a, c, parts, s);
  }
}
template <typename T>
int launch_in(const WgradTileArgs& a, const wcn_rows::ColumnPart& c, int parts, hipStream_t s) {
  switch (blocks_of(a.c_in)) {
    case 1: return launch_out<T, 1>(a, c, parts, s);
    case 2: return launch_out<T, 2>(a, c, parts, s);
    case 3: return launch_out<T, 3>(a, c, parts, s);
    default: return launch_out<T, 4>(a, c, parts, s);
  }
}

}  // namespace

bool wcn_wgrad_tiles_takes(int dtype, int c_in, int c_out, const void* features, const void* grad_out) {
  return dtype != WCN_DTYPE_F32 && c_in % 8 == 0 && c_out % 8 == 0 && (uintptr_t)features % 16 == 0 && (uintptr_t)grad_out % 16 == 0;
}

extern "C" int64_t wcn_conv_wgrad_chunk_pairs(const int64_t* host_offsets, int32_t num_offsets, int32_t identity_offset,
                                              int64_t identity_rows, int32_t c_in, int32_t c_out) {
  if (!host_offsets || num_offsets < 1 || num_offsets > WCN_MAX_OFFSETS || c_in < 8 || c_out < 8 || c_in % 8 || c_out % 8 ||
      identity_offset >= num_offsets || identity_rows < 0 || host_offsets[0] != 0 || host_offsets[num_offsets] > INT32_MAX)
    return 0;
  for (int k = 0; k < num_offsets; ++k)
    if (host_offsets[k + 1] < host_offsets[k]) return 0;
  return wgrad_chunking(host_offsets, num_offsets, identity_offset, identity_offset >= 0 ? identity_rows : 0, c_in, c_out).per;
}

size_t wcn_wgrad_tiles_partial_bytes(int num_offsets, int c_in, int c_out, int64_t pairs) {
  const int64_t chunks = pairs / wgrad_pairs_per_chunk(pairs, num_offsets, c_in, c_out) + num_offsets;
  return wcn_align256(sizeof(float) * (size_t)chunks * padded(c_in) * padded(c_out));
}

int wcn_wgrad_tiles_launch(const void* features, int64_t num_in, int c_in, const void* grad_out, int64_t num_out, int c_out,
                           int dtype, const int32_t* in_maps, const int32_t* out_maps, const int64_t* host_offsets,
                           const int64_t* device_offsets, int num_offsets, int identity, void* grad_weight,
                           int weight_dtype, float* partial, const WcnColumnSums* columns, hipStream_t s) {
  WgradTileArgs a;
  a.X = features;
  a.dY = grad_out;
  a.in_maps = in_maps;
  a.out_maps = out_maps;
  a.offsets = device_offsets;
  a.partial = partial;
  a.num_in = num_in;
  a.num_out = num_out;
  a.identity_rows = identity >= 0 ? std::min(num_in, num_out) : 0;
  a.K = num_offsets;
  a.c_in = c_in;
  a.c_out = c_out;
  a.c_in_pad = padded(c_in);
  a.c_out_pad = padded(c_out);
  a.identity = identity;
  a.tiles_in = a.c_in_pad / (32 * blocks_of(c_in));
  a.tiles_out = a.c_out_pad / (32 * blocks_of(c_out));
  // The device computes the same numbers from the same inputs.
  const WgradChunking plan = wgrad_chunking(host_offsets, num_offsets, identity, a.identity_rows, c_in, c_out);
  if (plan.most < 0) return WCN_ERR_INVALID_ARGUMENT;
  a.chunks = (int)plan.most;
  a.pairs_per_chunk = (int)plan.per;
  a.grid = 0;
  const WcnColumnSums sums = columns ? *columns : WcnColumnSums{};
  const wcn_rows::ColumnPart part = wcn_rows::column_part_of(grad_out, num_out, dtype, sums);
  const int st = dtype == WCN_DTYPE_F16 ? launch_in<_Float16>(a, part, sums.parts, s) : launch_in<__bf16>(a, part, sums.parts, s);
  if (st != WCN_OK) return st;
  const int planes = num_offsets * (a.c_in_pad * a.c_out_pad / 256);
  const dim3 grid((unsigned)(planes + (sums.channels + 15) / 16)), block(256);
  if (weight_dtype == WCN_DTYPE_F32)
    hipLaunchKernelGGL(wgrad_tiles_reduce<float>, grid, block, 0, s, a, (float*)grad_weight, planes, sums);
  else if (dtype == WCN_DTYPE_F16)
    hipLaunchKernelGGL(wgrad_tiles_reduce<_Float16>, grid, block, 0, s, a, (_Float16*)grad_weight, planes, sums);
  else
    hipLaunchKernelGGL(wgrad_tiles_reduce<__bf16>, grid, block, 0, s, a, (__bf16*)grad_weight, planes, sums);
  WCN_LAUNCH_CHECK();
  return WCN_OK;
}
