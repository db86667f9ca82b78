// The MXFP8 rows GEMM for groups of few rows (a decode step, a short prompt): y[i] =
// a[i] b[g(i)]^T as grouped_mx.hip's, for calls whose time is reading the experts' kernels.
// That file's schedule (one workgroup a CU on a 256 x 256 tile, operands shared through
// LDS) has too few tiles there to fill the chip, and a tile of 5 rows costs it 128.
//
// Here a wave is a workgroup of its own and takes 32 rows by 64 columns (or 64 rows, where
// rows may crowd: rows_direct), its operands straight from global memory to registers, two K
// pairs (256 bytes of K; of 64 rows one) ahead: no LDS, no barrier, no other wave to wait for,
// and two waves a SIMD, so that one's epilogue runs beside another's loads. The tiled layout
// serves that as it serves LDS: a block's 64-byte K chunks are one run of 2 KiB. What bounds it is each CU's loads in flight, so the waves
// have to spread evenly over the CUs: in workgroups of four the unevenly loaded ones last
// (16 groups of K 6400, N 4096, 32 rows on Zipf loads 60 -> 55 us, 96 rows 110 -> 85). Half
// the columns a wave, four pairs ahead and non-temporal loads of B were all slower. 128
// groups of K 2048, N 1536: 5.5 TB/s.
//
// The sums are grouped_mx.hip's to the bit (v_mfma_scale_f32_32x32x64_f8f6f4 over the K
// steps in order, from 0), so that a call may go either way.

#include <type_traits>

#include "mx_direct.h"
#include "tiles.h"

namespace bux {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int CB = 2;  // a wave's blocks of 32 columns

// A 32-row block's operand registers of one MFMA (the lane's 16 bytes of each of the
// step's two 32-byte blocks).
__device__ __forceinline__ v8i operand(const uint4& lo, const uint4& hi) {
  v8i v;
  v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
  v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
  return v;
}

__device__ __forceinline__ uint4 load16(const uint8_t* base, uint32_t at) {
  return *reinterpret_cast<const uint4*>(base + at);
}

// One K pair (128 bytes: two MFMA steps and one scale word a row) of a wave's R blocks of A
// and its CB blocks of B.
template <int R>
struct Pair {
  uint4 a[R][4], b[CB][4];
  uint32_t sa[R], sb[CB];
};

// A wave's R blocks of 32 rows by CB of 32 columns: rows row0 on, those below `end` stored.
template <int R, typename T>
__device__ __forceinline__ void direct_tile(
    const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* bv, const uint8_t* bs,
    int32_t a_rows, int32_t n, int32_t pairs, int64_t row0, int64_t end, int32_t col0,
    const T* bias, T* y) {
  constexpr int D = R == 1 ? 2 : 1;  // K pairs in flight: what leaves room for two waves a SIMD
  const int lane = threadIdx.x, half = lane >> 5, r32 = lane & 31;
  const int64_t a_chunk = static_cast<int64_t>(a_rows) * 64, b_chunk = static_cast<int64_t>(n) * 64;
  // rows past an operand's are its last one's again, and not stored
  uint32_t ar[R], br[CB];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t row = row0 + 32 * i + r32;
    ar[i] = static_cast<uint32_t>(row < a_rows ? row : a_rows - 1);
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) br[j] = static_cast<uint32_t>(smaller(col0 + 32 * j + r32, n - 1));
  v16f acc[R][CB];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;

  Pair<R> in[D];
  auto load = [&](Pair<R>& s, int32_t p) {
    const uint8_t* a0 = a_values + 2 * p * a_chunk;
    const uint8_t* b0 = bv + 2 * p * b_chunk;
    const uint8_t* as0 = a_scales + static_cast<int64_t>(p) * a_rows * 4;
    const uint8_t* bs0 = bs + static_cast<int64_t>(p) * n * 4;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
      const uint32_t at = br[j] * 64 + 16 * half;
      s.b[j][0] = load16(b0, at);
      s.b[j][1] = load16(b0, at + 32);
      s.b[j][2] = load16(b0 + b_chunk, at);
      s.b[j][3] = load16(b0 + b_chunk, at + 32);
      s.sb[j] = *reinterpret_cast<const uint32_t*>(bs0 + br[j] * 4);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t at = ar[i] * 64 + 16 * half;
      s.a[i][0] = load16(a0, at);
      s.a[i][1] = load16(a0, at + 32);
      s.a[i][2] = load16(a0 + a_chunk, at);
      s.a[i][3] = load16(a0 + a_chunk, at + 32);
      s.sa[i] = *reinterpret_cast<const uint32_t*>(as0 + ar[i] * 4);
    }
  };
  // Lane half h's scale byte is byte h of a word in its first step and 2 + h in its
  // second: the word shifted by h bytes, the MFMA taking its byte 0, then 2.
  auto multiply = [&](const Pair<R>& s) {
    int wa[R], wb[CB];
#pragma unroll
    for (int i = 0; i < R; ++i) wa[i] = static_cast<int>(s.sa[i] >> (8 * half));
#pragma unroll
    for (int j = 0; j < CB; ++j) wb[j] = static_cast<int>(s.sb[j] >> (8 * half));
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            operand(s.b[j][0], s.b[j][1]), operand(s.a[i][0], s.a[i][1]), acc[i][j], 0, 0, 0, wb[j],
            0, wa[i]);
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < CB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            operand(s.b[j][2], s.b[j][3]), operand(s.a[i][2], s.a[i][3]), acc[i][j], 0, 0, 2, wb[j],
            2, wa[i]);
  };
#pragma unroll
  for (int i = 0; i < D; ++i)
    if (i < pairs) load(in[i], i);
  int32_t p = 0;
  for (; p + 2 * D <= pairs; p += D) {
#pragma unroll
    for (int i = 0; i < D; ++i) {
      multiply(in[i]);
      __builtin_amdgcn_sched_barrier(0);
      load(in[i], p + D + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last D to 2 D - 1 pairs (all of them where there are fewer)
#pragma unroll
  for (int i = 0; i < D; ++i) {
    if (p + i < pairs) multiply(in[i]);
    __builtin_amdgcn_sched_barrier(0);
    if (p + D + i < pairs) load(in[i], p + D + i);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < D; ++i)
    if (p + D + i < pairs) multiply(in[i]);

  // lane l holds row l % 32, run g the columns 8 g + 4 (l / 32) .. + 3 of each block
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int64_t row = row0 + 32 * i + r32;
    if (row >= end) continue;
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int32_t col = col0 + 32 * j + 8 * g + 4 * half;
        if (col >= n) continue;  // n is a multiple of 4
        T* at = y + row * n + col;
        const v16f& a = acc[i][j];
        float c[4] = {a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
        if (bias != nullptr) {  // the product rounded, then the sum
#pragma unroll
          for (int q = 0; q < 4; ++q) c[q] = Elem<T>::round(c[q]) + Elem<T>::value(bias[col + q]);
        }
        if constexpr (std::is_same<T, uint16_t>::value)
          *reinterpret_cast<uint2*>(at) = make_uint2(pack_bf16x2(c[0], c[1]), pack_bf16x2(c[2], c[3]));
        else
          *reinterpret_cast<float4*>(at) = make_float4(c[0], c[1], c[2], c[3]);
      }
  }
}

// A wave takes up to R blocks of a tile's rows, blockIdx.y of them on; those past most tiles'
// rows leave at once, and come last in the grid.
template <typename T, int R>
__global__ __launch_bounds__(64) void rows_direct_kernel(
    const uint8_t* __restrict__ a_values, const uint8_t* __restrict__ a_scales,
    const uint8_t* __restrict__ b_values, const uint8_t* __restrict__ b_scales, int32_t k,
    int32_t a_rows, int32_t n, int32_t groups, int32_t height, const int32_t* __restrict__ starts,
    const Tile* __restrict__ tiles, int32_t col_blocks, const T* __restrict__ bias,
    T* __restrict__ y) {
  if (!list_fits(starts, groups, a_rows, height)) return;
  const int32_t id = blockIdx.x / col_blocks;
  if (id >= starts[groups + 1]) return;
  const Tile t = tiles[id];
  const int64_t row0 = direct_row(t.lo, blockIdx.y * R), end = smaller(t.hi, height);
  if (row0 >= end) return;
  const int32_t col0 = (blockIdx.x % col_blocks) * 32 * CB;
  const int32_t pairs = t.group < groups ? k / 128 : 0;  // rows past the groups: zeros
  const int32_t group = t.group < groups ? t.group : 0;
  const uint8_t* const bv = b_values + static_cast<int64_t>(group) * n * k;
  const uint8_t* const bs = b_scales + static_cast<int64_t>(group) * n * (k / 32);
  const T* const added = bias != nullptr && pairs > 0 ? bias + static_cast<int64_t>(group) * n : nullptr;
  if (R > 1 && end - row0 > DIRECT_BLOCK)
    direct_tile<R>(a_values, a_scales, bv, bs, a_rows, n, pairs, row0, end, col0, added, y);
  else
    direct_tile<1>(a_values, a_scales, bv, bs, a_rows, n, pairs, row0, end, col0, added, y);
}

template <typename T, int R>
int launch_as(const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* b_values,
              const uint8_t* b_scales, const void* list, int64_t slots, int32_t groups, int64_t m,
              int64_t n, int64_t k, int64_t height, const void* bias, void* y, hipStream_t s) {
  const int64_t col_blocks = ceil_div(n, 32 * CB);
  if (slots * col_blocks >= (1LL << 31)) return fail(BUX_E_ARGUMENT, "bux_mx_grouped_rows: too many tiles");
  const int64_t rows = m > height ? m : height;  // no tile holds more
  const int64_t row_blocks = ceil_div(rows < BM ? rows : BM, R * DIRECT_BLOCK);
  hipLaunchKernelGGL((rows_direct_kernel<T, R>),
                     dim3(static_cast<unsigned>(slots * col_blocks), static_cast<unsigned>(row_blocks)),
                     dim3(64), 0, s, a_values, a_scales, b_values, b_scales, static_cast<int32_t>(k),
                     static_cast<int32_t>(m), static_cast<int32_t>(n), groups,
                     static_cast<int32_t>(height), starts_in(list), tiles_in(list, groups),
                     static_cast<int32_t>(col_blocks), static_cast<const T*>(bias), static_cast<T*>(y));
  return launched("rows_direct_kernel");
}

}  // namespace

// The line between the two kernels, by what the host knows, rows, groups and columns; how the
// rows fall on the groups is the device's. A group of more rows than a wave takes has its B
// read again for each wave's here, and for each 256 rows by grouped_mx.hip, so the line is set
// by loads of rows crowded into few groups: half of the rows with one group, all with one, or
// with a fifth of the groups, and groups of 33, 65 and 129 rows.
//  - The tiles of even full groups fill at most half of the chip, up to a block a group; or the
//    tiles that the rows could fill in blocks of 32, crowded or not, are at most 64: waves of a
//    block. No load measured slower.
//  - Past it, up to 512 of them and 16 rows a group (rows crowded into a quarter of the groups
//    still fit one wave of 64): waves of two blocks, which read B half as often; their second
//    pair of K in flight would cost them the second wave a SIMD. Even loads gain, and Zipf(1.2)
//    ones too, save where grouped_mx.hip's tiles fill the chip once exactly (5% slower; half of
//    the rows with one group 14%). Calls that crowding has made short lose: all rows with one
//    group or a fifth of them up to 1.7 near 16 rows a group, within a fifth up to 13.
//  - Further on crowded loads lose more (waves of a block: 128 groups of K 2944, N 5760, 2048
//    rows with one group 38 -> 132), and Zipf loads begin to (469 -> 491).
// us, grouped_mx.hip's and this (even; Zipf; with a fifth of the groups; all with one):
//   128 groups of K 2048, N 1536, 320 rows (60 tiles)  103  75;   61  54;   29  19;  27  15
//   16 of K 6400, N 4096, 128 rows (64)                 95  81;   89  87;   72  28;  71  26
//   256 of K 7168, N 4096, 128 rows (64)               721 628;  332 280;  340 276;  78  40
//   8 of K 7168, N 4096, 256 rows (few tiles)           84  44;   82  60;   80  30;  64  49
// in waves of two blocks, and before them in waves of one:
//   128 of K 2048, N 1536, 1600 rows (300)      99  77 ( 78);  110  89 ( 91);  30  23 (34);  27  31 (29)
//   128 of K 768, N 2048, 1600 rows (400)       55  44 ( 47);   64  49 ( 52);  16  14 (21);  14  16 (18)
//   16 of K 6400, N 4096, 256 rows (128)        98  79 ( 81);   92  89 (101);  73  41 (27);  58  40 (44)
//   128 of K 2944, N 5760, 512 rows (368)      462 384 (392);  380 328 (337); 114  95 (96);  33  54 (55)
//   256 of K 2048, N 1024, 4096 rows (512)     123 108 (111);  137 124 (129);  30  51 (68);  24  39 (39)
//   32 of K 2048, N 2048, 512 rows (128)        34  32 ( 33);   36  37 ( 38);  28  17 (14);  24  16 (17)
int rows_direct(int64_t m, int32_t groups, int64_t n) {
  const int64_t tiles = ceil_div(n, BN), full = groups * tiles;
  const int64_t crowded = ceil_div(m, DIRECT_BLOCK) * tiles;
  if (m <= 0) return 0;
  if (full <= 128) return m <= DIRECT_BLOCK * static_cast<int64_t>(groups) ? 1 : 0;
  if (m > 16 * static_cast<int64_t>(groups)) return 0;
  if (crowded <= 64) return 1;
  return crowded <= 512 ? 2 : 0;
}

int launch_rows_direct(const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* b_values,
                       const uint8_t* b_scales, const void* list, int64_t slots, int32_t groups,
                       int64_t m, int64_t n, int64_t k, int64_t height, int out_dtype,
                       const void* bias, void* y, hipStream_t s) {
  auto go = [&](auto launch) {
    return launch(a_values, a_scales, b_values, b_scales, list, slots, groups, m, n, k, height, bias,
                  y, s);
  };
  if (rows_direct(m, groups, n) == 1)
    return out_dtype == BUX_BF16 ? go(launch_as<uint16_t, 1>) : go(launch_as<float, 1>);
  return out_dtype == BUX_BF16 ? go(launch_as<uint16_t, 2>) : go(launch_as<float, 2>);
}

}  // namespace bux

// Which kernel a call takes, for tests alone (not in bux_amd.h: the line may move).
extern "C" int bux_rows_direct(int64_t m, int32_t groups, int64_t n) {
  return bux::rows_direct(m, groups, n);
}
