// The MXFP8 rows GEMM for groups of few rows (a decode step, a short prompt): y[i] =
// a[i] b[g(i)]^T as grouped_mx.hip's, for calls whose time is reading the experts' kernels.
// That file's schedule (one workgroup a CU on a 256 x 256 tile, operands shared through
// LDS) has too few tiles there to fill the chip, and a tile of 5 rows costs it 128.
//
// Here a wave is a workgroup of its own and takes 32 rows by 64 columns, its operands
// straight from global memory to registers, two K pairs (256 bytes of K) ahead: no LDS, no
// barrier, no other wave to wait for, and two waves a SIMD, so that one's epilogue runs
// beside another's loads. The tiled layout serves that as it serves LDS: a block's 64-byte
// K chunks are one run of 2 KiB. What bounds it is each CU's loads in flight, so the waves
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

constexpr int CB = 2;      // its blocks of 32 columns
constexpr int D = 2;       // K pairs in flight

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

// One K pair (128 bytes: two MFMA steps and one scale word a row) of a wave's block of A
// and its CB blocks of B.
struct Pair {
  uint4 a[4], b[CB][4];
  uint32_t sa, sb[CB];
};

// blockIdx.y: a tile's block of 32 rows; those past most tiles' rows leave at once, and come
// last in the grid.
template <typename T>
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
  const int64_t row0 = direct_row(t.lo, blockIdx.y), end = smaller(t.hi, height);
  if (row0 >= end) return;
  const int lane = threadIdx.x, half = lane >> 5, r32 = lane & 31;
  const int32_t col0 = (blockIdx.x % col_blocks) * 32 * CB;
  const int32_t pairs = t.group < groups ? k / 128 : 0;  // rows past the groups: zeros
  const int32_t group = t.group < groups ? t.group : 0;
  const uint8_t* const bv = b_values + static_cast<int64_t>(group) * n * k;
  const uint8_t* const bs = b_scales + static_cast<int64_t>(group) * n * (k / 32);
  const int64_t a_chunk = static_cast<int64_t>(a_rows) * 64, b_chunk = static_cast<int64_t>(n) * 64;
  // rows past an operand's are its last one's again, and not stored
  const uint32_t ar = static_cast<uint32_t>(row0 + r32 < a_rows ? row0 + r32 : a_rows - 1);
  uint32_t br[CB];
#pragma unroll
  for (int j = 0; j < CB; ++j) br[j] = static_cast<uint32_t>(smaller(col0 + 32 * j + r32, n - 1));
  v16f acc[CB];
#pragma unroll
  for (int j = 0; j < CB; ++j)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[j][q] = 0.0f;

  Pair in[D];
  auto load = [&](Pair& s, int32_t p) {
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
    const uint32_t at = ar * 64 + 16 * half;
    s.a[0] = load16(a0, at);
    s.a[1] = load16(a0, at + 32);
    s.a[2] = load16(a0 + a_chunk, at);
    s.a[3] = load16(a0 + a_chunk, at + 32);
    s.sa = *reinterpret_cast<const uint32_t*>(as0 + ar * 4);
  };
  // Lane half h's scale byte is byte h of a word in its first step and 2 + h in its
  // second: the word shifted by h bytes, the MFMA taking its byte 0, then 2.
  auto multiply = [&](const Pair& s) {
    const int wa = static_cast<int>(s.sa >> (8 * half));
    int wb[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) wb[j] = static_cast<int>(s.sb[j] >> (8 * half));
#pragma unroll
    for (int j = 0; j < CB; ++j)
      acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
          operand(s.b[j][0], s.b[j][1]), operand(s.a[0], s.a[1]), acc[j], 0, 0, 0, wb[j], 0, wa);
#pragma unroll
    for (int j = 0; j < CB; ++j)
      acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
          operand(s.b[j][2], s.b[j][3]), operand(s.a[2], s.a[3]), acc[j], 0, 0, 2, wb[j], 2, wa);
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
  const int64_t row = row0 + r32;
  if (row >= end) return;
#pragma unroll
  for (int j = 0; j < CB; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int32_t col = col0 + 32 * j + 8 * g + 4 * half;
      if (col >= n) continue;  // n is a multiple of 4
      T* at = y + row * n + col;
      float c[4] = {acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]};
      if (bias != nullptr && pairs > 0) {  // the product rounded, then the sum
        const T* b = bias + static_cast<int64_t>(group) * n + col;
#pragma unroll
        for (int q = 0; q < 4; ++q) c[q] = Elem<T>::round(c[q]) + Elem<T>::value(b[q]);
      }
      if constexpr (std::is_same<T, uint16_t>::value)
        *reinterpret_cast<uint2*>(at) = make_uint2(pack_bf16x2(c[0], c[1]), pack_bf16x2(c[2], c[3]));
      else
        *reinterpret_cast<float4*>(at) = make_float4(c[0], c[1], c[2], c[3]);
    }
}

template <typename T>
int launch_as(const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* b_values,
              const uint8_t* b_scales, const void* list, int64_t slots, int32_t groups, int64_t m,
              int64_t n, int64_t k, int64_t height, const void* bias, void* y, hipStream_t s) {
  const int64_t col_blocks = ceil_div(n, 32 * CB);
  if (slots * col_blocks >= (1LL << 31)) return fail(BUX_E_ARGUMENT, "bux_mx_grouped_rows: too many tiles");
  const int64_t rows = m > height ? m : height;  // no tile holds more
  const int64_t row_blocks = ceil_div(rows < BM ? rows : BM, DIRECT_BLOCK);
  hipLaunchKernelGGL(rows_direct_kernel<T>,
                     dim3(static_cast<unsigned>(slots * col_blocks), static_cast<unsigned>(row_blocks)),
                     dim3(64), 0, s, a_values, a_scales, b_values, b_scales, static_cast<int32_t>(k),
                     static_cast<int32_t>(m), static_cast<int32_t>(n), groups,
                     static_cast<int32_t>(height), starts_in(list), tiles_in(list, groups),
                     static_cast<int32_t>(col_blocks), static_cast<const T*>(bias), static_cast<T*>(y));
  return launched("rows_direct_kernel");
}

}  // namespace

// The line between the two kernels, by what the host knows, rows, groups and columns; how the
// rows fall on the groups is the device's. A group of more than a block of rows has its B read
// once a block here and once a tile of 256 rows by grouped_mx.hip, so rows crowded into few
// groups are what the line must bear: below it no load measured slower (even, Zipf(1.2), half
// of the rows with one group, all with one, with a fifth of the groups, groups of 33 and of
// 65 rows). Either the tiles of even full groups would fill at most half of the chip, up to a
// block of rows a group; or the tiles that the rows could fill in blocks of 32, crowded or
// not, are a quarter of its CUs. us, grouped_mx.hip's and this (even; all rows with one group;
// groups of 33 rows, each a second block of one row):
//   128 groups of K 2048, N 1536, 320 rows (60 tiles)     103 and  74;  27 and 15;  28 and 13
//   128 of K 768, N 2048, 256 rows (64)                    56 and  43;  14 and 12;  14 and 12
//   16 of K 6400, N 4096, 128 rows (64; Zipf 88 and 86)   100 and  82;  71 and 26;  71 and 27
//   256 of K 7168, N 4096, 128 rows (64)                  736 and 626;  78 and 40;  78 and 62
//   8 of K 7168, N 4096, 256 rows (few tiles)              83 and  44;  63 and 46;  83 and 62
// and past it even loads gain as before, crowded ones lose:
//   128 of K 2048, N 1536, 1024 rows (192)                100 and  77;  24 and 21;  29 and 35
//   16 of K 6400, N 4096, 256 rows (128; Zipf 91 and 100)  99 and  81;  58 and 43;  74 and 56
//   128 of K 2944, N 5760, 256 rows (184)                 464 and 386;  31 and 40;  37 and 51
//   256 of K 2048, N 7168, 192 rows (168)                 585 and 494;  25 and 41;  28 and 56
bool rows_direct(int64_t m, int32_t groups, int64_t n) {
  const int64_t tiles = ceil_div(n, BN);
  if (m <= 0) return false;
  if (groups * tiles <= 128) return m <= DIRECT_BLOCK * static_cast<int64_t>(groups);
  return m <= 16 * static_cast<int64_t>(groups) && ceil_div(m, DIRECT_BLOCK) * tiles <= 64;
}

int launch_rows_direct(const uint8_t* a_values, const uint8_t* a_scales, const uint8_t* b_values,
                       const uint8_t* b_scales, const void* list, int64_t slots, int32_t groups,
                       int64_t m, int64_t n, int64_t k, int64_t height, int out_dtype,
                       const void* bias, void* y, hipStream_t s) {
  return out_dtype == BUX_BF16
             ? launch_as<uint16_t>(a_values, a_scales, b_values, b_scales, list, slots, groups, m, n,
                                   k, height, bias, y, s)
             : launch_as<float>(a_values, a_scales, b_values, b_scales, list, slots, groups, m, n, k,
                                height, bias, y, s);
}

}  // namespace bux

// Which kernel a call takes, for tests alone (not in bux_amd.h: the line may move).
extern "C" int bux_rows_direct(int64_t m, int32_t groups, int64_t n) {
  return bux::rows_direct(m, groups, n);
}
