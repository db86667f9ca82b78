// Sorting an MoE's picks by expert, stably: order, its inverse, each expert's size
// and the groups' offsets (src/bux/architecture/experts/moe.py:776-797: a stable
// argsort of the flat picks with those outside [0, E) as E, bincount, argsort of the
// order; the offsets cumsum(sizes) - sizes of grouped_mxfp8.py:142).
//
// A counting sort over segments of 256 picks (one wave a segment):
//   1. count:   each wave counts its segment's picks per bin (E bins and one for the
//               picks outside) in LDS; counts[bin][segment] goes to the workspace.
//   2. rows:    a workgroup a bin scans its row of counts exclusively, in place, and
//               leaves the bin's total.
//   3. bases:   one workgroup scans the bins' totals: where each bin starts in `order`
//               (the offsets; the totals are the sizes).
//   4. scatter: each wave walks its segment 64 picks at a time, in order, from its
//               bins' starts (base + row prefix). A pick's rank among the same bin's
//               picks of those 64 comes from ballots over its bin's bits (the lanes that
//               agree on every bit), and the lowest lane of each bin moves the bin's
//               running position on by the count: a stable order.
// All integer work: bit-exact by construction.
//
// Up to SMALL_PICKS picks the four are one kernel of one workgroup (small_kernel): the
// counts of 16 waves' segments stay in LDS.
//
// The layer's sort (bux_moe_permute_layer) gives what the layer makes of it too: each
// sorted pick's weight, from the pick as it is scattered, and the MXFP8 GEMMs' tile list
// (prologue_kernel's, tiles.h), from the offsets as they are scanned. That spares the
// layer two launches that wait for the sort (a gather and the list's prologue, 10 us at
// config 3's 131072 picks).

#include "common.h"
#include "tiles.h"

namespace bux {
namespace {

constexpr int SEGMENT = 256;  // picks a wave takes
constexpr int WAVES = 4;      // waves a workgroup
constexpr int MAX_BINS = 8192;  // experts + 1 (the LDS of count and scatter limits them further)

__device__ __forceinline__ int bin_of(int32_t expert, int32_t num_experts) {
  return (expert >= 0 && expert < num_experts) ? expert : num_experts;
}

__global__ __launch_bounds__(64 * WAVES) void count_kernel(const int32_t* __restrict__ idx,
                                                           int64_t n, int32_t num_experts,
                                                           int64_t segments,
                                                           int32_t* __restrict__ counts) {
  extern __shared__ int32_t lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bins = num_experts + 1;
  int32_t* mine = lds + wave * bins;
  for (int b = lane; b < bins; b += 64) mine[b] = 0;
  __syncthreads();
  const int64_t seg = static_cast<int64_t>(blockIdx.x) * WAVES + wave;
  if (seg < segments) {
    for (int i = lane; i < SEGMENT; i += 64) {
      const int64_t p = seg * SEGMENT + i;
      if (p < n) atomicAdd(&mine[bin_of(idx[p], num_experts)], 1);
    }
  }
  __syncthreads();
  if (seg < segments) {
    for (int b = lane; b < bins; b += 64) counts[static_cast<int64_t>(b) * segments + seg] = mine[b];
  }
}

constexpr int SCAN_THREADS = 256;

// Exclusive scan of one value a thread over the workgroup (NT lanes), by wave prefix sums
// and one pass over the waves' totals; returns the workgroup's total. `wave_sums` NT / 64
// ints of LDS, free again when it returns.
template <int NT>
__device__ __forceinline__ int32_t block_exclusive(int32_t v, int32_t& prefix, int32_t* wave_sums) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) wave_sums[wave] = x;
  __syncthreads();
  int32_t before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const int32_t t = wave_sums[w];
    if (w < wave) before += t;
    total += t;
  }
  __syncthreads();
  prefix = before + x - v;
  return total;
}

// What the layer's sort writes besides: each sorted pick's weight (words of `word` bytes;
// none where row_weights is NULL), and a tile list (none where header is NULL) of `slots`
// records for GEMMs of m rows into `height`.
struct LayerOuts {
  const void* weights;
  void* row_weights;
  int32_t word;
  int32_t* header;
  Tile* tiles;
  int64_t slots, m, height;
};

__device__ __forceinline__ uint32_t load_weight(const LayerOuts& o, int64_t p) {
  if (o.row_weights == nullptr) return 0;
  return o.word == 2 ? static_cast<const uint16_t*>(o.weights)[p]
                     : static_cast<const uint32_t*>(o.weights)[p];
}
__device__ __forceinline__ void store_weight(const LayerOuts& o, void* to, int32_t pos, uint32_t w) {
  if (o.row_weights == nullptr) return;
  if (o.word == 2) static_cast<uint16_t*>(to)[pos] = static_cast<uint16_t>(w);
  else static_cast<uint32_t*>(to)[pos] = w;
}

// The tile list prologue_kernel would make of these groups (align 1): the header, the
// starts, a group's rows in tiles of BM from its first, then the rows from the groups' end
// to `height`, then empty records. offs: the E + 1 offsets (LDS, or global memory this
// workgroup wrote before a barrier); the host checked that m or height holds every pick,
// so no start passes them. The whole workgroup calls it.
template <int NT>
__device__ __forceinline__ void write_list(const LayerOuts& o, const int32_t* offs,
                                           int32_t num_experts, int32_t* wave_sums) {
  if (threadIdx.x < LIST_HEADER / 4) {
    const int32_t i = threadIdx.x;
    o.header[i] = i == 0 ? LIST_MAGIC : i == 1 ? num_experts : i == 2 ? static_cast<int32_t>(o.m)
                : i == 3 ? static_cast<int32_t>(o.height) : 0;
  }
  int32_t* starts = o.header + LIST_HEADER / 4;
  const int32_t height = static_cast<int32_t>(o.height);
  int32_t used = 0;
  for (int32_t base = 0; base <= num_experts; base += NT) {
    const int32_t g = base + static_cast<int32_t>(threadIdx.x);
    const int32_t lo = g <= num_experts ? offs[g] : 0;
    const int32_t hi = g < num_experts ? offs[g + 1] : g == num_experts && height > lo ? height : lo;
    const int32_t count = static_cast<int32_t>(tile_count(lo, hi));
    int32_t before;
    const int32_t total = block_exclusive<NT>(count, before, wave_sums);
    if (g <= num_experts) starts[g] = lo;
    for (int32_t j = 0; j < count && used + before + j < o.slots; ++j)
      o.tiles[used + before + j] = tile_at(g, lo, hi, j);
    used += total;
  }
  for (int64_t i = used + threadIdx.x; i < o.slots; i += NT) o.tiles[i] = Tile{0, 0, 0};
  if (threadIdx.x == 0)
    starts[num_experts + 1] = used < o.slots ? used : static_cast<int32_t>(o.slots);
}

// Workgroup b scans counts[b][0 .. segments) exclusively in place; totals[b] = the sum.
__global__ __launch_bounds__(SCAN_THREADS) void rows_kernel(int32_t* __restrict__ counts,
                                                            int64_t segments,
                                                            int32_t* __restrict__ totals) {
  __shared__ int32_t wave_sums[SCAN_THREADS / 64];
  int32_t* row = counts + static_cast<int64_t>(blockIdx.x) * segments;
  int32_t carry = 0;
  for (int64_t base = 0; base < segments; base += SCAN_THREADS) {
    const int64_t i = base + threadIdx.x;
    const int32_t v = i < segments ? row[i] : 0;
    int32_t prefix;
    const int32_t total = block_exclusive<SCAN_THREADS>(v, prefix, wave_sums);
    if (i < segments) row[i] = carry + prefix;
    carry += total;
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// One workgroup: bases[b] = the totals of the bins before b; sizes and offsets of the
// experts (offsets[E] = the picks of experts: `filled`).
__global__ __launch_bounds__(SCAN_THREADS) void bases_kernel(const int32_t* __restrict__ totals,
                                                             int32_t bins,
                                                             int32_t* __restrict__ bases,
                                                             int32_t* __restrict__ sizes,
                                                             int32_t* offsets, LayerOuts outs) {
  __shared__ int32_t wave_sums[SCAN_THREADS / 64];
  int32_t carry = 0;
  for (int32_t base = 0; base < bins; base += SCAN_THREADS) {
    const int32_t b = base + threadIdx.x;
    const int32_t v = b < bins ? totals[b] : 0;
    int32_t prefix;
    const int32_t total = block_exclusive<SCAN_THREADS>(v, prefix, wave_sums);
    if (b < bins) {
      bases[b] = carry + prefix;
      if (b < bins - 1) {
        sizes[b] = v;
        offsets[b] = carry + prefix;
      } else {
        offsets[b] = carry + prefix;  // past the last expert: the sum of their sizes
      }
    }
    carry += total;
  }
  if (outs.header != nullptr) {
    __syncthreads();
    write_list<SCAN_THREADS>(outs, offsets, bins - 1, wave_sums);
  }
}

// A wave's next 64 picks, lane l's in bin b (`valid`: it has one): how many of them share
// the lane's bin, and how many of those come before it.
struct Peers {
  int32_t count, rank;
};
__device__ __forceinline__ Peers peers_of(int b, bool valid, int32_t bits) {
  const uint64_t below = (1ull << (threadIdx.x & 63)) - 1ull;
  uint64_t peers = __ballot(valid);
  for (int bit = 0; bit < bits; ++bit) {
    const bool set = (b >> bit) & 1;
    const uint64_t m = __ballot(set);
    peers &= set ? m : ~m;
  }
  return Peers{static_cast<int32_t>(__popcll(peers)), static_cast<int32_t>(__popcll(peers & below))};
}

// The picks' places, in order; `running` (LDS, the wave's own): where each bin's next pick
// goes.
__device__ __forceinline__ int32_t place(int b, bool valid, const Peers& peers, int32_t* running) {
  const int32_t start = valid ? running[b] : 0;
  __builtin_amdgcn_wave_barrier();
  if (valid && peers.rank == 0) running[b] = start + peers.count;
  __builtin_amdgcn_wave_barrier();
  return start + peers.rank;
}

__global__ __launch_bounds__(64 * WAVES) void scatter_kernel(
    const int32_t* __restrict__ idx, int64_t n, int32_t num_experts, int32_t bits,
    int64_t segments, const int32_t* __restrict__ base, const int32_t* __restrict__ bases,
    int32_t* __restrict__ order, int32_t* __restrict__ inverse, LayerOuts outs) {
  extern __shared__ int32_t lds[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bins = num_experts + 1;
  int32_t* running = lds + wave * bins;
  const int64_t seg = static_cast<int64_t>(blockIdx.x) * WAVES + wave;
  if (seg >= segments) return;  // whole waves leave; no workgroup barrier follows
  for (int b = lane; b < bins; b += 64)
    running[b] = bases[b] + base[static_cast<int64_t>(b) * segments + seg];
  __builtin_amdgcn_wave_barrier();
  // the segment's picks and weights are read at once, their latency paid once
  constexpr int TURNS = SEGMENT / 64;
  const int64_t p0 = seg * SEGMENT + lane;
  int bin[TURNS];
  uint32_t w[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 64 * i;
    bin[i] = p < n ? bin_of(idx[p], num_experts) : 0;
    w[i] = p < n ? load_weight(outs, p) : 0;
  }
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int64_t p = p0 + 64 * i;
    const int32_t pos = place(bin[i], p < n, peers_of(bin[i], p < n, bits), running);
    if (p >= n) continue;
    order[pos] = static_cast<int32_t>(p);
    inverse[p] = pos;
    store_weight(outs, outs.row_weights, pos, w[i]);
  }
}

// The whole sort by one workgroup: wave w takes the picks [w per, (w + 1) per). A wave's
// picks and weights are read at once (TURNS of 64), and the order and the sorted weights
// are put together in LDS and written in runs (scattered from one CU, a store of 64 lines
// holds its memory pipe 64 cycles). What bounds it is one CU's VALU: `peers_of` takes 16
// waves' 1024 picks in about 1 us. In a graph, with weights and list, against the four
// kernels and the two the layer ran after them (us): 64 picks 4.8 and 21, 1600 picks 5.9
// and 20. Alone 8192 picks take 9.4, 16000 would take 19; the four kernels take 12 to 13
// from 16000 picks to 131072.
constexpr int SMALL_THREADS = 1024;
constexpr int SMALL_WAVES = SMALL_THREADS / 64;
constexpr int64_t SMALL_PICKS = 8192;
constexpr int SMALL_BINS = 900;  // at most SMALL_THREADS: a thread a bin

// Its LDS: the waves' counts, the offsets, the order, the sorted weights (16-byte aligned).
__host__ __device__ constexpr size_t small_lds(int32_t n, int32_t bins, int32_t word) {
  const size_t ints = (static_cast<size_t>(SMALL_WAVES + 1) * bins + n + 3) / 4 * 4;
  return ints * sizeof(int32_t) + static_cast<size_t>(n) * word;
}
static_assert(small_lds(SMALL_PICKS, SMALL_BINS, 4) <= 152 * 1024, "small_kernel fits a CU's LDS");

template <int TURNS>
__global__ __launch_bounds__(SMALL_THREADS) void small_kernel(
    const int32_t* __restrict__ idx, int32_t n, int32_t num_experts, int32_t bits,
    int32_t* __restrict__ order, int32_t* __restrict__ inverse, int32_t* __restrict__ sizes,
    int32_t* __restrict__ offsets, LayerOuts outs) {
  extern __shared__ __align__(16) int32_t lds[];
  __shared__ int32_t wave_sums[SMALL_WAVES];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bins = num_experts + 1;
  int32_t* offs = lds + SMALL_WAVES * bins;  // bins ints
  int32_t* sorted = offs + bins;             // n ints
  uint8_t* sorted_weights = reinterpret_cast<uint8_t*>(lds) + small_lds(n, bins, 0);
  int32_t* mine = lds + wave * bins;
  const int32_t per = (n + SMALL_THREADS - 1) / SMALL_THREADS * 64;  // at most 64 TURNS
  const int32_t p0 = wave * per + lane, end = smaller(n, (wave + 1) * per);
  int bin[TURNS];
  uint32_t w[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int32_t p = p0 + 64 * i;
    bin[i] = p < end ? bin_of(idx[p], num_experts) : 0;
    w[i] = p < end ? load_weight(outs, p) : 0;
  }
  for (int b = lane; b < bins; b += 64) mine[b] = 0;
  __builtin_amdgcn_wave_barrier();
  // one lane adds a bin's picks of a turn: a lane a pick, 8192 picks all in one bin took 15.5
  // us (the additions to one address go one after another), now 9.4
  Peers peers[TURNS];
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    if (p0 - lane + 64 * i >= end) break;  // the whole wave
    const bool valid = p0 + 64 * i < end;
    peers[i] = peers_of(bin[i], valid, bits);
    if (valid && peers[i].rank == 0) atomicAdd(&mine[bin[i]], peers[i].count);
  }
  __syncthreads();
  const int b = threadIdx.x;
  int32_t total = 0;
  if (b < bins)
#pragma unroll
    for (int v = 0; v < SMALL_WAVES; ++v) total += lds[v * bins + b];
  int32_t start;
  block_exclusive<SMALL_THREADS>(total, start, wave_sums);
  if (b < bins) {
    offs[b] = start;
    offsets[b] = start;
    if (b < num_experts) sizes[b] = total;
#pragma unroll
    for (int v = 0; v < SMALL_WAVES; ++v) {  // counts to where the wave's picks of the bin start
      const int32_t c = lds[v * bins + b];
      lds[v * bins + b] = start;
      start += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TURNS; ++i) {
    const int32_t p = p0 + 64 * i;
    if (p - lane >= end) break;  // the whole wave
    const int32_t pos = place(bin[i], p < end, peers[i], mine);
    if (p >= end) continue;
    sorted[pos] = p;
    inverse[p] = pos;
    store_weight(outs, sorted_weights, pos, w[i]);
  }
  __syncthreads();
  for (int32_t i = threadIdx.x; i < n; i += SMALL_THREADS) {
    order[i] = sorted[i];
    if (outs.row_weights == nullptr) continue;
    store_weight(outs, outs.row_weights, i,
                 outs.word == 2 ? reinterpret_cast<const uint16_t*>(sorted_weights)[i]
                                : reinterpret_cast<const uint32_t*>(sorted_weights)[i]);
  }
  if (outs.header != nullptr) write_list<SMALL_THREADS>(outs, offs, num_experts, wave_sums);
}

}  // namespace
}  // namespace bux

extern "C" size_t bux_moe_permute_workspace_size(int64_t n_picks, int32_t num_experts) {
  // counts[bins][segments], then the bins' totals and bases
  const int64_t segments = (n_picks + bux::SEGMENT - 1) / bux::SEGMENT;
  return static_cast<size_t>(segments + 2) * static_cast<size_t>(num_experts + 1) * sizeof(int32_t);
}

namespace bux {
namespace {

int permute(const char* name, const int32_t* idx, int64_t n_picks, int32_t num_experts,
            int32_t* order, int32_t* inverse, int32_t* sizes, int32_t* offsets,
            const LayerOuts& outs, void* workspace, size_t workspace_bytes, void* stream) {
  BUX_CHECK(n_picks >= 0 && n_picks <= 2147483647LL, "%s: n_picks=%lld outside [0, 2^31)", name,
            (long long)n_picks);
  BUX_CHECK(num_experts >= 1 && num_experts < MAX_BINS, "%s: num_experts=%d outside [1, %d)", name,
            num_experts, MAX_BINS);
  BUX_CHECK(sizes && offsets, "%s: sizes and offsets are needed", name);
  BUX_CHECK(n_picks == 0 || (idx && order && inverse), "%s: idx, order and inverse are needed", name);
  const size_t need = bux_moe_permute_workspace_size(n_picks, num_experts);
  if (workspace_bytes < need || workspace == nullptr)
    return fail(BUX_E_WORKSPACE, "%s: workspace of %zu bytes, %zu needed", name, workspace_bytes,
                need);
  const int64_t segments = ceil_div(n_picks, SEGMENT);
  const int bins = num_experts + 1;
  int bits = 0;
  while ((1 << bits) < bins) ++bits;
  hipStream_t s = as_stream(stream);
  if (n_picks <= SMALL_PICKS && bins <= SMALL_BINS) {
    const size_t lds =
        small_lds(static_cast<int32_t>(n_picks), bins, outs.row_weights ? outs.word : 0);
    auto go = [&](auto kernel) {
      if (lds > 64 * 1024)
        if (int rc = allow_lds(kernel, lds, "small_kernel")) return rc;
      hipLaunchKernelGGL(kernel, dim3(1), dim3(SMALL_THREADS), lds, s, idx,
                         static_cast<int32_t>(n_picks), num_experts, bits, order, inverse, sizes,
                         offsets, outs);
      return launched("small_kernel");
    };
    return n_picks <= 4096 ? go(small_kernel<4>) : go(small_kernel<8>);
  }
  int32_t* counts = static_cast<int32_t*>(workspace);
  const size_t lds = static_cast<size_t>(WAVES) * bins * sizeof(int32_t);
  BUX_CHECK(lds <= 64 * 1024, "%s: %d experts exceed the LDS a workgroup takes", name, num_experts);
  const unsigned blocks = static_cast<unsigned>(ceil_div(segments, WAVES));
  if (segments > 0) {
    hipLaunchKernelGGL(count_kernel, dim3(blocks), dim3(64 * WAVES), lds, s, idx, n_picks,
                       num_experts, segments, counts);
    if (int rc = launched("count_kernel")) return rc;
  }
  int32_t* totals = counts + segments * bins;
  int32_t* bases = totals + bins;
  hipLaunchKernelGGL(rows_kernel, dim3(bins), dim3(SCAN_THREADS), 0, s, counts, segments, totals);
  if (int rc = launched("rows_kernel")) return rc;
  hipLaunchKernelGGL(bases_kernel, dim3(1), dim3(SCAN_THREADS), 0, s, totals, bins, bases, sizes,
                     offsets, outs);
  if (int rc = launched("bases_kernel")) return rc;
  if (segments > 0) {
    hipLaunchKernelGGL(scatter_kernel, dim3(blocks), dim3(64 * WAVES), lds, s, idx, n_picks,
                       num_experts, bits, segments, counts, bases, order, inverse, outs);
    if (int rc = launched("scatter_kernel")) return rc;
  }
  return BUX_OK;
}

}  // namespace
}  // namespace bux

extern "C" int bux_moe_permute(const int32_t* idx, int64_t n_picks, int32_t num_experts,
                               int32_t* order, int32_t* inverse, int32_t* sizes, int32_t* offsets,
                               void* workspace, size_t workspace_bytes, void* stream) {
  bux::clear_error();
  return bux::permute("bux_moe_permute", idx, n_picks, num_experts, order, inverse, sizes, offsets,
                      bux::LayerOuts{}, workspace, workspace_bytes, stream);
}

extern "C" int bux_moe_permute_layer(const int32_t* idx, int64_t n_picks, int32_t num_experts,
                                     const void* weights, int32_t weight_bytes, int32_t* order,
                                     int32_t* inverse, int32_t* sizes, int32_t* offsets,
                                     void* row_weights, void* list, size_t list_bytes, int64_t m,
                                     int64_t height, void* workspace, size_t workspace_bytes,
                                     void* stream) {
  using namespace bux;
  const char* const name = "bux_moe_permute_layer";
  clear_error();
  LayerOuts outs{};
  BUX_CHECK(weight_bytes == 2 || weight_bytes == 4, "%s: weight_bytes=%d is neither 2 nor 4", name,
            weight_bytes);
  BUX_CHECK(n_picks <= 0 || (weights && row_weights), "%s: weights and row_weights are needed", name);
  outs.weights = weights;
  outs.row_weights = row_weights;
  outs.word = weight_bytes;
  if (list != nullptr) {
    BUX_CHECK(num_experts >= 1 && num_experts <= MAX_GROUPS, "%s: a list of groups=%d outside [1, %d]",
              name, num_experts, MAX_GROUPS);
    BUX_CHECK(m >= 0 && height >= 0 && height < (1LL << 31) && m < (1LL << 31) &&
                  (m > height ? m : height) >= n_picks,
              "%s: bad shape m=%lld height=%lld for %lld picks", name, (long long)m,
              (long long)height, (long long)n_picks);
    const size_t need = bux_mx_grouped_rows_workspace_size(num_experts, m, height);
    if (list_bytes < need)
      return fail(BUX_E_WORKSPACE, "%s: list of %zu bytes, %zu needed", name, list_bytes, need);
    outs.header = header_in(list);
    outs.tiles = tiles_in(list, num_experts);
    outs.slots = row_slots(num_experts, m, height);
    outs.m = m;
    outs.height = height;
  }
  return permute(name, idx, n_picks, num_experts, order, inverse, sizes, offsets, outs, workspace,
                 workspace_bytes, stream);
}
