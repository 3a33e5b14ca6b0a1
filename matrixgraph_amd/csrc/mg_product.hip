// Numeric pass of the handle-level tile products C = A * B (B supplied transposed).
//
// The product of two tiles is the OR over their common inner indices j of (column j of the A tile)
// x (row j of the B tile), and column words of both operands (row j of B = column j of Bt) are all
// it needs: 8 bytes a side for a j, dense tile or not. Most pairs of tiles that meet share few j:
// on C = A*A of R-MAT 14 (25.8 K tiles, 16 edges a vertex) the 3.7 M structural pairs have 6.0 M
// common j in all, and 47 % of them none.
//
// Two kernels; by_tiles chooses. tile_product_kernel: a wave per C tile, where few pairs meet in each and
// on grids wider than kBitmapStrips. product_kernel, the rest of this comment:
//
// A workgroup takes a tile row x of A and a window of up to kWindow strips of C, whose tiles it
// keeps in LDS. The pairs come straight from the lists, A(x, t) against the B(t, y) of the window,
// nothing is searched, and each of three stages queues in LDS for the next so that every stage runs
// on full waves:
//   1. lane = A tile: the window's strips y of B row t (a few bits of its bitmap word);
//   2. lane = pair: the two heads (16 bytes each), common j = the ANDed masks;
//   3. lane = (pair, j): one column word of each side, then the fewer ORs of two: the column word of
//      B into each row the A word has, or the A word into each column of the transposed C tile.
// Stages 2 and 3 fetch a batch before they work on the one before it. Pairs with more than
// kFewCommon common j go through stage 3 at once, lane = j, their column words being contiguous. The
// two halves of a C tile, by rows and by columns, meet at the end (wave_transpose).
//
// Measured (both operands prepared), against one wave per C tile that searches the shorter tile list
// in the longer one and multiplies payloads of 16 bytes: A*A of R-MAT 14 119 us, before 518; of
// R-MAT 16 with 16 planted communities (191 K tiles, 70 M pairs) 1.28 ms, before 4.63; a frontier of
// 1000 rows x R-MAT 18 (7.3 K tiles, 6.8 M pairs) 140 us, before 482. Bound by the chains of ballots
// and LDS writes between the stages and by the vector ALUs (58 % of the issue slots on the second): filling
// the queue of stage 3 is half of the time, the ORs themselves nothing.
#include <algorithm>
#include <cmath>
#include <string>

#include "mg_device.hpp"
#include "mg_product.hpp"

namespace mgamd {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;

// Lanes below this one whose bit of `mask` is set.
__device__ inline uint32_t lanes_under(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}
__device__ inline uint32_t lane_u32(uint32_t v, int src) {
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), src));
}
// Sum over the wave (DPP: within rows of 16, then across them; lane 63 has it).
__device__ inline uint32_t wave_sum32(uint32_t v) {
  int x = static_cast<int>(v);
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, true);   // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, true);   // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, true);   // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, true);   // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
  return lane_u32(static_cast<uint32_t>(x), kWave - 1);
}
__device__ inline int lowest(uint64_t m) { return __ffsll(static_cast<unsigned long long>(m)) - 1; }

// --- heads and column words ------------------------------------------------------------

// Where a tile's head goes: its own place (bm null) or the position of B(t, y).
struct PositionMap {
  const uint32_t* row;  // per tile of Bt: y and t
  const uint32_t* col;
  const BitmapWord* bm;
  uint32_t wpr;         // bitmap words per row
  __device__ uint32_t operator()(uint32_t i) const {
    if (!bm) return i;
    const uint32_t y = row[i], t = col[i];
    const BitmapWord w = bm[static_cast<uint64_t>(t) * wpr + (y >> 6)];
    return w.at + static_cast<uint32_t>(__popcll(w.bits & ((1ull << (y & 63)) - 1)));
  }
};
struct HeadJob {
  const uint64_t* data;
  uint32_t n;
  PositionMap where;
  TileHead* head;          // by where(i)
  TileHead* head_by_tile;  // may be null
  uint32_t* tile;          // inverse of where (may be null)
  uint8_t* used;           // columns in use, by tile (may be null)
  uint32_t words0;         // first word (tile_heads_kernel without `next`)
};

// Heads and column words of the tiles of two operands (blockIdx.y). One pass over the tiles is
// what bounds it: a wave has kHeadLoads of them in flight and transposes each (wave_transpose); a
// workgroup takes the place of all its non-zero words in `words` with one atomic (12 ns each on one
// address: one per wave and round would take longer than the reads). No room left, or none
// asked for (cap 0): kNoWords. next null: tile i has the 64 words from job.words0 + 64 i on.
constexpr int kHeadLoads = 8;
constexpr int kHeadWaves = 16;
template <int kLoads, int kWaves>
__global__ void __launch_bounds__(kWaves* kWave) tile_heads_kernel(HeadJob job0, HeadJob job1, bool want_bits,
                                                                       uint64_t* __restrict__ words, uint64_t cap,
                                                                       unsigned long long* __restrict__ next) {
  constexpr uint32_t kTiles = kWaves * kLoads;  // of a workgroup's round
  __shared__ uint32_t s_count[kWaves];
  __shared__ unsigned long long s_base;
  const HeadJob& job = blockIdx.y ? job1 : job0;
  const uint32_t lane = lane_id(), wave = read_first_lane(threadIdx.x / kWave), n = job.n;
  for (uint64_t r0 = static_cast<uint64_t>(blockIdx.x) * kTiles; r0 < n;
       r0 += static_cast<uint64_t>(gridDim.x) * kTiles) {
    const uint64_t i0 = r0 + wave * kLoads;
    uint64_t word[kLoads];
#pragma unroll
    for (int q = 0; q < kLoads; ++q)
      word[q] = i0 + q < n ? __builtin_nontemporal_load(job.data + (i0 + q) * kTile + lane) : 0ull;
    const bool writes = lane < kLoads && i0 + lane < n;  // lane q: tile i0 + q
    const uint32_t at = writes ? job.where(static_cast<uint32_t>(i0) + lane) : 0u;
    uint64_t l_mask = 0;
    uint32_t l_at = 0, l_bits = 0, count = 0;
#pragma unroll
    for (int q = 0; q < kLoads; ++q) {
      word[q] = wave_transpose(word[q]);
      const uint64_t mask = ballot(word[q] != 0);
      const uint32_t bits = want_bits ? wave_sum32(static_cast<uint32_t>(__popcll(word[q]))) : 0u;
      if (lane == q) {
        l_mask = mask;
        l_at = count;
        l_bits = bits;
      }
      count += static_cast<uint32_t>(__popcll(mask));
    }
    bool fits = false;
    uint64_t base = 0;
    if (!next) {
      fits = true;
      base = job.words0 + i0 * kTile;
      l_at = lane * kTile;
    } else if (cap) {
      if (lane == 0) s_count[wave] = count;
      __syncthreads();
      uint32_t before = 0, total = 0;
      for (uint32_t w = 0; w < kWaves; ++w) {
        const uint32_t c = s_count[w];
        if (w < wave) before += c;
        total += c;
      }
      if (threadIdx.x == 0 && total) s_base = atomicAdd(next, static_cast<unsigned long long>(total));
      __syncthreads();
      fits = total != 0 && s_base + total <= cap;
      base = s_base + before;
      __syncthreads();
    }
    if (fits) {
      uint64_t to = base;
#pragma unroll
      for (int q = 0; q < kLoads; ++q) {
        const uint64_t mask = ballot(word[q] != 0);
        if (word[q]) words[to + lanes_under(mask)] = word[q];
        to += next ? static_cast<uint32_t>(__popcll(mask)) : kTile;
      }
    }
    if (writes) {
      const uint64_t i = i0 + lane;
      const TileHead h{l_mask, fits ? static_cast<uint32_t>(base) + l_at : kNoWords, l_bits};
      job.head[at] = h;
      if (job.head_by_tile) job.head_by_tile[i] = h;
      if (job.tile) job.tile[at] = static_cast<uint32_t>(i);
      if (job.used) job.used[i] = static_cast<uint8_t>(__popcll(l_mask));
    }
  }
}

// Weights of an operand's tile rows: the columns in use of their tiles, summed; then the sums of kWindow
// rows each and of all (an estimate: it may wrap). A workgroup takes kWindow rows, a wave each.
constexpr uint32_t kWindow = 16;  // strips of C per workgroup of the product: 16 KiB of LDS for their tiles
struct WeightJob {
  const uint8_t* used;
  const uint32_t* off;
  uint32_t* weight;  // n_strips, total (cleared), groups; null: none
};
__global__ void __launch_bounds__(kWindow* kWave) row_weights_kernel(WeightJob job0, WeightJob job1, uint32_t n_strips) {
  __shared__ uint32_t s_sum[kWindow];
  const WeightJob& job = blockIdx.y ? job1 : job0;
  if (!job.weight) return;
  const uint32_t lane = lane_id(), wave = read_first_lane(threadIdx.x / kWave);
  uint32_t all = 0;
  for (uint32_t g = blockIdx.x; g * kWindow < n_strips; g += gridDim.x) {
    const uint32_t x = g * kWindow + wave;
    uint32_t sum = 0;
    if (x < n_strips) {
      const uint32_t end = job.off[x + 1];
      for (uint32_t i = job.off[x] + lane; i < end; i += kWave) sum += job.used[i];
    }
    sum = wave_sum32(sum);
    if (lane == 0) {
      s_sum[wave] = sum;
      if (x < n_strips) job.weight[x] = sum;
    }
    __syncthreads();
    if (wave == 0) {
      const uint32_t group = wave_sum32(lane < kWindow ? s_sum[lane] : 0u);
      if (lane == 0) job.weight[n_strips + 1 + g] = group;
      all += group;
    }
    __syncthreads();
  }
  if (threadIdx.x == 0 && all) atomicAdd(job.weight + n_strips, all);
}

// --- B by tile rows, windows of C ----------------------------------------------------------

__global__ void __launch_bounds__(kBlock) clear_words_kernel(uint64_t* __restrict__ v, uint64_t n) {
  for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += static_cast<uint64_t>(gridDim.x) * kBlock) v[i] = 0;
}

__global__ void __launch_bounds__(kBlock) clear_u32_kernel(uint32_t* __restrict__ v, uint32_t n) {
  for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) v[i] = 0;
}

__global__ void __launch_bounds__(kBlock) b_bitmap_kernel(const uint32_t* __restrict__ row,
                                                          const uint32_t* __restrict__ col, uint32_t n, uint32_t wpr,
                                                          BitmapWord* __restrict__ bm) {
  for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += static_cast<uint64_t>(gridDim.x) * kBlock) {
    const uint32_t y = row[i];
    atomicOr(reinterpret_cast<unsigned long long*>(&bm[static_cast<uint64_t>(col[i]) * wpr + (y >> 6)].bits),
             1ull << (y & 63));
  }
}

// Tiles of every row; then (off: the rows' first positions) the position of every word. One wave
// per row.
__global__ void __launch_bounds__(kBlock) b_rank_kernel(BitmapWord* __restrict__ bm, uint32_t n, uint32_t wpr,
                                                        uint32_t* __restrict__ count, const uint32_t* __restrict__ off) {
  const uint32_t lane = lane_id();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t t = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); t < n; t += n_waves) {
    uint32_t before = off ? off[t] : 0u;
    for (uint32_t w0 = 0; w0 < wpr; w0 += kWave) {
      BitmapWord* const word = bm + static_cast<uint64_t>(t) * wpr + w0 + lane;
      const uint32_t c = w0 + lane < wpr ? static_cast<uint32_t>(__popcll(word->bits)) : 0u;
      uint32_t incl = c;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), d, kWave));
        if (lane >= static_cast<uint32_t>(d)) incl += o;
      }
      if (off && w0 + lane < wpr) word->at = before + incl - c;
      before += lane_u32(incl, kWave - 1);
    }
    if (lane == 0 && !off) count[t] = before;
  }
}

// off[0 .. n] = exclusive prefix sums of count[0 .. n), returned: their sum. One workgroup.
constexpr int kScanWaves = 16;
__device__ inline uint32_t row_offsets(const uint32_t* __restrict__ count, uint32_t n, uint32_t* __restrict__ off) {
  __shared__ uint32_t s_sum[kScanWaves];
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  uint32_t before = 0;
  for (uint32_t i0 = 0; i0 < n; i0 += kScanWaves * kWave) {
    const uint32_t i = i0 + threadIdx.x;
    const uint32_t c = i < n ? count[i] : 0u;
    uint32_t incl = c;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), d, kWave));
      if (lane >= static_cast<uint32_t>(d)) incl += o;
    }
    if (lane == kWave - 1) s_sum[wave] = incl;
    __syncthreads();
    uint32_t base = before, total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kScanWaves; ++w) {
      if (w < wave) base += s_sum[w];
      total += s_sum[w];
    }
    if (i < n) off[i] = base + incl - c;
    before += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) off[n] = before;
  return before;
}
__global__ void __launch_bounds__(kScanWaves* kWave) row_offsets_kernel(const uint32_t* __restrict__ count, uint32_t n,
                                                                        uint32_t* __restrict__ off) {
  row_offsets(count, n, off);
}

// Windows of C in use: kWindow strips; kWindow / 4 or one where they would be much work. A
// window's work is about the columns in use in A's row times those in its rows of Bt, and one
// with more than 1 / kShares of the whole product's is cut: the hubs of a power-law graph make
// windows that one workgroup would still be at long after the rest (A*A of R-MAT 14: 405 us without
// the cut, 172 with; 1024 or 16384 shares: 177, 194).
constexpr float kShares = 4096;
__global__ void __launch_bounds__(kScanWaves* kWave) windows_kernel(ProductTiles C, uint32_t n_strips,
                                                         const uint32_t* __restrict__ off_a,
                                                         const uint32_t* __restrict__ weight_a,
                                                         const uint32_t* __restrict__ weight_b,
                                                         const uint32_t* __restrict__ group_b,
                                                         Window* __restrict__ windows,
                                                         uint32_t* __restrict__ n_windows) {
  const uint32_t lane = lane_id();
  __shared__ uint32_t s_count[kScanWaves], s_base;
  const float total = static_cast<float>(weight_a[n_strips]) * static_cast<float>(weight_b[n_strips]);
  const uint32_t wave = threadIdx.x / kWave;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * blockDim.x; i0 < C.n_c; i0 += stride) {
    const uint64_t i = i0 + threadIdx.x;
    bool head = false;
    uint32_t width = kWindow;
    if (i < C.n_c) {
      const uint32_t x = C.row[i], y = C.col[i];
      const float share =
          total > 0 ? static_cast<float>(weight_a[x]) * static_cast<float>(group_b[y / kWindow]) * kShares / total : 0.0f;
      width = share <= 1.0f ? kWindow : share <= 4.0f ? kWindow / 4 : 1;
      head = i == 0 || C.row[i - 1] != x || C.col[i - 1] / width != y / width;
    }
    const uint64_t m = ballot(head);
    if (lane == 0) s_count[wave] = static_cast<uint32_t>(__popcll(m));
    __syncthreads();
    uint32_t before = 0, sum = 0;
    for (uint32_t w = 0; w < kScanWaves; ++w) {
      if (w < wave) before += s_count[w];
      sum += s_count[w];
    }
    if (threadIdx.x == 0) s_base = sum ? atomicAdd(n_windows, sum) : 0u;
    __syncthreads();
    const uint32_t base = s_base + before;
    __syncthreads();
    if (head) {
      const uint32_t x = C.row[i], y = C.col[i];
      windows[base + lanes_under(m)] = Window{static_cast<uint32_t>(i), x, y / kWindow * kWindow,
                                              y / width * width + width, off_a[x], off_a[x + 1], {0, 0}};
    }
  }
}

// Structural pass. Workgroup = tile row x: lane = word of B's bitmap rows, ORed over A's tiles in
// registers, kUnionLoads rows in flight per wave; the waves meet in LDS. A frontier has few rows and
// many tiles in each, so a row has 16 waves.
constexpr int kUnionWaves = 16;
constexpr int kUnionLoads = 8;
__global__ void __launch_bounds__(kUnionWaves* kWave) union_rows_kernel(const uint32_t* __restrict__ off_a,
                                                                        const uint32_t* __restrict__ col_a,
                                                                        const BitmapWord* __restrict__ bm,
                                                                        const uint32_t* __restrict__ off_b, uint32_t n,
                                                                        uint32_t wpr, SymbolicRows S) {
  __shared__ unsigned long long s_or[kWave], s_tp;
  const uint32_t lane = lane_id(), wave = read_first_lane(threadIdx.x / kWave);
  for (uint32_t x = blockIdx.x; x < n; x += gridDim.x) {
    const uint32_t a0 = off_a[x], a1 = off_a[x + 1];
    if (a0 == a1) {  // uniform
      if (threadIdx.x == 0) {
        S.cnt[x] = 0;
        S.tp[x] = 0;
      }
      continue;
    }
    if (threadIdx.x == 0) s_tp = 0;
    __syncthreads();
    uint64_t tp = 0;
    for (uint32_t k = a0 + threadIdx.x; k < a1; k += kUnionWaves * kWave) {
      const uint32_t t = col_a[k];
      tp += off_b[t + 1] - off_b[t];
      S.ref[t] = 1;
    }
    tp = wave_sum(tp);
    if (lane == 0 && tp) atomicAdd(&s_tp, static_cast<unsigned long long>(tp));
    uint32_t count = 0;
    for (uint32_t w0 = 0; w0 < wpr; w0 += kWave) {
      if (wave == 0) s_or[lane] = 0;
      __syncthreads();
      const bool has = w0 + lane < wpr;
      uint64_t acc = 0;
      for (uint32_t k0 = a0 + wave * kUnionLoads; k0 < a1; k0 += kUnionWaves * kUnionLoads) {
        uint64_t word[kUnionLoads];
#pragma unroll
        for (int q = 0; q < kUnionLoads; ++q) {
          word[q] = 0;
          if (k0 + q < a1 && has) word[q] = bm[static_cast<uint64_t>(col_a[k0 + q]) * wpr + w0 + lane].bits;
        }
#pragma unroll
        for (int q = 0; q < kUnionLoads; ++q) acc |= word[q];
      }
      if (acc) atomicOr(&s_or[lane], static_cast<unsigned long long>(acc));
      __syncthreads();
      if (wave == 0) {
        const uint64_t bits = s_or[lane];
        if (has) S.c_bits[static_cast<uint64_t>(x) * wpr + w0 + lane] = bits;
        count += wave_sum32(static_cast<uint32_t>(__popcll(bits)));
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      S.cnt[x] = count;
      S.tp[x] = s_tp;
    }
    __syncthreads();
  }
}

// C's row pointer and the totals; one workgroup.
__global__ void __launch_bounds__(kScanWaves* kWave) symbolic_totals_kernel(SymbolicRows S,
                                                                            const uint32_t* __restrict__ off_b,
                                                                            uint32_t n) {
  __shared__ unsigned long long s_tp, s_used;
  if (threadIdx.x == 0) s_tp = s_used = 0;
  __syncthreads();
  uint64_t tp = 0, used = 0;
  for (uint32_t x = threadIdx.x; x < n; x += kScanWaves * kWave) {
    tp += S.tp[x];
    if (S.ref[x]) used += off_b[x + 1] - off_b[x];
  }
  tp = wave_sum(tp);
  used = wave_sum(used);
  if (lane_id() == 0) {
    atomicAdd(&s_tp, static_cast<unsigned long long>(tp));
    atomicAdd(&s_used, static_cast<unsigned long long>(used));
  }
  const uint32_t n_c = row_offsets(S.cnt, n, S.off_c);
  if (threadIdx.x == 0) {
    S.sums[0] = s_tp;
    S.sums[1] = s_used;
    S.sums[2] = n_c;  // fits: kBitmapStrips rows of as many strips
  }
}

// One wave per row: each word's tiles, lane = strip.
__global__ void __launch_bounds__(kBlock) symbolic_emit_kernel(SymbolicRows S, uint32_t n, uint32_t wpr,
                                                               uint32_t* __restrict__ row_c,
                                                               uint32_t* __restrict__ col_c) {
  const uint32_t lane = lane_id();
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * kWavesPerBlock, per_row = (wpr + kWave - 1) / kWave;
  for (uint64_t i = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); i < n * per_row; i += n_waves) {
    const uint32_t x = static_cast<uint32_t>(i / per_row), w0 = static_cast<uint32_t>(i % per_row) * kWave;
    uint32_t at = S.off_c[x];
    if (at == S.off_c[x + 1]) continue;
    const uint64_t* const row = S.c_bits + static_cast<uint64_t>(x) * wpr;
    for (uint32_t w = lane; w < w0; w += kWave) at += static_cast<uint32_t>(__popcll(row[w]));
    at = wave_sum32(at) - (kWave - 1) * S.off_c[x];
    const uint64_t bits = w0 + lane < wpr ? row[w0 + lane] : 0ull;
    for (uint64_t m = ballot(bits != 0); m; m &= m - 1) {
      const int w = lowest(m);
      const uint64_t word = read_lane(bits, w);
      if ((word >> lane) & 1) {
        const uint32_t to = at + lanes_under(word);
        row_c[to] = x;
        col_c[to] = (w0 + static_cast<uint32_t>(w)) * 64 + lane;
      }
      at += static_cast<uint32_t>(__popcll(word));
    }
  }
}

// Set bits of row t of B / its tiles with at least min_bits; one wave per row of a bitmap grid, else
// per tile with atomics into a cleared out.
__device__ inline uint64_t row_term(const TileHead& h, uint32_t min_bits, bool count) {
  return count ? (h.bits >= min_bits ? 1u : 0u) : h.bits;
}
__global__ void __launch_bounds__(kBlock) row_sum_kernel(RightOperand B, uint32_t n, uint32_t min_bits, bool count,
                                                         unsigned long long* __restrict__ out) {
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t t = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); t < n; t += n_waves) {
    uint64_t sum = 0;
    const uint32_t end = B.off[t + 1];
    for (uint32_t p = B.off[t] + lane_id(); p < end; p += kWave) sum += row_term(B.head[p], min_bits, count);
    sum = wave_sum(sum);
    if (lane_id() == 0) out[t] = sum;
  }
}
__global__ void __launch_bounds__(kBlock) tile_sum_kernel(RightOperand B, uint32_t n_b, uint32_t min_bits, bool count,
                                                          unsigned long long* __restrict__ out) {
  for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n_b; i += static_cast<uint64_t>(gridDim.x) * kBlock) {
    const uint64_t v = row_term(B.head[i], min_bits, count);
    if (v) atomicAdd(out + B.bt_col[i], static_cast<unsigned long long>(v));
  }
}
// Pairs of tiles that both have at least min_bits set bits (count: B's per row).
__global__ void __launch_bounds__(kBlock) heavy_pairs_kernel(LeftOperand A, uint32_t n_a, uint32_t min_bits,
                                                             const unsigned long long* __restrict__ count,
                                                             unsigned long long* __restrict__ out) {
  uint64_t local = 0;
  for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n_a; i += static_cast<uint64_t>(gridDim.x) * kBlock)
    if (A.head[i].bits >= min_bits) local += count[A.col[i]];
  local = wave_sum(local);
  if (lane_id() == 0 && local) atomicAdd(out, static_cast<unsigned long long>(local));
}

// --- the product ------------------------------------------------------------------------

constexpr uint32_t kQueue = 192;     // entries of a wave's queues: less than a wave's, and two from each lane
// Common inner indices up to which a pair is queued per index (8 or 64: 7 and 6 % slower on the
// communities above).
constexpr int kFewCommon = 16;
constexpr int kPairBatch = 4;        // pairs with more whose loads are in flight together (8: 7 % slower)
// Waves of a workgroup. More do not shorten a window's chain of loads, they only halve its batches:
// 1.45 ms with 4, 2.14 with 8, 3.21 with 16 (communities, before the queues took two entries a step).
constexpr uint32_t kProductWaves = 4;

struct WaveQueues {
  uint32_t pair_a[kQueue], pair_b[kQueue];  // tile of A, position of B
  uint32_t item_a[kQueue], item_b[kQueue];  // column words
  uint8_t pair_s[kQueue], item_s[kQueue];   // strip of the window
};

// A dense pair of C tile `c`, to be multiplied on the matrix cores: the rank-th that was found there.
struct HeavyPair {
  uint32_t c, rank, a, b;
};
// The record has kHeavyParts parts of `part` places, each with a counter on a cache line of its own:
// additions to one address come 12 ns apart, and recording 16.8 M pairs took 3.3 ms on one counter, now
// 0.18. A wave that finds its part full goes on with the next; the parts together have room for all.
// The rank, taken in LDS, gives heavy_scatter_kernel the pair's place (0.10 ms; 1.15 with a cursor
// in memory for each C tile).
constexpr uint32_t kHeavyParts = 64;
constexpr uint32_t kPartStride = 16;  // u64 counters
struct HeavyRecord {
  HeavyPair* pairs;
  uint32_t* count;              // per C tile
  unsigned long long* counter;  // places taken of each part, or more
  uint32_t part;
  uint32_t min_bits;
};

// First index of a[lo, hi) (ascending) not below key.
__device__ inline uint32_t lower_bound(const uint32_t* __restrict__ a, uint32_t lo, uint32_t hi, uint32_t key) {
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (a[mid] < key) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// The outer product rows x cols into the C tile at `by_row` / `by_col`; true if into by_col. Each lane
// starts at another bit: neighbours' words are often alike, and equal addresses would queue up.
__device__ inline bool or_outer(unsigned long long* by_row, unsigned long long* by_col, uint64_t rows, uint64_t cols,
                                uint32_t lane) {
  const bool r = __popcll(rows) <= __popcll(cols);
  unsigned long long* const acc = r ? by_row : by_col;
  const uint64_t word = r ? rows : cols;
  const unsigned long long val = r ? cols : rows;
  uint64_t each = (word >> lane) | (word << ((64 - lane) & 63));
  if (val)
    for (; each; each &= each - 1) atomicOr(acc + ((lowest(each) + lane) & 63), val);
  return !r && val;
}

// Records the pairs of the lanes of `hm` (h: this lane's).
__device__ inline void record_heavy(const HeavyRecord& heavy, uint32_t& part, bool h, uint64_t hm, const HeavyPair& pair,
                                    uint32_t lane) {
  const uint32_t order = lanes_under(hm), n = static_cast<uint32_t>(__popcll(hm));
  uint32_t done = 0;
  for (uint32_t tries = 0; done < n && tries < kHeavyParts; ++tries) {
    unsigned long long at = 0;
    if (lane == 0) at = atomicAdd(heavy.counter + part * kPartStride, static_cast<unsigned long long>(n - done));
    at = read_first_lane64(at);
    const uint32_t room = at < heavy.part ? min(n - done, heavy.part - static_cast<uint32_t>(at)) : 0u;
    if (h && order >= done && order - done < room)
      heavy.pairs[static_cast<uint64_t>(part) * heavy.part + at + (order - done)] = pair;
    done += room;
    if (done < n) part = (part + 1) % kHeavyParts;
  }
}

// The pairs of the lanes of `wm`, which share many inner indices (or have column words that are not
// stored), one after the other with lane = j; s: the pair's C tile in by_row / by_col. True if by_col
// was used.
template <int kBatch>
__device__ inline bool or_whole_pairs(uint64_t wm, const LeftOperand& A, const RightOperand& B, const TileHead& ha,
                                      const TileHead& hb, uint32_t ia, uint32_t pb, uint32_t s,
                                      unsigned long long* by_row, unsigned long long* by_col, uint32_t lane) {
  bool cols = false;
  while (wm) {
    uint64_t r[kBatch], c[kBatch];
    uint32_t sp[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      r[k] = 0;
      c[k] = 0;
      sp[k] = 0;
      if (wm) {
        const int src = lowest(wm);
        wm &= wm - 1;
        const uint64_t ma = read_lane(ha.mask, src), mb = read_lane(hb.mask, src);
        const uint32_t oa = lane_u32(ha.off, src), ob = lane_u32(hb.off, src);
        sp[k] = lane_u32(s, src) * kTile;
        const bool use = ((ma & mb) >> lane) & 1;
        if (oa != kNoWords) {
          if (use) r[k] = A.words[oa + lanes_under(ma)];
        } else {
          const uint64_t t = wave_transpose(A.data[static_cast<uint64_t>(lane_u32(ia, src)) * kTile + lane]);
          if (use) r[k] = t;
        }
        if (ob != kNoWords) {
          if (use) c[k] = B.words[ob + lanes_under(mb)];
        } else {
          const uint32_t p = lane_u32(pb, src);
          const uint64_t t = wave_transpose(B.data[static_cast<uint64_t>(B.tile ? B.tile[p] : p) * kTile + lane]);
          if (use) c[k] = t;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) cols |= or_outer(by_row + sp[k], by_col + sp[k], r[k], c[k], lane);
  }
  return cols;
}

template <bool kHeavy, int kOut>
__global__ void __launch_bounds__(kProductWaves* kWave) product_kernel(ProductTiles C, const Window* __restrict__ windows,
                                                                   const uint32_t* __restrict__ n_windows, uint32_t wpr,
                                                                   LeftOperand A, RightOperand B, ProductOut out,
                                                                   HeavyRecord heavy) {
  __shared__ unsigned long long by_row[kWindow * kTile], by_col[kWindow * kTile];
  __shared__ WaveQueues s_queues[kProductWaves];
  __shared__ uint32_t s_used;
  __shared__ uint32_t s_heavy[kHeavy ? kWindow : 1];  // dense pairs of each strip's tile
  __shared__ unsigned long long s_slot;
  const uint32_t lane = lane_id();
  const uint32_t wave = read_first_lane(threadIdx.x / kWave);
  constexpr uint32_t n_waves = kProductWaves;
  WaveQueues& q = s_queues[wave];
  uint32_t heavy_part = (blockIdx.x * kProductWaves + wave) % kHeavyParts;
  const uint32_t n_items = *n_windows;
  for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
    const Window win = windows[item];
    const uint32_t y0 = win.y0, a0 = win.a0, a1 = win.a1;
    const uint32_t mine = win.first + lane;
    const bool in_row = lane < kWindow && lane < C.n_c - win.first && C.row[mine] == win.x;
    const uint32_t col = in_row ? C.col[mine] : win.end;
    uint32_t present = col < win.end ? 1u << (col - y0) : 0u;  // strips with a tile of C
#pragma unroll
    for (uint32_t d = 1; d < kWindow; d <<= 1) present |= shfl_xor32(present, static_cast<int>(d));
    present = read_first_lane(present);
    if constexpr (kOut == kOutRest) {  // windows without a tile to write: uniform over the workgroup
      if (!ballot(col < win.end && out.flag[mine] && out.slot[mine] >= out.capacity)) continue;
    }
    const auto c_tile = [&](uint32_t s) { return win.first + static_cast<uint32_t>(__popc(present & ((1u << s) - 1))); };
    for (uint32_t i = threadIdx.x; i < kWindow * kTile; i += kProductWaves * kWave) by_row[i] = by_col[i] = 0;
    if constexpr (kHeavy) {
      if (threadIdx.x < kWindow) s_heavy[threadIdx.x] = 0;
    }
    __syncthreads();

    uint32_t n_pairs = 0, n_queued = 0;  // queued (wave-uniform)
    // Stages 2 and 3 issue the loads of one batch before they work on the one before it.
    uint64_t item_r = 0, item_c = 0;
    uint32_t item_s = 0;
    // Stage 3: fetches the last n <= 64 queued (pair, j).
    const auto multiply = [&](uint32_t n) {
      n_queued -= n;
      wave_lds_sync();
      uint64_t r = 0, c = 0;
      uint32_t s = 0;
      if (lane < n) {
        const uint32_t at = n_queued + lane;
        r = A.words[q.item_a[at]];
        c = B.words[q.item_b[at]];
        s = q.item_s[at] * kTile;
      }
      or_outer(by_row + item_s, by_col + item_s, item_r, item_c, lane);
      item_r = r;
      item_c = c;
      item_s = s;
      wave_lds_sync();
    };
    uint32_t next_a = 0, next_b = 0, next_s = 0;
    TileHead next_ha{0, 0, 0}, next_hb{0, 0, 0};
    uint32_t fetched = 0;  // pairs (wave-uniform)
    // Stage 2: fetches the heads of the last n <= 64 queued pairs.
    const auto filter = [&](uint32_t n) {
      const uint32_t ia = next_a, pb = next_b, s = next_s;
      const TileHead ha = next_ha, hb = next_hb;
      n_pairs -= n;
      wave_lds_sync();
      next_ha.mask = next_hb.mask = 0;
      if constexpr (kHeavy) next_ha.bits = next_hb.bits = 0;
      if (lane < n) {
        const uint32_t at = n_pairs + lane;
        next_a = q.pair_a[at];
        next_b = q.pair_b[at];
        next_s = q.pair_s[at];
        next_ha = A.head[next_a];
        next_hb = B.head[next_b];
      }
      wave_lds_sync();
      const bool has = lane < fetched;
      fetched = n;
      uint64_t common = ha.mask & hb.mask;
      if constexpr (kHeavy) {
        const bool h = has && ha.bits >= heavy.min_bits && hb.bits >= heavy.min_bits;
        const uint64_t hm = ballot(h);
        if (hm) {
          const uint32_t rank = h ? atomicAdd(&s_heavy[s], 1u) : 0u;
          record_heavy(heavy, heavy_part, h, hm, h ? HeavyPair{c_tile(s), rank, ia, B.tile ? B.tile[pb] : pb} : HeavyPair{}, lane);
          if (h) common = 0;
        }
      }
      const int n_common = __popcll(common);
      const bool whole = n_common > kFewCommon || (common && (ha.off == kNoWords || hb.off == kNoWords));
      or_whole_pairs<kPairBatch>(ballot(whole), A, B, ha, hb, ia, pb, s, by_row, by_col, lane);
      if (whole) common = 0;
      // The rest, two j per lane at a time (1.32 ms instead of 1.43: a step's ballots, branch and LDS
      // writes are one dependent chain), a 32-bit half of the masks after the other: bits of the half
      // below j, counted onto the words before it, give the two column words.
      const auto queue = [&](uint32_t left, uint32_t in_a, uint32_t in_b, uint32_t first_a, uint32_t first_b) {
        const auto put = [&](uint32_t bits, uint64_t m) {
          if (bits) {
            const uint32_t below = (bits - 1) & ~bits;
            const uint32_t to = n_queued + lanes_under(m);
            q.item_a[to] = first_a + static_cast<uint32_t>(__popc(in_a & below));
            q.item_b[to] = first_b + static_cast<uint32_t>(__popc(in_b & below));
            q.item_s[to] = static_cast<uint8_t>(s);
          }
          n_queued += static_cast<uint32_t>(__popcll(m));
        };
        for (uint64_t m = ballot(left != 0); m; m = ballot(left != 0)) {
          const uint32_t next = left & (left - 1);
          const uint64_t m_next = ballot(next != 0);
          put(left, m);
          put(next, m_next);
          left = next & (next - 1);
          while (n_queued >= kWave) multiply(kWave);
        }
      };
      const uint32_t lo_a = static_cast<uint32_t>(ha.mask), lo_b = static_cast<uint32_t>(hb.mask);
      queue(static_cast<uint32_t>(common), lo_a, lo_b, ha.off, hb.off);
      queue(static_cast<uint32_t>(common >> 32), static_cast<uint32_t>(ha.mask >> 32), static_cast<uint32_t>(hb.mask >> 32),
            ha.off + static_cast<uint32_t>(__popc(lo_a)), hb.off + static_cast<uint32_t>(__popc(lo_b)));
    };

    // Stage 1: the row's tiles, dealt one by one to the waves, so that short rows use them all.
    for (uint32_t k0 = a0; k0 < a1; k0 += kWave * n_waves) {
      const uint32_t ia = k0 + lane * n_waves + wave;
      uint32_t bits = 0, pb = 0;  // strips of the window, and the position of the lowest
      if (ia < a1) {
        const uint32_t t = A.col[ia];
        const BitmapWord w = B.bm[static_cast<uint64_t>(t) * wpr + (y0 >> 6)];
        bits = static_cast<uint32_t>(w.bits >> (y0 & 63)) & ((1u << kWindow) - 1);
        pb = w.at + static_cast<uint32_t>(__popcll(w.bits & ((1ull << (y0 & 63)) - 1)));
      }
      const uint32_t all = bits;
      bits &= present;
      const auto put = [&](uint32_t left, uint64_t m) {
        if (left) {
          const uint32_t below = (left - 1) & ~left;
          const uint32_t to = n_pairs + lanes_under(m);
          q.pair_a[to] = ia;
          q.pair_b[to] = pb + static_cast<uint32_t>(__popc(all & below));
          q.pair_s[to] = static_cast<uint8_t>(__popc(below));
        }
        n_pairs += static_cast<uint32_t>(__popcll(m));
      };
      for (uint64_t m = ballot(bits != 0); m; m = ballot(bits != 0)) {
        const uint32_t next = bits & (bits - 1);
        const uint64_t m_next = ballot(next != 0);
        put(bits, m);
        put(next, m_next);
        bits = next & (next - 1);
        while (n_pairs >= kWave) filter(kWave);
      }
    }
    while (n_pairs || fetched) filter(n_pairs);
    multiply(n_queued);
    multiply(0);
    __syncthreads();
    if constexpr (kHeavy) {
      if (threadIdx.x < kWindow && (present >> threadIdx.x) & 1) heavy.count[c_tile(threadIdx.x)] = s_heavy[threadIdx.x];
    }
    // Write-out: one C tile per wave at a time.
    if constexpr (kOut == kOutAppend) {
      // The window's non-empty tiles take their slots together: one counter for all of C.
      if (threadIdx.x == 0) s_used = 0;
      __syncthreads();
      for (uint32_t s = wave; s < kWindow; s += n_waves) {
        if (!((present >> s) & 1)) continue;
        const uint64_t val = by_row[s * kTile + lane] | wave_transpose(by_col[s * kTile + lane]);
        by_row[s * kTile + lane] = val;
        if (ballot(val != 0) && lane == 0) atomicOr(&s_used, 1u << s);
      }
      __syncthreads();
      const uint32_t used = s_used;
      if (threadIdx.x == 0) s_slot = used ? atomicAdd(out.counter, static_cast<unsigned long long>(__popc(used))) : 0ull;
      __syncthreads();
      for (uint32_t s = wave; s < kWindow; s += n_waves) {
        if (!((present >> s) & 1)) continue;
        const bool nz = (used >> s) & 1;
        const uint64_t slot = s_slot + static_cast<uint32_t>(__popc(used & ((1u << s) - 1)));
        const uint32_t i = c_tile(s);
        if (lane == 0) {
          out.flag[i] = nz ? 1u : 0u;
          if (nz) out.slot[i] = static_cast<uint32_t>(slot);
        }
        if (nz && slot < out.capacity) out.data[slot * kTile + lane] = by_row[s * kTile + lane];
      }
      __syncthreads();
      continue;
    }
    for (uint32_t s = wave; s < kWindow; s += n_waves) {
      if (!((present >> s) & 1)) continue;
      const uint64_t val = by_row[s * kTile + lane] | wave_transpose(by_col[s * kTile + lane]);
      const uint32_t i = c_tile(s);
      if constexpr (kOut == kOutStruct) {
        // Only this wave has the tile; an atomic needs no answer, a load would be waited for.
        if (val) atomicOr(reinterpret_cast<unsigned long long*>(out.data) + static_cast<uint64_t>(i) * kTile + lane,
                          static_cast<unsigned long long>(val));
      } else if constexpr (kOut == kOutRest) {
        const uint64_t slot = out.flag[i] ? out.slot[i] : 0u;
        if (slot >= out.capacity) out.data[(slot - out.capacity) * kTile + lane] = val;
      } else {
        const bool nz = ballot(val != 0) != 0;
        if constexpr (kOut == kOutFlag) {
          if (lane == 0) out.flag[i] = nz ? 1u : 0u;
        } else if (nz) {
          out.data[static_cast<uint64_t>(out.pos[i]) * kTile + lane] = val;
        }
      }
    }
    __syncthreads();
  }
}

// The product C tile by C tile, for products that by_tiles picks: a wave takes `run` neighbouring C
// tiles, one after the other, each with 1 KiB of LDS. Lane = tile of the shorter of A's row and Bt's,
// searched in the longer, then the same two stages as product_kernel's, without queues: few pairs meet
// here, and what bounds it is the chain of dependent loads (rows, search, heads, words), which 32
// waves a CU hide, not idle lanes. A window that holds a tile or two costs a workgroup, 30 KiB of LDS
// and their clearing. Erdos-Renyi A*A with a quarter of an edge a vertex, operands prepared: 2^18
// vertices (1.0 M C tiles) 0.255 ms, by windows 1.40; 2^20 (4.2 M) 1.21 and 7.86; 2^21 (8.3 M, too wide
// for windows by bitmap) 2.57, by windows that search 25.9. 2^12 vertices with half an edge, 4096 C
// tiles: 15 us and 29.
constexpr uint32_t kTileRun = 8;
constexpr int kTilePairBatch = 2;  // as kPairBatch; 64 registers hold no more
template <bool kHeavy, int kOut>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) tile_product_kernel(ProductTiles C, LeftOperand A, RightOperand B,
                                                              ProductOut out, HeavyRecord heavy, uint32_t run) {
  __shared__ unsigned long long s_row[kWavesPerBlock][kTile], s_col[kWavesPerBlock][kTile];
  __shared__ uint64_t s_done[kOut == kOutAppend ? kWavesPerBlock * kTileRun * kTile : 1];
  const uint32_t lane = lane_id(), wave = read_first_lane(threadIdx.x / kWave);
  unsigned long long* const by_row = s_row[wave];
  unsigned long long* const by_col = s_col[wave];
  by_row[lane] = by_col[lane] = 0;
  wave_lds_sync();
  const uint32_t first = blockIdx.x * kWavesPerBlock + wave;
  uint32_t heavy_part = first % kHeavyParts;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kWavesPerBlock * run;
  for (uint64_t i0 = static_cast<uint64_t>(first) * run; i0 < C.n_c; i0 += stride) {
    const uint32_t n = C.n_c - i0 < run ? static_cast<uint32_t>(C.n_c - i0) : run;
    uint32_t used = 0;  // of the run's tiles (kOutAppend)
    // Lane q: the rows of tile i0 + q, so that a run waits for them once.
    uint32_t ra0 = 0, ra1 = 0, rb0 = 0, rb1 = 0;
    if (lane < n) {
      const uint32_t x = C.row[i0 + lane], y = C.col[i0 + lane];
      ra0 = A.off[x];
      ra1 = A.off[x + 1];
      rb0 = B.bt_off[y];
      rb1 = B.bt_off[y + 1];
    }
    for (uint32_t q = 0; q < n; ++q) {
      const uint32_t i = static_cast<uint32_t>(i0) + q;
      if constexpr (kOut == kOutRest) {
        if (!out.flag[i] || out.slot[i] < out.capacity) continue;
      }
      const int src = static_cast<int>(q);
      const uint32_t a0 = lane_u32(ra0, src), a1 = lane_u32(ra1, src), b0 = lane_u32(rb0, src), b1 = lane_u32(rb1, src);
      const bool a_short = a1 - a0 <= b1 - b0;
      const uint32_t s0 = a_short ? a0 : b0, s1 = a_short ? a1 : b1, l0 = a_short ? b0 : a0, l1 = a_short ? b1 : a1;
      const uint32_t* const s_idx = a_short ? A.col : B.bt_col;
      const uint32_t* const l_idx = a_short ? B.bt_col : A.col;
      uint32_t n_heavy = 0;
      uint64_t some = 0;  // lanes with a common index so far
      bool cols = false;  // this lane used by_col
      for (uint32_t k0 = s0; k0 < s1; k0 += kWave) {
        const uint32_t k = k0 + lane;
        uint32_t at = l1;
        bool has = k < s1;
        if (has) {
          const uint32_t key = s_idx[k];
          at = lower_bound(l_idx, l0, l1, key);
          has = at < l1 && l_idx[at] == key;
        }
        const uint32_t ia = a_short ? k : at, ib = a_short ? at : k;
        TileHead ha{0, 0, 0}, hb{0, 0, 0};
        if (has) {
          ha = A.head[ia];
          hb = B.head[ib];
        }
        uint64_t common = ha.mask & hb.mask;
        if constexpr (kHeavy) {
          const bool h = has && ha.bits >= heavy.min_bits && hb.bits >= heavy.min_bits;
          const uint64_t hm = ballot(h);
          if (hm) {
            record_heavy(heavy, heavy_part, h, hm, HeavyPair{i, n_heavy + lanes_under(hm), ia, ib}, lane);
            n_heavy += static_cast<uint32_t>(__popcll(hm));
            if (h) common = 0;
          }
        }
        some |= ballot(common != 0);
        const bool whole = __popcll(common) > kFewCommon || (common && (ha.off == kNoWords || hb.off == kNoWords));
        cols |= or_whole_pairs<kTilePairBatch>(ballot(whole), A, B, ha, hb, ia, ib, 0, by_row, by_col, lane);
        if (whole) common = 0;
        while (ballot(common != 0)) {
          uint64_t r[2] = {0, 0}, c[2] = {0, 0};
#pragma unroll
          for (int u = 0; u < 2; ++u)
            if (common) {
              const uint64_t below = (common - 1) & ~common;
              r[u] = A.words[ha.off + static_cast<uint32_t>(__popcll(ha.mask & below))];
              c[u] = B.words[hb.off + static_cast<uint32_t>(__popcll(hb.mask & below))];
              common &= common - 1;
            }
          cols |= or_outer(by_row, by_col, r[0], c[0], lane);
          cols |= or_outer(by_row, by_col, r[1], c[1], lane);
        }
      }
      // Tiles with no common index (63 of 64 pairs of tiles with a bit each) stay out of LDS.
      uint64_t val = 0;
      if (some) {
        wave_lds_sync();
        val = by_row[lane];
        by_row[lane] = 0;
        if (ballot(cols)) {
          val |= wave_transpose(by_col[lane]);
          by_col[lane] = 0;
        }
        wave_lds_sync();
      }
      if constexpr (kHeavy) {
        if (lane == 0) heavy.count[i] = n_heavy;
      }
      if constexpr (kOut == kOutStruct) {
        if (val) atomicOr(reinterpret_cast<unsigned long long*>(out.data) + static_cast<uint64_t>(i) * kTile + lane,
                          static_cast<unsigned long long>(val));
      } else if constexpr (kOut == kOutAppend) {
        s_done[(wave * kTileRun + q) * kTile + lane] = val;
        used |= ballot(val != 0) ? 1u << q : 0u;
      } else if constexpr (kOut == kOutRest) {
        out.data[(out.slot[i] - out.capacity) * kTile + lane] = val;
      } else {
        const bool nz = ballot(val != 0) != 0;
        if constexpr (kOut == kOutFlag) {
          if (lane == 0) out.flag[i] = nz ? 1u : 0u;
        } else if (nz) {
          out.data[static_cast<uint64_t>(out.pos[i]) * kTile + lane] = val;
        }
      }
    }
    if constexpr (kOut == kOutAppend) {
      // The run's non-empty tiles take their slots together: one counter for all of C.
      unsigned long long slot0 = 0;
      if (lane == 0 && used) slot0 = atomicAdd(out.counter, static_cast<unsigned long long>(__popc(used)));
      slot0 = read_first_lane64(slot0);
      for (uint32_t q = 0; q < n; ++q) {
        const bool nz = (used >> q) & 1;
        const uint64_t slot = slot0 + static_cast<uint32_t>(__popc(used & ((1u << q) - 1)));
        if (lane == 0) {
          out.flag[i0 + q] = nz ? 1u : 0u;
          if (nz) out.slot[i0 + q] = static_cast<uint32_t>(slot);
        }
        // Each lane reads back what it wrote itself.
        if (nz && slot < out.capacity) out.data[slot * kTile + lane] = s_done[(wave * kTileRun + q) * kTile + lane];
      }
    }
  }
}

// Heavy pairs to their C tile's place (grid: x over a part of the record, y = the part).
__global__ void __launch_bounds__(kBlock) heavy_scatter_kernel(const HeavyPair* __restrict__ in,
                                                               const unsigned long long* __restrict__ counter,
                                                               uint32_t part, const uint32_t* __restrict__ base,
                                                               uint2* __restrict__ pairs) {
  const unsigned long long taken = counter[blockIdx.y * kPartStride];
  const uint32_t n = taken < part ? static_cast<uint32_t>(taken) : part;
  in += static_cast<uint64_t>(blockIdx.y) * part;
  for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += static_cast<uint64_t>(gridDim.x) * kBlock) {
    const HeavyPair p = in[i];
    pairs[base[p.c] + p.rank] = uint2{p.a, p.b};
  }
}

// Dense tile pairs on the matrix cores, as one contraction per C tile: for every pair
// (A(x,k), Bt(y,k)) whose two tiles both hold at least min_bits set bits, the vector kernel
// records the pair (its two tile indices) instead of multiplying it; then
// dense_contract_kernel sums, per C tile, the products of all its recorded pairs in FP32
// (v_mfma_f32_32x32x64, operands in 4 bits, four 32 x 32 output blocks, the 64 inner indices of a
// pair in one step) and turns sums > 0 into bit rows once, ORed into C. Operands are expanded from
// the bit tiles in registers: a bit becomes 1.0 or 2.0 or 0, the same power for an inner index on
// both sides, so that a product is 1, 4 or 0 and the sums (at most 2^14) are exact.
// Lane layout: lane l holds 32 values of A row l % 32 and of B column l % 32, half l / 32 of the
// inner indices (any order works if both operands use it); result register v of lane l is
// C[8 * (v / 4) + 4 * (l / 32) + v % 4][l % 32].
typedef int mg_v8i __attribute__((ext_vector_type(8)));
typedef float mg_v16f __attribute__((ext_vector_type(16)));
constexpr int kFp4 = 4;            // operand format of the instruction: e2m1
constexpr int kOne = 0x7F7F7F7F;   // block scales of 1

// The bits of x as 32 values of four bits, bit 4 i + q in nibble i of register q: nibble 2 is 1.0,
// nibble 4 is 2.0.
__device__ inline mg_v8i bits_to_fp4(uint32_t x) {
  mg_v8i out = {};
  out[0] = static_cast<int>((x << 1) & 0x22222222u);
  out[1] = static_cast<int>(x & 0x22222222u);
  out[2] = static_cast<int>(x & 0x44444444u);
  out[3] = static_cast<int>((x >> 1) & 0x44444444u);
  return out;
}
// From row `lane` of a tile: rows lane % 32 and 32 + lane % 32, half lane / 32 (lanes 32 to 63 of the
// low halves change places with lanes 0 to 31 of the high ones).
__device__ inline void split_rows(uint64_t row, uint32_t& first, uint32_t& second) {
  const auto r = __builtin_amdgcn_permlane32_swap(static_cast<uint32_t>(row), static_cast<uint32_t>(row >> 32), false, false);
  first = r[0];
  second = r[1];
}
__device__ inline mg_v16f mfma_fp4(mg_v8i a, mg_v8i b, mg_v16f c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, kFp4, kFp4, 0, kOne, 0, kOne);
}

// Up to kTaskPairs of a C tile's dense pairs.
constexpr uint32_t kTaskPairs = 64;
struct DenseTask {
  uint32_t tile, base, n;
};
// One wave per recorded task: the sums of the 64 x 64 output over all the task's pairs on the
// matrix cores, then one threshold; the rows are ORed into C atomically (several tasks may share a
// C tile). The pairs are read once, one per lane, and kStep pairs' operands are loaded before the
// step in front of them is multiplied; a last step that is not full takes the last pair twice.
// 16.8 M pairs, 64 to a C tile: 1.9 ms (4.6e15 operations a second; the matrix instructions alone 0.9),
// 5.9 with operands in bytes, whose expansion was 124 vector instructions a pair, now 26. One 512-byte
// load a tile and a swap of halves: 2.3 ms with two 256-byte loads of every second word. Neighbours
// in C's order kept to one XCD: no difference. Four waves a SIMD: left to itself the compiler takes
// 204 registers, enough for two.
constexpr uint32_t kStep = 2;
static_assert(kTaskPairs <= kWave);
// Every operand value is 0, 1 or 2 and every product 0, 1 or 4, so the FP32 sums are integers below 2^24
// in any order of the additions: no bit of a count is lost and sums > 0 is exactly counts > 0.
static_assert(kTaskPairs * kTile * 4 <= 1u << 24, "FP32 sums of a task are exact");
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) dense_contract_kernel(const DenseTask* __restrict__ tasks,
                                                                const uint32_t* __restrict__ n_tasks_ptr,
                                                                const uint2* __restrict__ pairs,
                                                                const uint64_t* __restrict__ data_a,
                                                                const uint64_t* __restrict__ data_bt,
                                                                uint64_t* __restrict__ data_c) {
  const uint32_t lane = lane_id();
  const uint32_t n_tasks = *n_tasks_ptr;
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t t = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); t < n_tasks; t += n_waves) {
    const DenseTask T = tasks[t];
    const uint32_t last = T.n - 1;
    const uint2 mine = pairs[T.base + min(lane, last)];
    mg_v16f acc00 = {}, acc01 = {}, acc10 = {}, acc11 = {};
    uint64_t ra[kStep], rb[kStep];  // row `lane` of both tiles
    const auto fetch = [&](uint32_t first) {
#pragma unroll
      for (uint32_t i = 0; i < kStep; ++i) {
        const int at = static_cast<int>(min(first + i, last));
        ra[i] = data_a[static_cast<uint64_t>(lane_u32(mine.x, at)) * kTile + lane];
        rb[i] = data_bt[static_cast<uint64_t>(lane_u32(mine.y, at)) * kTile + lane];
      }
    };
    fetch(0);
    for (uint32_t p = 0; p < T.n; p += kStep) {
      mg_v8i fa0[kStep], fa1[kStep], fb0[kStep], fb1[kStep];
#pragma unroll
      for (uint32_t i = 0; i < kStep; ++i) {
        uint32_t a0, a1, b0, b1;
        split_rows(ra[i], a0, a1);
        split_rows(rb[i], b0, b1);
        fa0[i] = bits_to_fp4(a0);
        fa1[i] = bits_to_fp4(a1);
        fb0[i] = bits_to_fp4(b0);
        fb1[i] = bits_to_fp4(b1);
      }
      if (p + kStep < T.n) fetch(p + kStep);
#pragma unroll
      for (uint32_t i = 0; i < kStep; ++i) {
        acc00 = mfma_fp4(fa0[i], fb0[i], acc00);
        acc01 = mfma_fp4(fa0[i], fb1[i], acc01);
        acc10 = mfma_fp4(fa1[i], fb0[i], acc10);
        acc11 = mfma_fp4(fa1[i], fb1[i], acc11);
      }
    }
    uint64_t out = 0;  // output row `lane`
#pragma unroll
    for (uint32_t v = 0; v < 16; ++v) {
      const uint32_t i0 = 8 * (v / 4) + (v % 4);
      const uint64_t b00 = ballot(acc00[v] > 0), b01 = ballot(acc01[v] > 0);
      const uint64_t b10 = ballot(acc10[v] > 0), b11 = ballot(acc11[v] > 0);
      if (lane == i0) out |= (b00 & 0xFFFFFFFFull) | ((b01 & 0xFFFFFFFFull) << 32);
      if (lane == i0 + 4) out |= (b00 >> 32) | ((b01 >> 32) << 32);
      if (lane == 32 + i0) out |= (b10 & 0xFFFFFFFFull) | ((b11 & 0xFFFFFFFFull) << 32);
      if (lane == 32 + i0 + 4) out |= (b10 >> 32) | ((b11 >> 32) << 32);
    }
    if (out) atomicOr(reinterpret_cast<unsigned long long*>(data_c) + static_cast<uint64_t>(T.tile) * kTile + lane,
                      static_cast<unsigned long long>(out));
  }
}


// The tasks of kBlock C tiles at a time take their places together (an addition for each wave's tiles
// took 50 us for 262 K tiles).
__global__ void __launch_bounds__(kBlock) heavy_tasks_kernel(const uint32_t* __restrict__ base, uint32_t n_c,
                                                             DenseTask* __restrict__ tasks,
                                                             uint32_t* __restrict__ n_tasks) {
  __shared__ uint32_t s_n, s_at;
  for (uint64_t first = static_cast<uint64_t>(blockIdx.x) * kBlock; first < n_c;
       first += static_cast<uint64_t>(gridDim.x) * kBlock) {
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const uint64_t i = first + threadIdx.x;
    uint32_t p = i < n_c ? base[i] : 0u;
    const uint32_t end = i < n_c ? base[i + 1] : 0u;
    uint32_t to = p < end ? atomicAdd(&s_n, (end - p + kTaskPairs - 1) / kTaskPairs) : 0u;
    __syncthreads();
    if (threadIdx.x == 0) s_at = s_n ? atomicAdd(n_tasks, s_n) : 0u;
    __syncthreads();
    for (to += s_at; p < end; p += kTaskPairs) tasks[to++] = DenseTask{static_cast<uint32_t>(i), p, min(kTaskPairs, end - p)};
  }
}

template <bool kHeavy, int kOut>
void launch_product(mg_context* ctx, const ProductInputs& P, const ProductOut& out, const HeavyRecord& heavy) {
  const ProductTiles& C = P.c;
  if (!C.n_c) return;
  if (P.b.bm) {
    product_kernel<kHeavy, kOut><<<std::min(65536u, C.n_c), kProductWaves * kWave, 0, ctx->stream>>>(
        C, P.windows, P.n_windows, (P.n_strips + 63) / 64, P.a, P.b, out, heavy);
  } else {
    // Runs that leave all the chip's waves work; where pairs are many they are not alike, and a run only
    // makes the last waves longer. Appends want runs: a slot counter's atomic each.
    const bool few = P.pairs <= (kOut == kOutAppend ? 16ull : 4ull) * C.n_c;
    const uint32_t per_run = kOut == kOutAppend ? (few ? 4096u : 65536u) : (few ? 32768u : ~0u);
    const uint32_t run = std::clamp(C.n_c / per_run, 1u, kTileRun);
    tile_product_kernel<kHeavy, kOut><<<grid_for(C.n_c, kWavesPerBlock * run, 65536), kBlock, 0, ctx->stream>>>(
        C, P.a, P.b, out, heavy, run);
  }
  MG_LAUNCH_CHECK();
}

void clear_u32(hipStream_t st, uint32_t* v, uint32_t n) {
  if (!n) return;
  clear_u32_kernel<<<grid_for(n, kBlock, 4096), kBlock, 0, st>>>(v, n);
  MG_LAUNCH_CHECK();
}

// B's index: the words of bm cleared, then its bits, its rows' tiles and the words' positions.
// count: n_strips of scratch.
void launch_right_index(hipStream_t st, const mg_tiled_matrix* bt, BitmapWord* bm, uint32_t* off, uint32_t* count) {
  const uint32_t ns = bt->n_strips, wpr = (ns + 63) / 64, n = bt->n_nz_tile;
  const uint64_t words = 2ull * ns * wpr;
  clear_words_kernel<<<grid_for(words, kBlock, 8192), kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(bm), words);
  MG_LAUNCH_CHECK();
  if (n) {
    b_bitmap_kernel<<<grid_for(n, kBlock, 4096), kBlock, 0, st>>>(bt->row_idx.get(), bt->col_idx.get(), n, wpr, bm);
    MG_LAUNCH_CHECK();
  }
  b_rank_kernel<<<grid_for(ns, kWavesPerBlock, 4096), kBlock, 0, st>>>(bm, ns, wpr, count, nullptr);
  MG_LAUNCH_CHECK();
  row_offsets_kernel<<<1, kScanWaves * kWave, 0, st>>>(count, ns, off);
  MG_LAUNCH_CHECK();
  b_rank_kernel<<<grid_for(ns, kWavesPerBlock, 4096), kBlock, 0, st>>>(bm, ns, wpr, count, off);
  MG_LAUNCH_CHECK();
}

void launch_heads(hipStream_t st, const HeadJob& a, const HeadJob& b, bool want_bits, uint64_t* words, uint64_t cap,
                  unsigned long long* next) {
  const uint32_t most = std::max(a.n, b.n);
  if (!most) return;
  if (next) {
    constexpr uint32_t kTiles = kHeadLoads * kHeadWaves;
    tile_heads_kernel<kHeadLoads, kHeadWaves><<<dim3(grid_for(most, kTiles, 4096), 2), kHeadWaves * kWave, 0, st>>>(
        a, b, want_bits, words, cap, next);
  } else {
    // Few tiles: a wave each, so that they spread over the chip.
    tile_heads_kernel<1, kWavesPerBlock><<<dim3(grid_for(most, kWavesPerBlock, 8192), 2), kBlock, 0, st>>>(
        a, b, want_bits, words, cap, nullptr);
  }
  MG_LAUNCH_CHECK();
}

void launch_weights(hipStream_t st, const WeightJob& a, const WeightJob& b, uint32_t ns) {
  if ((!a.weight && !b.weight) || !ns) return;
  row_weights_kernel<<<dim3(grid_for(ns, kWindow, 512), 2), kWindow * kWave, 0, st>>>(a, b, ns);
  MG_LAUNCH_CHECK();
}

// Words of an operand's row weights: the rows', their total, and those of kWindow rows each.
uint32_t weight_words(uint32_t ns) { return ns + 1 + (ns + kWindow - 1) / kWindow; }

constexpr uint64_t kSpreadHeads = 65536;
// Room for column words: every one of up to 2^20 tiles, 16 a tile beyond (and no less than that).
uint64_t word_room(uint64_t n) {
  return std::min<uint64_t>(kNoWords - 1ull, std::min<uint64_t>(n * kTile, std::max<uint64_t>(1ull << 26, 16 * n)));
}

// Which kernel a product runs on: tile_product_kernel (true) or product_kernel by windows of C, from the
// numbers of tiles and of the tile pairs that meet; `indexed`: B's index is there already.
// Times in ns, fitted to products of R-MAT and Erdos-Renyi graphs of 2^8 to 2^21 vertices with 1/16 to 16
// edges a vertex and of frontiers with them: by windows 12 us of launches (45 with B's index to build, and 3
// passes over its bitmap), 2.5 a window that holds a tile and 0.02 a pair; by tiles 0.22 a tile, 0.06 a pair
// and twice that for pairs beyond kFewPairsPerTile in each C tile, which come from denser tiles (R-MAT 13, 46
// pairs: 108 us by windows, 122 by tiles; Erdos-Renyi 2^12 vertices, 62 pairs: 60 and 20). Where many meet, one wave
// is at it for long (up to 2.6 us a pair of dense tiles): windows, sooner where they cost no index, and
// for callers that ask for set bits, whose tiles are dense (64 pairs a C tile, all of them recorded: 0.18 ms
// by windows, 0.38 by tiles).
constexpr uint64_t kPairsPerTile = 64, kFewPairsPerTile = 12;
bool by_tiles(uint32_t ns, uint64_t n_a, uint64_t n_c, uint64_t pairs, bool indexed, bool want_bits) {
  if (ns > kBitmapStrips) return true;
  if (pairs > (indexed || want_bits ? kFewPairsPerTile : kPairsPerTile) * n_c) return false;
  const double strip_windows = static_cast<double>((ns + kWindow - 1) / kWindow);
  const double slots = std::max(1.0, std::min<double>(ns, static_cast<double>(n_a)) * strip_windows);
  const double windows = -slots * std::expm1(-static_cast<double>(n_c) / slots);  // tiles spread evenly
  const double index = indexed ? 12e3 : 45e3 + 0.01 * ns * ((ns + 63) / 64);
  const double few = static_cast<double>(std::min(pairs, kFewPairsPerTile * n_c)), all = static_cast<double>(pairs);
  return 0.22 * static_cast<double>(n_c) + 0.06 * few + 0.12 * (all - few) < index + 2.5 * windows + 0.02 * all;
}

}  // namespace

bool prepared(const mg_tiled_matrix* m) { return m->prep_version == m->version && m->prep_head.get(); }

void prepare_operand(mg_context* ctx, mg_tiled_matrix* m, uint64_t used_columns) {
  hipStream_t st = ctx->stream;
  const uint32_t n = m->n_nz_tile, ns = m->n_strips;
  const bool bitmap = ns <= kBitmapStrips;
  const uint32_t wpr = (ns + 63) / 64;
  const uint64_t bm = bitmap ? 2ull * ns * wpr : 0;  // u64 words
  m->prep_head.alloc(2ull * std::max<uint32_t>(1, n));
  StreamBuf<unsigned long long> next(1, st);
  clear_words_kernel<<<1, kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(next.get()), 1);
  MG_LAUNCH_CHECK();
  StreamBuf<uint8_t> used(n, st);
  m->prep_weight.alloc(weight_words(ns));
  clear_u32(st, m->prep_weight.get(), weight_words(ns));
  HeadJob as_a{m->data.get(), n, {}, reinterpret_cast<TileHead*>(m->prep_head.get()), nullptr, nullptr,
               used.get(), 0};
  HeadJob as_b{};
  if (bitmap) {
    m->prep_right_head.alloc(2ull * std::max<uint32_t>(1, n));
    m->prep_bitmap.alloc(std::max<uint64_t>(1, bm));
    m->prep_index.alloc(ns + 1ull + n);
    StreamBuf<uint32_t> count(ns, st);
    BitmapWord* const words = reinterpret_cast<BitmapWord*>(m->prep_bitmap.get());
    launch_right_index(st, m, words, m->prep_index.get(), count.get());
    as_b = as_a;
    as_b.where = PositionMap{m->row_idx.get(), m->col_idx.get(), words, wpr};
    as_b.head_by_tile = as_a.head;
    as_b.head = reinterpret_cast<TileHead*>(m->prep_right_head.get());
    as_b.tile = m->prep_index.get() + ns + 1;
    as_a.n = 0;
  }
  // Last, as many column words as the tiles have, or, without memory for them (or 32-bit places), none:
  // the products then make them from the tiles.
  uint64_t room = used_columns < kNoWords ? used_columns : 0;
  try {
    m->prep_words.alloc(std::max<uint64_t>(1, room));
  } catch (const Failure& e) {
    if (e.code != MG_ERR_OOM || !room) throw;
    room = 0;
    m->prep_words.alloc(1);
  }
  launch_heads(st, as_a, as_b, true, m->prep_words.get(), room, next.get());
  launch_weights(st, WeightJob{used.get(), m->offset_row.get(), m->prep_weight.get()}, WeightJob{}, ns);
}

void product_inputs(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, const ProductTiles& c,
                    bool want_bits, bool want_words, uint64_t pairs, ProductInputs& P, const RightIndex& known) {
  hipStream_t st = ctx->stream;
  const uint32_t ns = a->n_strips, wpr = (ns + 63) / 64;
  const bool pa = prepared(a), pb = prepared(bt), same = a == bt;
  // Unknown: as many as there are where the tiles spread evenly.
  P.pairs = pairs ? pairs : static_cast<uint64_t>(a->n_nz_tile) * bt->n_nz_tile / std::max(1u, ns);
  const bool bitmap = !by_tiles(ns, a->n_nz_tile, c.n_c, P.pairs, pb || known.bm, want_bits);
  const uint64_t na = pa ? 0 : a->n_nz_tile, nb = pb ? 0 : bt->n_nz_tile;
  const bool index_b = bitmap && !pb;
  const uint64_t bm = index_b && !known.bm ? 2ull * ns * wpr : 0;  // u64 words
  // Cleared: counters (column words taken; windows) and the weights. No windows or weights by tiles.
  const uint64_t weights = !bitmap || (pa && pb) ? 0 : 2ull * weight_words(ns);
  const uint64_t clear = (2 + (weights + 1) / 2 + 1) & ~1ull;
  const uint64_t heads_at = clear + bm, windows_at = heads_at + 2 * (na + nb), words_at = windows_at + (bitmap ? 4ull * c.n_c : 0);
  const uint64_t index32 = index_b ? 2ull * ns + 1 + nb : 0;  // row pointer, scratch, tiles by position
  const uint64_t u32s = index32 + (bitmap ? (na + nb + 3) / 4 : 0);  // then the tiles' columns in use (u8)
  const uint64_t n_heads = same && !pa ? nb : na + nb;
  uint64_t room = want_words ? word_room(n_heads) : 0;
  uint64_t* base = nullptr;
  try {
    base = ctx_scratch(ctx, words_at + room + (u32s + 1) / 2);
  } catch (const std::exception&) {
    // No memory for the column words: the product makes them from the tiles (wave_transpose).
    if (!room) throw;
    room = 0;
    base = ctx_scratch(ctx, words_at + (u32s + 1) / 2);
  }
  unsigned long long* const next = reinterpret_cast<unsigned long long*>(base);
  uint32_t* const weight = reinterpret_cast<uint32_t*>(base + 2);
  uint32_t* const weight2 = weight + weight_words(ns);
  TileHead* const head_a = reinterpret_cast<TileHead*>(base + heads_at);
  TileHead* const head_b = head_a + na;
  P.n_strips = ns;
  P.c = c;
  P.n_windows = reinterpret_cast<uint32_t*>(next + 1);
  P.windows = reinterpret_cast<Window*>(base + windows_at);
  uint64_t* const words = base + words_at;
  uint32_t* const at32 = reinterpret_cast<uint32_t*>(words + room);
  // By tiles, few heads: 64 words a tile (32 MiB here) need no counter, so that two launches are all.
  const bool spread = !bitmap && n_heads <= kSpreadHeads && room == n_heads * kTile;
  if (bitmap || (n_heads && !spread)) {
    clear_words_kernel<<<grid_for(clear, kBlock, 4096), kBlock, 0, st>>>(base, clear);
    MG_LAUNCH_CHECK();
  }
  uint8_t* const used = reinterpret_cast<uint8_t*>(at32 + index32);
  HeadJob job_a{a->data.get(), static_cast<uint32_t>(na), {}, head_a, nullptr, nullptr, bitmap ? used : nullptr,
                static_cast<uint32_t>(nb * kTile)};
  HeadJob job_b{bt->data.get(), static_cast<uint32_t>(nb), {}, head_b, nullptr, nullptr, bitmap ? used + na : nullptr, 0};
  if (index_b) {
    P.b.bm = known.bm;
    P.b.off = known.off;
    if (!known.bm) {
      BitmapWord* const words_b = reinterpret_cast<BitmapWord*>(base + clear);
      launch_right_index(st, bt, words_b, at32, at32 + ns + 1);
      P.b.bm = words_b;
      P.b.off = at32;
    }
    job_b.where = PositionMap{bt->row_idx.get(), bt->col_idx.get(), P.b.bm, wpr};
    job_b.tile = at32 + 2ull * ns + 1;
    P.b.tile = job_b.tile;
  }
  if (same && !pa) {  // one pass makes both operands' heads
    job_b.head_by_tile = bitmap ? head_a : nullptr;
    job_a.n = 0;
  }
  launch_heads(st, job_a, job_b, want_bits, words, room, spread ? nullptr : next);
  if (bitmap && c.n_c) {
    launch_weights(st, pa || same ? WeightJob{} : WeightJob{used, a->offset_row.get(), weight},
                   pb ? WeightJob{} : WeightJob{used + na, bt->offset_row.get(), weight2}, ns);
    const uint32_t* const weight_b = pb ? bt->prep_weight.get() : weight2;
    const uint32_t* const weight_a = pa ? a->prep_weight.get() : same ? weight_b : weight;
    windows_kernel<<<grid_for(c.n_c, kScanWaves * kWave, 1024), kScanWaves * kWave, 0, st>>>(c, ns, a->offset_row.get(), weight_a, weight_b,
                                                                      weight_b + ns + 1, P.windows, P.n_windows);
    MG_LAUNCH_CHECK();
  }
  P.a = {same && !bitmap ? head_b : head_a, words, a->data.get(), a->offset_row.get(), a->col_idx.get()};
  if (pa) {
    P.a.head = reinterpret_cast<const TileHead*>(a->prep_head.get());
    P.a.words = a->prep_words.get();
  }
  P.b.head = head_b;
  P.b.words = words;
  P.b.data = bt->data.get();
  P.b.bt_off = bt->offset_row.get();
  P.b.bt_col = bt->col_idx.get();
  if (pb) {
    P.b.words = bt->prep_words.get();
    P.b.head = reinterpret_cast<const TileHead*>(bt->prep_head.get());
    if (bitmap) {
      P.b.head = reinterpret_cast<const TileHead*>(bt->prep_right_head.get());
      P.b.bm = reinterpret_cast<const BitmapWord*>(bt->prep_bitmap.get());
      P.b.off = bt->prep_index.get();
      P.b.tile = P.b.off + ns + 1;
    }
  }
}

RightIndex right_index(mg_context* ctx, const mg_tiled_matrix* bt, StreamBuf<uint64_t>& mem) {
  if (prepared(bt)) return {reinterpret_cast<const BitmapWord*>(bt->prep_bitmap.get()), bt->prep_index.get()};
  const uint32_t ns = bt->n_strips;
  const uint64_t words = 2ull * ns * ((ns + 63) / 64);
  mem.alloc(words + ns + 1, ctx->stream);  // then the row pointer and scratch
  BitmapWord* const bm = reinterpret_cast<BitmapWord*>(mem.get());
  uint32_t* const off = reinterpret_cast<uint32_t*>(mem.get() + words);
  launch_right_index(ctx->stream, bt, bm, off, off + ns + 1);
  return {bm, off};
}

void symbolic_rows(mg_context* ctx, const mg_tiled_matrix* a, const RightIndex& b, const SymbolicRows& S) {
  hipStream_t st = ctx->stream;
  const uint32_t ns = a->n_strips, wpr = (ns + 63) / 64;
  clear_u32(st, S.ref, ns);
  if (ns) {
    union_rows_kernel<<<grid_for(ns, 1, 16384), kUnionWaves * kWave, 0, st>>>(a->offset_row.get(), a->col_idx.get(), b.bm,
                                                                             b.off, ns, wpr, S);
    MG_LAUNCH_CHECK();
  }
  symbolic_totals_kernel<<<1, kScanWaves * kWave, 0, st>>>(S, b.off, ns);
  MG_LAUNCH_CHECK();
}

void symbolic_emit(mg_context* ctx, uint32_t n_strips, const SymbolicRows& S, uint32_t* row_c, uint32_t* col_c) {
  const uint32_t wpr = (n_strips + 63) / 64;
  const uint64_t waves = static_cast<uint64_t>(n_strips) * ((wpr + kWave - 1) / kWave);
  symbolic_emit_kernel<<<grid_for(waves, kWavesPerBlock, 16384), kBlock, 0, ctx->stream>>>(S, n_strips, wpr, row_c, col_c);
  MG_LAUNCH_CHECK();
}

void run_product(mg_context* ctx, const ProductInputs& P, int out_mode, const ProductOut& out) {
  switch (out_mode) {
    case kOutStruct: launch_product<false, kOutStruct>(ctx, P, out, HeavyRecord{}); break;
    case kOutAppend: launch_product<false, kOutAppend>(ctx, P, out, HeavyRecord{}); break;
    case kOutFlag: launch_product<false, kOutFlag>(ctx, P, out, HeavyRecord{}); break;
    case kOutPos: launch_product<false, kOutPos>(ctx, P, out, HeavyRecord{}); break;
    case kOutRest: launch_product<false, kOutRest>(ctx, P, out, HeavyRecord{}); break;
    default: fail(MG_ERR_INTERNAL, "run_product: output mode");
  }
}

namespace {
void right_row_sums(mg_context* ctx, const mg_tiled_matrix* bt, const ProductInputs& P, uint32_t min_bits, bool count,
                    unsigned long long* out) {
  hipStream_t st = ctx->stream;
  if (!P.n_strips) return;
  if (P.b.bm) {
    row_sum_kernel<<<grid_for(P.n_strips, kWavesPerBlock, 4096), kBlock, 0, st>>>(P.b, P.n_strips, min_bits, count, out);
    MG_LAUNCH_CHECK();
    return;
  }
  clear_words_kernel<<<grid_for(P.n_strips, kBlock, 4096), kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(out), P.n_strips);
  MG_LAUNCH_CHECK();
  tile_sum_kernel<<<grid_for(bt->n_nz_tile, kBlock, 4096), kBlock, 0, st>>>(P.b, bt->n_nz_tile, min_bits, count, out);
  MG_LAUNCH_CHECK();
}
}  // namespace

void right_row_bits(mg_context* ctx, const mg_tiled_matrix* bt, const ProductInputs& P, unsigned long long* out) {
  right_row_sums(ctx, bt, P, 0, false, out);
}

uint64_t run_product_dense(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                           const ProductInputs& P, uint32_t min_bits, uint64_t* data_c) {
  hipStream_t st = ctx->stream;
  ProductOut out{};
  out.data = data_c;
  // The structural pairs of two heavy tiles: what the record may hold at most.
  uint64_t most = 0;
  if (a->n_nz_tile && bt->n_nz_tile) {
    StreamBuf<unsigned long long> count(P.n_strips + 1ull, st);
    unsigned long long* const total = count.get() + P.n_strips;
    right_row_sums(ctx, bt, P, min_bits, true, count.get());
    clear_words_kernel<<<1, kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(total), 1);
    MG_LAUNCH_CHECK();
    heavy_pairs_kernel<<<grid_for(a->n_nz_tile, kBlock, 1024), kBlock, 0, st>>>(P.a, a->n_nz_tile, min_bits, count.get(),
                                                                               total);
    MG_LAUNCH_CHECK();
    unsigned long long h = 0;
    read_words(ctx, {total, &h, sizeof(h)});
    most = h;
  }
  MG_REQUIRE(most < (1ull << 31), "mg_multiply_numeric_dense: more than 2^31 dense tile pairs");
  if (!P.c.n_c) return 0;
  if (!most) {
    launch_product<false, kOutStruct>(ctx, P, out, HeavyRecord{});
    return 0;
  }
  const uint32_t part = static_cast<uint32_t>((most + kHeavyParts - 1) / kHeavyParts);
  StreamBuf<HeavyPair> found(static_cast<uint64_t>(part) * kHeavyParts, st);
  constexpr uint32_t kCounters = kHeavyParts * kPartStride;
  StreamBuf<unsigned long long> taken(kCounters + (P.c.n_c + 1ull) / 2, st);  // then the C tiles' counts (u32)
  uint32_t* const count = reinterpret_cast<uint32_t*>(taken.get() + kCounters);
  clear_words_kernel<<<grid_for(taken.size(), kBlock, 4096), kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(taken.get()),
                                                                              taken.size());
  MG_LAUNCH_CHECK();
  launch_product<true, kOutStruct>(ctx, P, out, HeavyRecord{found.get(), count, taken.get(), part, min_bits});
  StreamBuf<uint32_t> base(P.c.n_c + 1ull, st);
  exclusive_scan_u32(ctx, count, base.get(), P.c.n_c);
  uint32_t n = 0;
  read_words(ctx, {base.get() + P.c.n_c, &n, sizeof(n)});
  MG_REQUIRE(n <= most, "mg_multiply_numeric_dense: more dense pairs recorded than counted");
  if (!n) return 0;
  StreamBuf<uint2> pairs(n, st);
  const uint64_t max_tasks = std::min<uint64_t>(n, static_cast<uint64_t>(P.c.n_c) + n / kTaskPairs);
  StreamBuf<DenseTask> tasks(max_tasks, st);
  StreamBuf<uint32_t> n_tasks(2, st);
  clear_words_kernel<<<1, kBlock, 0, st>>>(reinterpret_cast<uint64_t*>(n_tasks.get()), 1);
  MG_LAUNCH_CHECK();
  heavy_scatter_kernel<<<dim3(static_cast<uint32_t>(grid_for(part, kBlock, 64)), kHeavyParts), kBlock, 0, st>>>(
      found.get(), taken.get(), part, base.get(), pairs.get());
  MG_LAUNCH_CHECK();
  heavy_tasks_kernel<<<grid_for(P.c.n_c, kBlock, 4096), kBlock, 0, st>>>(base.get(), P.c.n_c, tasks.get(), n_tasks.get());
  MG_LAUNCH_CHECK();
  dense_contract_kernel<<<grid_for(max_tasks, kWavesPerBlock, 16384), kBlock, 0, st>>>(
      tasks.get(), n_tasks.get(), pairs.get(), a->data.get(), bt->data.get(), data_c);
  MG_LAUNCH_CHECK();
  return n;
}

}  // namespace mgamd
