// General bit-tiled Boolean product C = A * B with B supplied transposed (Bt):
//   - layout-level entry points of the reference wrapper (MatrixBitAnd,
//     InitBitTiledMatrixMetadataByLayoutMatrix, FillTiles);
//   - the handle-based symbolic pass (structural tile set of C, tile-product count)
//     and numeric pass.
// Tile product on a wave64: lane r holds L[r] (row r of the left tile), lane c holds
// Rt[c] (row c of the transposed right tile); output row r bit c = (L[r] & Rt[c]) != 0.
// The loop runs only over non-zero Rt rows (wave ballot), so sparse tiles cost a few
// instructions; dense tiles (64 non-zero rows) take 64 iterations. The handle-based numeric
// passes are in mg_product.hip, except the allocation-free one: it multiplies pairs of tiles with at
// most 10 bits from their entry lists, one pair per lane (fill_tiles_payload_kernel), and keeps
// the wave product for denser tiles.
#include <mutex>
#include <string>

#include "mg_device.hpp"
#include "mg_internal.hpp"
#include "mg_product.hpp"

namespace mgamd {
namespace {

constexpr int kBlock = 256;
constexpr int kWavesPerBlock = kBlock / kWave;
#ifndef MG_PAIR_BATCH
#define MG_PAIR_BATCH 4
#endif
constexpr int kPairBatch = MG_PAIR_BATCH;  // tile pairs whose loads fill_tiles_kernel issues together
constexpr uint32_t kRowFeatures = MG_ROW_FEATURES;  // features per C row (mg_multiply_row_features)

__device__ inline uint64_t tile_product(uint64_t l_row, uint64_t rt_row) {
  uint64_t nz = ballot(rt_row != 0);
  if (ballot(l_row != 0) == 0) return 0;
  uint64_t out = 0;
  while (nz) {
    const int c = __ffsll(static_cast<unsigned long long>(nz)) - 1;
    nz &= nz - 1;
    const uint64_t w = read_lane(rt_row, c);
    out |= static_cast<uint64_t>((l_row & w) != 0) << c;
  }
  return out;
}

// Index of key in sorted a[lo, hi), or -1.
__device__ inline int64_t find_sorted(const uint32_t* __restrict__ a, uint32_t lo, uint32_t hi, uint32_t key) {
  uint32_t l = lo, h = hi;
  while (l < h) {
    const uint32_t mid = l + ((h - l) >> 1);
    if (a[mid] < key) l = mid + 1; else h = mid;
  }
  return (l < hi && a[l] == key) ? static_cast<int64_t>(l) : -1;
}

// One wave per tile of C: intersect A.row(x) with Bt.row(y) on the tile column,
// OR the tile products, OR the result into data_c (FillTiles semantics,
// core/task/gpu_task/kernel/matrix_operations.cu:318-366 with the intended
// offsets of B at :356 and the intended 64x64 product of :212-233). Whole-tile products on
// the vector ALUs (the layer-1 entry point, whose operands are raw tile arrays).
__global__ void __launch_bounds__(kBlock) fill_tiles_kernel(
    uint32_t n_c, const uint32_t* __restrict__ off_a, const uint32_t* __restrict__ off_bt,
    const uint32_t* __restrict__ row_c, const uint32_t* __restrict__ col_c, const uint32_t* __restrict__ col_a,
    const uint32_t* __restrict__ col_bt, const uint64_t* __restrict__ data_a, const uint64_t* __restrict__ data_bt,
    uint64_t* __restrict__ data_c) {
  const uint32_t lane = lane_id();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t i = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); i < n_c; i += n_waves) {
    const uint32_t x = row_c[i];
    const uint32_t y = col_c[i];
    const uint32_t a0 = off_a[x], a1 = off_a[x + 1];
    const uint32_t b0 = off_bt[y], b1 = off_bt[y + 1];
    const bool a_short = (a1 - a0) <= (b1 - b0);
    const uint32_t s0 = a_short ? a0 : b0, s1 = a_short ? a1 : b1;
    const uint32_t l0 = a_short ? b0 : a0, l1 = a_short ? b1 : a1;
    const uint32_t* s_col = a_short ? col_a : col_bt;
    const uint32_t* l_col = a_short ? col_bt : col_a;
    uint64_t acc = 0;
    for (uint32_t base = s0; base < s1; base += kWave) {
      const uint32_t j = base + lane;
      int64_t pos = -1;
      if (j < s1) pos = find_sorted(l_col, l0, l1, s_col[j]);
      uint64_t hit = ballot(pos >= 0);
      // kPairBatch matching pairs at a time, all their tile loads issued before the first
      // product, so a wave waits once per batch instead of once per pair.
      while (hit) {
        uint64_t l_row[kPairBatch], rt_row[kPairBatch];
        uint32_t n_pairs = 0;  // wave-uniform
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          l_row[q] = 0;
          rt_row[q] = 0;
          if (hit) {
            const int k = __ffsll(static_cast<unsigned long long>(hit)) - 1;
            hit &= hit - 1;
            const uint32_t js = base + k;
            const uint32_t jl = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(pos), k));
            const uint64_t ia = a_short ? js : jl;
            const uint64_t ib = a_short ? jl : js;
            l_row[q] = data_a[ia * kTile + lane];
            rt_row[q] = data_bt[ib * kTile + lane];
            ++n_pairs;
          }
        }
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q)
          if (static_cast<uint32_t>(q) < n_pairs) acc |= tile_product(l_row[q], rt_row[q]);
      }
    }
    uint64_t* dst = data_c + static_cast<uint64_t>(i) * kTile + lane;
    if (acc) *dst |= acc;
  }
}

// Product of two dense tiles through their common inner indices (`common`: the columns in use
// in both, wave-uniform): for each such j, the rows r with L(r, j) set receive the columns c
// with Rt(c, j) set (a ballot). The loop runs over the j the two tiles share, where
// tile_product runs over every non-zero row of Rt; on R-MAT tiles above kWideMax bits that
// is about half the steps.
__device__ inline uint64_t tile_product_common(uint64_t l_row, uint64_t rt_row, uint64_t common) {
  uint64_t out = 0;
  for (; common; common &= common - 1) {
    const int j = __ffsll(static_cast<unsigned long long>(common)) - 1;
    const uint64_t cols = ballot((rt_row >> j) & 1);
    if ((l_row >> j) & 1) out |= cols;
  }
  return out;
}

// 16-byte compact payload of a tile with at most kWideMax set bits: entry i = (row << 6) |
// column in bits 12(i % 5).. of word i / 5, the entry count in bits 60..63 of word 1; count
// kWideDense marks a denser tile, whose word 0 then holds the OR of its rows (the columns in use:
// the inner indices j through which it meets the other operand's tiles).
typedef uint64_t WidePayload __attribute__((ext_vector_type(2)));
constexpr uint32_t kWideMax = 10;
constexpr uint32_t kWideDense = 15;

__device__ inline uint32_t wide_count(WidePayload p) { return static_cast<uint32_t>(p.y >> 60); }
__device__ inline uint32_t wide_entry(WidePayload p, uint32_t i) {
  return static_cast<uint32_t>((i < 5 ? p.x : p.y) >> (12 * (i < 5 ? i : i - 5))) & 0xFFFu;
}

// Wide payload of every tile of both operands, one wave per tile (lane r holds row r): tiles
// [0, n_a) of data_a, then the n_bt tiles of data_bt, at the same positions of `payload`. used (may be
// null) gets the tiles' columns in use added up.
__global__ void __launch_bounds__(kBlock) payload_kernel(const uint64_t* __restrict__ data_a, uint32_t n_a,
                                                         const uint64_t* __restrict__ data_bt, uint32_t n_bt,
                                                         WidePayload* __restrict__ payload,
                                                         unsigned long long* __restrict__ used) {
  __shared__ unsigned long long s_used;
  if (threadIdx.x == 0) s_used = 0;
  __syncthreads();
  uint64_t n_used = 0;
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  const uint64_t n_tiles = static_cast<uint64_t>(n_a) + n_bt;
  for (uint64_t i = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); i < n_tiles; i += n_waves) {
    const uint64_t word = i < n_a ? data_a[i * kTile + lane_id()] : data_bt[(i - n_a) * kTile + lane_id()];
    const uint64_t total = wave_sum(__popcll(word));
    WidePayload pl = {0, static_cast<uint64_t>(kWideDense) << 60};
    const uint64_t cols = wave_or(word);
    n_used += static_cast<uint32_t>(__popcll(cols));
    if (total > kWideMax) pl.x = cols;
    if (total <= kWideMax) {
      uint64_t w[2] = {0, 0};
      uint32_t n = 0;
      for (uint64_t m = ballot(word != 0); m; m &= m - 1) {
        const int r = __ffsll(static_cast<unsigned long long>(m)) - 1;
        for (uint64_t wr = read_lane(word, r); wr; wr &= wr - 1) {
          const uint64_t c = static_cast<uint64_t>(__ffsll(static_cast<unsigned long long>(wr)) - 1);
          w[n / 5] |= ((static_cast<uint64_t>(r) << 6) | c) << (12 * (n % 5));
          ++n;
        }
      }
      pl.x = w[0];
      pl.y = w[1] | (static_cast<uint64_t>(n) << 60);
    }
    if (lane_id() == 0) payload[i] = pl;
  }
  if (!used) return;
  if (lane_id() == 0 && n_used) atomicAdd(&s_used, static_cast<unsigned long long>(n_used));
  __syncthreads();
  if (threadIdx.x == 0 && s_used) atomicAdd(used, s_used);
}

// Payloads alone of A's tiles at pl[0, n_a) and of Bt's at pl[n_a, n_a + n_bt) (the allocation-free
// pass); those of a prepared operand are copied.
void launch_payloads(hipStream_t st, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, WidePayload* pl) {
  const uint32_t na = a->n_nz_tile, nb = bt->n_nz_tile;
  const bool pa = prepared(a) && na, pb = prepared(bt) && nb;
  if (pa) MG_HIP(hipMemcpyAsync(pl, a->prep_payload.get(), sizeof(WidePayload) * na, hipMemcpyDeviceToDevice, st));
  if (pb) MG_HIP(hipMemcpyAsync(pl + na, bt->prep_payload.get(), sizeof(WidePayload) * nb, hipMemcpyDeviceToDevice, st));
  const uint32_t ma = pa ? 0 : na, mb = pb ? 0 : nb;
  if (ma + mb == 0) return;
  payload_kernel<<<grid_for(static_cast<uint64_t>(ma) + mb, kWavesPerBlock, 65536), kBlock, 0, st>>>(
      a->data.get(), ma, bt->data.get(), mb, pa ? pl + na : pl, nullptr);
  MG_LAUNCH_CHECK();
}

// fill_tiles_kernel for operands whose tiles are mostly sparse, from their wide payloads
// (pl_a, pl_bt). The intersection gives each lane its own tile pair; a pair of two compact
// tiles is multiplied by that lane alone: every entry (r, j) of the A tile meets every entry
// (c, j) of the Bt tile with the same j and sets bit c of row r in the wave's LDS
// accumulator. Pairs with a denser tile take the full-tile wave product, kPairBatch at a time.
// Only the allocation-free pass runs it: its 16 bytes of scratch per tile hold neither heads nor column
// words (product_kernel takes 119 us where this one takes 518: C = A*A, R-MAT 14).
__global__ void __launch_bounds__(kBlock) fill_tiles_payload_kernel(
    uint32_t n_c, const uint32_t* __restrict__ off_a, const uint32_t* __restrict__ off_bt,
    const uint32_t* __restrict__ row_c, const uint32_t* __restrict__ col_c, const uint32_t* __restrict__ col_a,
    const uint32_t* __restrict__ col_bt, const uint64_t* __restrict__ data_a, const uint64_t* __restrict__ data_bt,
    const WidePayload* __restrict__ pl_a, const WidePayload* __restrict__ pl_bt, uint64_t* __restrict__ data_c) {
  __shared__ unsigned long long s_acc[kWavesPerBlock][kTile];
  const uint32_t lane = lane_id();
  unsigned long long* const acc_l = s_acc[threadIdx.x / kWave];
  acc_l[lane] = 0;
  wave_lds_sync();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t i = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); i < n_c; i += n_waves) {
    const uint32_t x = row_c[i];
    const uint32_t y = col_c[i];
    const uint32_t a0 = off_a[x], a1 = off_a[x + 1];
    const uint32_t b0 = off_bt[y], b1 = off_bt[y + 1];
    const bool a_short = (a1 - a0) <= (b1 - b0);
    const uint32_t s0 = a_short ? a0 : b0, s1 = a_short ? a1 : b1;
    const uint32_t l0 = a_short ? b0 : a0, l1 = a_short ? b1 : a1;
    const uint32_t* s_col = a_short ? col_a : col_bt;
    const uint32_t* l_col = a_short ? col_bt : col_a;
    uint64_t acc = 0;
    for (uint32_t base = s0; base < s1; base += kWave) {
      const uint32_t j = base + lane;
      int64_t pos = -1;
      if (j < s1) pos = find_sorted(l_col, l0, l1, s_col[j]);
      const bool has = pos >= 0;
      const uint32_t ia = has ? (a_short ? j : static_cast<uint32_t>(pos)) : 0u;
      const uint32_t ib = has ? (a_short ? static_cast<uint32_t>(pos) : j) : 0u;
      WidePayload pa = {0, 0}, pb = {0, 0};
      if (has) {
        pa = pl_a[ia];
        pb = pl_bt[ib];
      }
      const uint32_t na = wide_count(pa), nb = wide_count(pb);
      const bool dense = has && (na == kWideDense || nb == kWideDense);
      if (has && !dense) {
        // Only the inner indices j present in both tiles give bits: per common j, the Bt
        // entries' columns are collected into one mask and ORed into the row of every A
        // entry with that j (na + nb steps per common j instead of na * nb comparisons).
        uint64_t jm_a = 0, jm_b = 0;
        for (uint32_t u = 0; u < na; ++u) jm_a |= 1ull << (wide_entry(pa, u) & 63u);
        for (uint32_t v = 0; v < nb; ++v) jm_b |= 1ull << (wide_entry(pb, v) & 63u);
        for (uint64_t common = jm_a & jm_b; common; common &= common - 1) {
          const uint32_t jj = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(common)) - 1);
          uint64_t cols = 0;
          for (uint32_t v = 0; v < nb; ++v) {
            const uint32_t eb = wide_entry(pb, v);
            if ((eb & 63u) == jj) cols |= 1ull << (eb >> 6);
          }
          for (uint32_t u = 0; u < na; ++u) {
            const uint32_t ea = wide_entry(pa, u);
            if ((ea & 63u) == jj) atomicOr(acc_l + (ea >> 6), cols);
          }
        }
      }
      // Pairs with one dense tile: the dense tile's rows (lane = row) against the other tile's
      // entries, kPairBatch pairs' loads at a time. An A entry (r, j) ORs column j of the Bt
      // tile (a ballot over its rows) into row r; a Bt entry (c, j) sets bit c of every row r
      // whose A row has bit j.
      const bool a_dense = na == kWideDense, b_dense = nb == kWideDense;
      for (uint64_t dm = ballot(dense && !a_dense); dm;) {
        uint64_t rt_row[kPairBatch], used[kPairBatch];
        WidePayload ent[kPairBatch];
        uint32_t n_pairs = 0;  // wave-uniform
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          rt_row[q] = 0;
          used[q] = 0;
          ent[q] = WidePayload{0, 0};
          if (dm) {
            const int k = __ffsll(static_cast<unsigned long long>(dm)) - 1;
            dm &= dm - 1;
            const uint64_t kb = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ib), k));
            rt_row[q] = data_bt[kb * kTile + lane];
            ent[q].x = read_lane(pa.x, k);
            ent[q].y = read_lane(pa.y, k);
            used[q] = read_lane(pb.x, k);  // columns in use of the dense Bt tile
            ++n_pairs;
          }
        }
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          if (static_cast<uint32_t>(q) >= n_pairs) continue;
          const uint32_t n = wide_count(ent[q]);
          for (uint32_t u = 0; u < n; ++u) {
            const uint32_t e = wide_entry(ent[q], u);
            if (!((used[q] >> (e & 63u)) & 1)) continue;  // no Bt row has bit j
            const uint64_t col = ballot((rt_row[q] >> (e & 63u)) & 1);
            if (lane == (e >> 6)) acc |= col;
          }
        }
      }
      for (uint64_t dm = ballot(dense && a_dense && !b_dense); dm;) {
        uint64_t l_row[kPairBatch], used[kPairBatch];
        WidePayload ent[kPairBatch];
        uint32_t n_pairs = 0;  // wave-uniform
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          l_row[q] = 0;
          used[q] = 0;
          ent[q] = WidePayload{0, 0};
          if (dm) {
            const int k = __ffsll(static_cast<unsigned long long>(dm)) - 1;
            dm &= dm - 1;
            const uint64_t ka = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ia), k));
            l_row[q] = data_a[ka * kTile + lane];
            ent[q].x = read_lane(pb.x, k);
            ent[q].y = read_lane(pb.y, k);
            used[q] = read_lane(pa.x, k);  // columns in use of the dense A tile
            ++n_pairs;
          }
        }
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          if (static_cast<uint32_t>(q) >= n_pairs) continue;
          const uint32_t n = wide_count(ent[q]);
          for (uint32_t v = 0; v < n; ++v) {
            const uint32_t e = wide_entry(ent[q], v);
            if (!((used[q] >> (e & 63u)) & 1)) continue;  // no A row has bit j
            acc |= ((l_row[q] >> (e & 63u)) & 1ull) << (e >> 6);
          }
        }
      }
      // Both tiles dense: the wave product through the inner indices both tiles use.
      for (uint64_t dm = ballot(dense && a_dense && b_dense); dm;) {
        uint64_t l_row[kPairBatch], rt_row[kPairBatch], common[kPairBatch];
        uint32_t n_pairs = 0;  // wave-uniform
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q) {
          l_row[q] = 0;
          rt_row[q] = 0;
          common[q] = 0;
          if (dm) {
            const int k = __ffsll(static_cast<unsigned long long>(dm)) - 1;
            dm &= dm - 1;
            const uint64_t ka = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ia), k));
            const uint64_t kb = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(ib), k));
            l_row[q] = data_a[ka * kTile + lane];
            rt_row[q] = data_bt[kb * kTile + lane];
            common[q] = read_lane(pa.x, k) & read_lane(pb.x, k);
            ++n_pairs;
          }
        }
#pragma unroll
        for (int q = 0; q < kPairBatch; ++q)
          if (static_cast<uint32_t>(q) < n_pairs) acc |= tile_product_common(l_row[q], rt_row[q], common[q]);
      }
    }
    wave_lds_sync();
    acc |= acc_l[lane];
    acc_l[lane] = 0;
    wave_lds_sync();
    uint64_t* dst = data_c + static_cast<uint64_t>(i) * kTile + lane;
    if (acc) *dst |= acc;
  }
}

// Block-wide exclusive scan of one u32 per thread (kWaves waves).
template <int kWaves>
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* s_tmp, uint32_t* total) {
  const uint32_t lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  uint32_t incl = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), d, kWave));
    if (lane >= static_cast<uint32_t>(d)) incl += o;
  }
  if (lane == kWave - 1) s_tmp[wave] = incl;
  __syncthreads();
  uint32_t base = 0, tot = 0;
  for (int w = 0; w < kWaves; ++w) {
    const uint32_t t = s_tmp[w];
    if (w < static_cast<int>(wave)) base += t;
    tot += t;
  }
  __syncthreads();
  *total = tot;
  return base + incl - v;
}

// len (<= 64) bits of a bit-packed array starting at bit `start`.
__device__ inline uint64_t bit_window(const uint64_t* __restrict__ p, uint64_t start, uint32_t len) {
  const uint64_t w = start >> 6;
  const uint32_t s = static_cast<uint32_t>(start & 63);
  uint64_t v = p[w] >> s;
  if (s != 0 && s + len > 64) v |= p[w + 1] << (64 - s);
  if (len < 64) v &= (1ull << len) - 1;
  return v;
}

// MatrixBitAnd (matrix_operations.cu:256-280), intended semantics: wave per
// (row i of a, 64 rows of b); c bit i*n+j |= any(a row i & b row j).
__global__ void __launch_bounds__(kBlock) bit_and_kernel(const uint64_t* __restrict__ a,
                                                         const uint64_t* __restrict__ b,
                                                         unsigned long long* __restrict__ c, uint32_t m,
                                                         uint32_t k, uint32_t n) {
  const uint32_t lane = lane_id();
  const uint32_t nj = (n + 63) / 64;
  const uint64_t n_tasks = static_cast<uint64_t>(m) * nj;
  const uint64_t n_waves = static_cast<uint64_t>(gridDim.x) * kWavesPerBlock;
  for (uint64_t task = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; task < n_tasks; task += n_waves) {
    const uint32_t i = static_cast<uint32_t>(task / nj);
    const uint32_t jc = static_cast<uint32_t>(task % nj);
    const uint32_t j = jc * 64 + lane;
    bool hit = false;
    if (j < n) {
      for (uint32_t t0 = 0; t0 < k && !hit; t0 += 64) {
        const uint32_t len = (k - t0) < 64 ? (k - t0) : 64;
        const uint64_t wa = bit_window(a, static_cast<uint64_t>(i) * k + t0, len);
        const uint64_t wb = bit_window(b, static_cast<uint64_t>(j) * k + t0, len);
        hit = (wa & wb) != 0;
      }
    }
    const uint64_t mask = ballot(hit);
    if (lane == 0 && mask) {
      const uint64_t start = static_cast<uint64_t>(i) * n + static_cast<uint64_t>(jc) * 64;
      const uint32_t s = static_cast<uint32_t>(start & 63);
      atomicOr(c + (start >> 6), static_cast<unsigned long long>(mask << s));
      if (s != 0 && (mask >> (64 - s)) != 0)
        atomicOr(c + (start >> 6) + 1, static_cast<unsigned long long>(mask >> (64 - s)));
    }
  }
}

// Layout row counts: cnt[x] = set bits in row x of an n x n layout.
__global__ void __launch_bounds__(kBlock) layout_row_count_kernel(const uint64_t* __restrict__ layout,
                                                                  uint32_t n, uint32_t* __restrict__ cnt) {
  const uint32_t lane = lane_id();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t x = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; x < n; x += n_waves) {
    uint64_t c = 0;
    for (uint32_t y0 = lane * 64; y0 < n; y0 += 64 * kWave) {
      const uint32_t len = (n - y0) < 64 ? (n - y0) : 64;
      c += __popcll(bit_window(layout, static_cast<uint64_t>(x) * n + y0, len));
    }
    c = wave_sum(c);
    if (lane == 0) cnt[x] = static_cast<uint32_t>(c);
  }
}

// Rank emission: (row_idx, col_idx)[rank] for every set bit, rank = row-major order.
__global__ void __launch_bounds__(kBlock) layout_emit_kernel(const uint64_t* __restrict__ layout, uint32_t n,
                                                             const uint32_t* __restrict__ row_start,
                                                             uint32_t* __restrict__ row_idx,
                                                             uint32_t* __restrict__ col_idx) {
  const uint32_t lane = lane_id();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t x = blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; x < n; x += n_waves) {
    uint32_t rank = row_start[x];
    for (uint32_t y0 = 0; y0 < n; y0 += 64) {
      const uint32_t len = (n - y0) < 64 ? (n - y0) : 64;
      const uint64_t w = bit_window(layout, static_cast<uint64_t>(x) * n + y0, len);  // uniform
      if (w == 0) continue;
      if ((w >> lane) & 1) {
        const uint32_t r = rank + __popcll(w & ((1ull << lane) - 1));
        row_idx[r] = x;
        col_idx[r] = y0 + lane;
      }
      rank += __popcll(w);
    }
  }
}

__global__ void add_counts_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src, uint32_t n) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += static_cast<uint64_t>(gridDim.x) * blockDim.x) dst[i] += src[i];
}

// --- symbolic pass ---------------------------------------------------------

// Row form of B from Bt: histogram of Bt's column index (entries [0, n_bt)); in the same
// launch, the rows of B that A references (its column index, entries [n_bt, n_bt + n_a)).
__global__ void col_hist_mark_kernel(const uint32_t* __restrict__ col_bt, uint32_t n_bt,
                                     const uint32_t* __restrict__ col_a, uint32_t n_a, uint32_t* __restrict__ hist,
                                     uint32_t* __restrict__ ref) {
  const uint64_t n = static_cast<uint64_t>(n_bt) + n_a;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    if (i < n_bt)
      atomicAdd(hist + col_bt[i], 1u);
    else
      ref[col_a[i - n_bt]] = 1u;
  }
}
__global__ void col_scatter_kernel(const uint32_t* __restrict__ row, const uint32_t* __restrict__ col, uint32_t n,
                                   const uint32_t* __restrict__ start, uint32_t* __restrict__ cursor,
                                   uint32_t* __restrict__ out) {
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const uint32_t t = col[i];
    out[start[t] + atomicAdd(cursor + t, 1u)] = row[i];
  }
}

// Per output row x: union over t in A.row(x) of B.row(t) in an LDS bitmap.
// EMIT = false: count[x] = |union|, tp[x] = sum |B.row(t)|; with `sums`, the block's totals are
// added to sums[0] (tile products), sums[1] (tiles of the B rows that A references, ref[x]:
// row x of B, as x runs over the strips) and sums[2] (C tiles).
// EMIT = true : write the union as ascending col_idx at off_c[x], row_idx = x.
// Grids wider than kBitmapStrips only (structural_pass), where no bitmap of B is kept.
// BLOCK threads per row (kRowBlock = 1024: a heavy row, such as a dense frontier's tile row
// against thousands of B rows, is the whole pass when few rows carry the work; 1024 threads
// took the 3-hop density-mixed product walk's symbolic passes from 39 to 16 ms and C = A*A of
// R-MAT 14 from 0.64 to 0.62 ms, with the two-hop of R-MAT 18 unchanged).
constexpr int kRowBlock = 1024;
template <bool EMIT, int BLOCK = kRowBlock>
__global__ void __launch_bounds__(BLOCK) symbolic_row_kernel(
    uint32_t n_strips, const uint32_t* __restrict__ off_a, const uint32_t* __restrict__ col_a,
    const uint32_t* __restrict__ off_b, const uint32_t* __restrict__ col_b, uint32_t* __restrict__ count,
    unsigned long long* __restrict__ tp, const uint32_t* __restrict__ off_c, uint32_t* __restrict__ row_c,
    uint32_t* __restrict__ col_c, const uint32_t* __restrict__ ref = nullptr,
    unsigned long long* __restrict__ sums = nullptr) {
  constexpr int kWaves = BLOCK / kWave;
  extern __shared__ uint64_t s_bm[];
  __shared__ uint32_t s_tmp[kWaves];
  __shared__ unsigned long long s_tp;
  const uint32_t n_words = (n_strips + 63) / 64;
  const uint32_t lane = lane_id();
  const uint32_t wave = threadIdx.x / kWave;
  uint64_t blk_tp = 0, blk_used = 0, blk_c = 0;  // thread 0's totals over the block's rows
  for (uint32_t x = blockIdx.x; x < n_strips; x += gridDim.x) {
    for (uint32_t w = threadIdx.x; w < n_words; w += BLOCK) s_bm[w] = 0;
    if (threadIdx.x == 0) s_tp = 0;
    __syncthreads();
    const uint32_t a0 = off_a[x], a1 = off_a[x + 1];
    uint64_t my_tp = 0;
    for (uint32_t k = a0 + wave; k < a1; k += kWaves) {
      const uint32_t t = col_a[k];
      const uint32_t r0 = off_b[t], r1 = off_b[t + 1];
      my_tp += r1 - r0;
      for (uint32_t j = r0 + lane; j < r1; j += kWave) {
        const uint32_t y = col_b[j];
        atomicOr(reinterpret_cast<unsigned long long*>(s_bm + (y >> 6)), 1ull << (y & 63));
      }
    }
    if (!EMIT && lane == 0 && my_tp) atomicAdd(&s_tp, static_cast<unsigned long long>(my_tp));
    __syncthreads();
    // Contiguous word range per thread so emitted columns come out ascending.
    const uint32_t per = (n_words + BLOCK - 1) / BLOCK;
    const uint32_t w0 = threadIdx.x * per;
    const uint32_t w1 = (w0 + per < n_words) ? w0 + per : n_words;
    uint32_t c = 0;
    for (uint32_t w = w0; w < w1; ++w) c += __popcll(s_bm[w]);
    uint32_t total = 0;
    const uint32_t before = block_exclusive_scan<kWaves>(c, s_tmp, &total);
    if (!EMIT) {
      if (threadIdx.x == 0) {
        count[x] = total;
        tp[x] = s_tp;
        blk_tp += s_tp;
        blk_c += total;
        if (ref && ref[x]) blk_used += off_b[x + 1] - off_b[x];
      }
    } else {
      uint32_t pos = off_c[x] + before;
      for (uint32_t w = w0; w < w1; ++w) {
        uint64_t bits = s_bm[w];
        while (bits) {
          const int b = __ffsll(static_cast<unsigned long long>(bits)) - 1;
          bits &= bits - 1;
          row_c[pos] = x;
          col_c[pos] = w * 64 + b;
          ++pos;
        }
      }
    }
    __syncthreads();
  }
  if (!EMIT && sums && threadIdx.x == 0) {
    if (blk_tp) atomicAdd(sums, static_cast<unsigned long long>(blk_tp));
    if (blk_used) atomicAdd(sums + 1, static_cast<unsigned long long>(blk_used));
    if (blk_c) atomicAdd(sums + 2, static_cast<unsigned long long>(blk_c));
  }
}

constexpr uint32_t kMaxLdsBitmapWords = 8192;  // 64 KiB: n_strips <= 524288

void launch_fill_tiles(hipStream_t s, uint32_t n_c, const uint32_t* off_a, const uint32_t* off_bt,
                       const uint32_t* row_c, const uint32_t* col_c, const uint32_t* col_a,
                       const uint32_t* col_bt, const uint64_t* data_a, const uint64_t* data_bt,
                       uint64_t* data_c) {
  if (n_c == 0) return;
  fill_tiles_kernel<<<grid_for(n_c, kWavesPerBlock, 65536), kBlock, 0, s>>>(n_c, off_a, off_bt, row_c, col_c,
                                                                            col_a, col_bt, data_a, data_bt, data_c);
  MG_LAUNCH_CHECK();
}

// Words of payload scratch of the allocation-free pass.
size_t payload_words(const mg_tiled_matrix* a, const mg_tiled_matrix* bt) {
  return 2 * (static_cast<size_t>(a->n_nz_tile) + bt->n_nz_tile + 1);
}

// --- structural pass shared by the handle-level products ----------------------
// Row form of B (B.row(t) = { y : Bt(y,t) present }), per-row structural counts and tile
// products of C = A*B, C's row pointer, and the totals.
struct Structural {
  uint32_t n = 0;  // n_strips
  StreamBuf<uint64_t> mem;      // rows: counts, tile products, row pointer, totals
  SymbolicRows rows{};
  StreamBuf<uint64_t> index;    // by bitmaps: B's
  RightIndex b{};
  StreamBuf<uint32_t> off_b, col_b;  // by lists: B's rows
  uint64_t n_c = 0, tile_products = 0, right_used = 0;
};

void structural_pass(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, Structural& S,
                     const char* who) {
  MG_REQUIRE(a->n_strips == bt->n_strips, std::string(who) + ": operands differ in n_strips");
  const uint32_t n = a->n_strips;
  const uint32_t n_words = (n + 63) / 64;
  if (n_words > kMaxLdsBitmapWords) fail(MG_ERR_UNSUPPORTED, std::string(who) + ": n_strips > 524288 not supported");
  hipStream_t s = ctx->stream;
  S.n = n;
  // Bitmaps wherever a grid has them: faster than the lists from 16 tiles to 2 M, on 64 to 16384 strips,
  // also where a row of B has one tile per 32 words (7.9 K tiles on 4096 strips: 163 us, by lists
  // 243; 1.0 M: 2.1 ms, 2.9, most of it the clearing of C).
  const bool bitmaps = n <= kBitmapStrips;
  // u64: totals (tile products, right tiles used, C tiles), tile products of the rows, C's bitmap;
  // u32: referenced-row flags, counts, row pointer; by lists also histogram and scatter cursors.
  const uint64_t c_bits = bitmaps ? static_cast<uint64_t>(n) * n_words : 0;
  S.mem.alloc(3 + n + c_bits + (5ull * n + 2) / 2, s);
  S.rows.sums = reinterpret_cast<unsigned long long*>(S.mem.get());
  S.rows.tp = S.rows.sums + 3;
  S.rows.c_bits = S.mem.get() + 3 + n;
  S.rows.ref = reinterpret_cast<uint32_t*>(S.rows.c_bits + c_bits);
  S.rows.cnt = S.rows.ref + n;
  S.rows.off_c = S.rows.cnt + n;
  if (bitmaps) {
    S.b = right_index(ctx, bt, S.index);
    symbolic_rows(ctx, a, S.b, S.rows);
  } else {
    uint32_t* const hist = S.rows.off_c + n + 1;
    uint32_t* const cursor = hist + n;
    MG_HIP(hipMemsetAsync(S.mem.get(), 0, S.mem.bytes(), s));
    S.off_b.alloc(n + 1ull, s);
    S.col_b.alloc(bt->n_nz_tile, s);
    if (bt->n_nz_tile || a->n_nz_tile) {
      col_hist_mark_kernel<<<grid_for(static_cast<uint64_t>(bt->n_nz_tile) + a->n_nz_tile, 256), 256, 0, s>>>(
          bt->col_idx.get(), bt->n_nz_tile, a->col_idx.get(), a->n_nz_tile, hist, S.rows.ref);
      MG_LAUNCH_CHECK();
    }
    exclusive_scan_u32(ctx, hist, S.off_b.get(), n);
    if (bt->n_nz_tile) {
      col_scatter_kernel<<<grid_for(bt->n_nz_tile, 256), 256, 0, s>>>(bt->row_idx.get(), bt->col_idx.get(),
                                                                      bt->n_nz_tile, S.off_b.get(), cursor,
                                                                      S.col_b.get());
      MG_LAUNCH_CHECK();
    }
    const size_t lds = sizeof(uint64_t) * n_words;
    const unsigned grid = grid_for(n, 1, 16384);
    // The row kernel also adds up the totals. C's tile index is 32-bit (the reference's
    // n_nz_tile is u32): the 64-bit C tile total is read with the other sums and checked before
    // anything uses the 32-bit scan.
    symbolic_row_kernel<false><<<grid, kRowBlock, lds, s>>>(n, a->offset_row.get(), a->col_idx.get(), S.off_b.get(),
                                                            S.col_b.get(), S.rows.cnt, S.rows.tp, nullptr, nullptr,
                                                            nullptr, S.rows.ref, S.rows.sums);
    MG_LAUNCH_CHECK();
    exclusive_scan_u32(ctx, S.rows.cnt, S.rows.off_c, n);
  }
  unsigned long long h_sums[3] = {0, 0, 0};
  read_words(ctx, {S.rows.sums, h_sums, sizeof(h_sums)});  // the one synchronisation of the pass: the totals
  const uint64_t n_c64 = h_sums[2];
  MG_REQUIRE(n_c64 <= 0xFFFFFFFFull, std::string(who) + ": " + std::to_string(n_c64) +
                                         " output tiles, more than a u32 tile index holds");
  S.n_c = n_c64;
  S.tile_products = h_sums[0];
  S.right_used = h_sums[1];
}

// The structural (row, col) index of C, row-major, into row_c / col_c (S.n_c entries).
void structural_emit(mg_context* ctx, const mg_tiled_matrix* a, const Structural& S, uint32_t* row_c,
                     uint32_t* col_c) {
  if (!S.n_c) return;
  if (S.b.bm) return symbolic_emit(ctx, S.n, S.rows, row_c, col_c);
  const size_t lds = sizeof(uint64_t) * ((S.n + 63) / 64);
  symbolic_row_kernel<true><<<grid_for(S.n, 1, 16384), kRowBlock, lds, ctx->stream>>>(
      S.n, a->offset_row.get(), a->col_idx.get(), S.off_b.get(), S.col_b.get(), nullptr, nullptr, S.rows.off_c,
      row_c, col_c);
  MG_LAUNCH_CHECK();
}

// --- pruned product: only the numerically non-empty tiles of C ------------------
// The pruned C from the flags of its structural tiles and their exclusive scan `pos` (n_s + 1): row and
// column of every flagged tile, the row pointer (pos at the structural rows' starts), and, for tiles
// that were appended, their data from their slots. A wave takes kPlaceTiles structural tiles and has
// up to four in flight.
constexpr uint32_t kPlaceTiles = 16;
struct PrunedTiles {
  uint32_t n_s, n_strips;
  const uint32_t *flag, *pos, *row, *col, *off;
  const uint32_t* slot;    // null: the data is in place
  const uint64_t* scratch; // slots below `capacity`; the others in `rest`
  const uint64_t* rest;
  uint64_t capacity;
};
__global__ void __launch_bounds__(kBlock) place_pruned_kernel(PrunedTiles S, uint32_t* __restrict__ row_c,
                                                              uint32_t* __restrict__ col_c,
                                                              uint32_t* __restrict__ off_c,
                                                              uint64_t* __restrict__ data_c) {
  const uint32_t lane = lane_id();
  for (uint64_t x = blockIdx.x * kBlock + threadIdx.x; x <= S.n_strips; x += static_cast<uint64_t>(gridDim.x) * kBlock)
    off_c[x] = S.pos[S.off[x]];
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kWavesPerBlock * kPlaceTiles;
  for (uint64_t i0 = static_cast<uint64_t>(read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave)) * kPlaceTiles;
       i0 < S.n_s; i0 += stride) {
    const uint64_t i = i0 + lane;
    const bool has = lane < kPlaceTiles && i < S.n_s && S.flag[i] != 0;
    const uint32_t to = has ? S.pos[i] : 0u, from = has && S.slot ? S.slot[i] : 0u;
    if (has) {
      row_c[to] = S.row[i];
      col_c[to] = S.col[i];
    }
    if (!S.slot) continue;
    for (uint64_t m = ballot(has); m;) {
      uint64_t word[4];
      uint32_t at[4];
      uint32_t n = 0;  // wave-uniform
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        word[q] = 0;
        at[q] = 0;
        if (m) {
          const int k = __ffsll(static_cast<unsigned long long>(m)) - 1;
          m &= m - 1;
          at[q] = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(to), k));
          const uint64_t src = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(from), k));
          word[q] = (src < S.capacity ? S.scratch + src * kTile : S.rest + (src - S.capacity) * kTile)[lane];
          ++n;
        }
      }
#pragma unroll
      for (uint32_t q = 0; q < 4; ++q)
        if (q < n) data_c[static_cast<uint64_t>(at[q]) * kTile + lane] = word[q];
    }
  }
}

__global__ void __launch_bounds__(kBlock) row_features_kernel(uint32_t n, const uint32_t* __restrict__ off_a,
                                                              const uint32_t* __restrict__ col_a,
                                                              const TileHead* __restrict__ head_a,
                                                              const unsigned long long* __restrict__ brow_bits,
                                                              const uint32_t* __restrict__ cnt,
                                                              const unsigned long long* __restrict__ tp,
                                                              float* __restrict__ feat) {
  const uint32_t lane = lane_id();
  const uint32_t n_waves = gridDim.x * kWavesPerBlock;
  for (uint32_t x = read_first_lane(blockIdx.x * kWavesPerBlock + threadIdx.x / kWave); x < n; x += n_waves) {
    const uint32_t a0 = off_a[x], a1 = off_a[x + 1];
    uint64_t abits = 0, bbits = 0, amax = 0;
    for (uint32_t k = a0 + lane; k < a1; k += kWave) {
      const uint64_t ab = head_a[k].bits;
      abits += ab;
      amax = ab > amax ? ab : amax;
      bbits += brow_bits[col_a[k]];
    }
    abits = wave_sum(abits);
    bbits = wave_sum(bbits);
    for (int o = 32; o >= 1; o >>= 1) {
      const uint64_t v = static_cast<uint64_t>(__shfl_xor(static_cast<long long>(amax), o, kWave));
      amax = v > amax ? v : amax;
    }
    if (lane == 0) {
      const float nt = static_cast<float>(a1 - a0);
      const float c = static_cast<float>(cnt[x]);
      const float t = static_cast<float>(tp[x]);
      float* f = feat + static_cast<uint64_t>(x) * kRowFeatures;
      f[0] = log1pf(c) / 16.0f;
      f[1] = log1pf(t) / 20.0f;
      f[2] = log1pf(nt) / 16.0f;
      f[3] = log1pf(static_cast<float>(abits)) / 20.0f;
      f[4] = log1pf(static_cast<float>(bbits)) / 24.0f;
      f[5] = log1pf(nt > 0 ? static_cast<float>(abits) / nt : 0.0f) / 8.0f;
      f[6] = log1pf(t > 0 ? static_cast<float>(bbits) / t : 0.0f) / 8.0f;
      f[7] = c / static_cast<float>(n);
    }
  }
}
}  // namespace

// Payload scratch of mg_multiply_numeric_noalloc: one copy per device, held from the moment
// the code object is loaded until the process ends. Host code never passes the name to a
// kernel: it stands for a host-side shadow, not a device address. noalloc_scratch_resolve
// (called by mg_context_create with the device current) looks up this device's address once;
// every later use goes through that pointer. All calls on one device share the array, so
// calls that overlap on one device (different streams or contexts) race.
static __device__ __align__(256) uint64_t scratch[kNoAllocScratchBytes / sizeof(uint64_t)];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

void noalloc_scratch_resolve(int device) {
  MG_REQUIRE(device >= 0 && device < kMaxDevices, "device index beyond the static scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return;
  void* ptr = nullptr;
  MG_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  MG_REQUIRE(ptr != nullptr, "hipGetSymbolAddress returned NULL for the static scratch");
  g_scratch_ptr[device] = ptr;
}

void* noalloc_scratch(int device) {
  MG_REQUIRE(device >= 0 && device < kMaxDevices, "device index beyond the static scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  MG_REQUIRE(g_scratch_ptr[device] != nullptr, "static scratch not resolved for this device");
  return g_scratch_ptr[device];
}

}  // namespace mgamd

using namespace mgamd;

extern "C" int mg_matrix_bit_and(void* stream, const uint64_t* matrix_a, const uint64_t* matrix_b,
                                 uint64_t* matrix_c, uint32_t m, uint32_t k, uint32_t n) {
  return guarded([&] {
    MG_REQUIRE(matrix_a && matrix_b && matrix_c, "mg_matrix_bit_and: NULL buffer");
    if (m == 0 || n == 0 || k == 0) return;
    const uint64_t tasks = static_cast<uint64_t>(m) * ((n + 63) / 64);
    bit_and_kernel<<<grid_for(tasks, kWavesPerBlock, 65536), kBlock, 0, static_cast<hipStream_t>(stream)>>>(
        matrix_a, matrix_b, reinterpret_cast<unsigned long long*>(matrix_c), m, k, n);
    MG_LAUNCH_CHECK();
  });
}

extern "C" int mg_init_bit_tiled_matrix_metadata_by_layout_matrix(void* stream, const uint64_t* layout_matrix,
                                                                  uint32_t n_strips, uint32_t* tile_count_row,
                                                                  uint32_t* tile_row_idx, uint32_t* tile_col_idx) {
  return guarded([&] {
    MG_REQUIRE(layout_matrix && tile_count_row && tile_row_idx && tile_col_idx,
               "mg_init_bit_tiled_matrix_metadata_by_layout_matrix: NULL buffer");
    if (n_strips == 0) return;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // Temporary row counts and their exclusive scan (the reference computes ranks
    // with an O(words) prefix popcount per bit instead, matrix_operations.cu:149-174).
    StreamBuf<uint32_t> cnt(n_strips, s), start(n_strips + 1ull, s);
    layout_row_count_kernel<<<grid_for(n_strips, kWavesPerBlock, 65536), kBlock, 0, s>>>(layout_matrix, n_strips,
                                                                                          cnt.get());
    MG_LAUNCH_CHECK();
    mg_context tmp;  // scan helper needs only the stream
    tmp.stream = s;
    exclusive_scan_u32(&tmp, cnt.get(), start.get(), n_strips);
    layout_emit_kernel<<<grid_for(n_strips, kWavesPerBlock, 65536), kBlock, 0, s>>>(
        layout_matrix, n_strips, start.get(), tile_row_idx, tile_col_idx);
    MG_LAUNCH_CHECK();
    add_counts_kernel<<<grid_for(n_strips, 256), 256, 0, s>>>(tile_count_row, cnt.get(), n_strips);
    MG_LAUNCH_CHECK();
  });
}

extern "C" int mg_fill_tiles(void* stream, size_t tile_size, size_t n_strips, size_t n_nz_tile_a,
                             size_t n_nz_tile_b, size_t n_nz_tile_c, const uint64_t* layout_matrix_c,
                             const uint32_t* tile_offset_row_a, const uint32_t* tile_offset_row_b,
                             const uint32_t* tile_offset_row_c, const uint32_t* tile_row_idx_a,
                             const uint32_t* tile_row_idx_b, const uint32_t* tile_row_idx_c,
                             const uint32_t* tile_col_idx_a, const uint32_t* tile_col_idx_b,
                             const uint32_t* tile_col_idx_c, const uint64_t* data_a, const uint64_t* data_b,
                             uint64_t* data_c) {
  (void)layout_matrix_c; (void)tile_row_idx_a; (void)tile_row_idx_b; (void)tile_offset_row_c;
  (void)n_nz_tile_a; (void)n_nz_tile_b; (void)n_strips;
  return guarded([&] {
    if (tile_size != kTile) fail(MG_ERR_UNSUPPORTED, "mg_fill_tiles: tile_size must be 64");
    if (n_nz_tile_c == 0) return;
    MG_REQUIRE(tile_offset_row_a && tile_offset_row_b && tile_row_idx_c && tile_col_idx_a && tile_col_idx_b &&
                   tile_col_idx_c && data_a && data_b && data_c,
               "mg_fill_tiles: NULL buffer");
    MG_REQUIRE(n_nz_tile_c < (1ull << 32), "mg_fill_tiles: n_nz_tile_c exceeds u32");
    launch_fill_tiles(static_cast<hipStream_t>(stream), static_cast<uint32_t>(n_nz_tile_c), tile_offset_row_a,
                      tile_offset_row_b, tile_row_idx_c, tile_col_idx_c, tile_col_idx_a, tile_col_idx_b, data_a,
                      data_b, data_c);
  });
}

extern "C" int mg_multiply_symbolic(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                    mg_tiled_matrix** c_out, mg_product_stats* stats) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && c_out, "mg_multiply_symbolic: NULL argument");
    *c_out = nullptr;
    DeviceGuard g(ctx->device);
    hipStream_t s = ctx->stream;
    Structural S;
    structural_pass(ctx, a, bt, S, "mg_multiply_symbolic");
    auto c = std::make_unique<mg_tiled_matrix>();
    c->device = ctx->device;
    alloc_tiled_matrix(c.get(), S.n, static_cast<uint32_t>(S.n_c));
    c->product_pairs = S.tile_products;
    MG_HIP(hipMemcpyAsync(c->offset_row.get(), S.rows.off_c, sizeof(uint32_t) * (S.n + 1ull),
                          hipMemcpyDeviceToDevice, s));
    if (S.n_c) {
      MG_HIP(hipMemsetAsync(c->data.get(), 0, c->data.bytes(), s));
      structural_emit(ctx, a, S, c->row_idx.get(), c->col_idx.get());
    }
    if (stats) {
      stats->tile_products = S.tile_products;
      stats->right_tiles_used = S.right_used;
      stats->out_tiles = S.n_c;
      stats->alg_bytes = 520ull * (a->n_nz_tile + S.right_used + S.n_c) + 4ull * (2ull * S.n + 2);
    }
    *c_out = c.release();
  });
}

extern "C" int mg_tiled_matrix_prepare_operand(mg_context* ctx, mg_tiled_matrix* m) {
  return guarded([&] {
    MG_REQUIRE(ctx && m, "mg_tiled_matrix_prepare_operand: NULL argument");
    MG_REQUIRE(m->tile_size == 64, "mg_tiled_matrix_prepare_operand: tile_size must be 64");
    if (prepared(m)) return;  // kept copy still current
    DeviceGuard g(ctx->device);
    hipStream_t st = ctx->stream;
    const uint32_t n = m->n_nz_tile;
    m->prep_payload.alloc(2ull * std::max<uint32_t>(1, n));
    unsigned long long used = 0;
    if (n) {
      unsigned long long* const sum = ctx->counters.get();
      MG_HIP(hipMemsetAsync(sum, 0, sizeof(*sum), st));
      payload_kernel<<<grid_for(n, kWavesPerBlock, 16384), kBlock, 0, st>>>(
          m->data.get(), n, nullptr, 0, reinterpret_cast<WidePayload*>(m->prep_payload.get()), sum);
      MG_LAUNCH_CHECK();
      read_words(ctx, {sum, &used, sizeof(used)});
    }
    prepare_operand(ctx, m, used);
    MG_HIP(hipStreamSynchronize(st));
    m->prep_version = m->version;
  });
}

extern "C" int mg_multiply_numeric(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                   mg_tiled_matrix* c) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && c, "mg_multiply_numeric: NULL argument");
    MG_REQUIRE(a->n_strips == bt->n_strips && c->n_strips == a->n_strips,
               "mg_multiply_numeric: operands differ in n_strips");
    DeviceGuard g(ctx->device);
    ScratchScope scratch(ctx);
    ++c->version;
    if (c->n_nz_tile == 0) return;
    ProductInputs in;
    product_inputs(ctx, a, bt, ProductTiles{c->n_nz_tile, c->row_idx.get(), c->col_idx.get()}, false, true, c->product_pairs, in);
    ProductOut out{};
    out.data = c->data.get();
    run_product(ctx, in, kOutStruct, out);
  });
}

namespace mgamd {
namespace {

// Structural index and operand inputs of a pruned product.
struct PrunedPlan {
  Structural S;
  StreamBuf<uint32_t> mem;  // the structural tiles: rows, columns, flags, slots, the flags' scan
  uint32_t *row_s, *col_s, *flag, *slot, *pos;
  unsigned long long* counter;
  ProductInputs in;
};

void pruned_prepare(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, PrunedPlan& P,
                    bool want_bits, const char* who) {
  hipStream_t s = ctx->stream;
  structural_pass(ctx, a, bt, P.S, who);
  const uint32_t n_s = static_cast<uint32_t>(P.S.n_c);
  P.mem.alloc(5ull * n_s + 4, s);
  P.counter = reinterpret_cast<unsigned long long*>(P.mem.get());
  P.row_s = P.mem.get() + 2;
  P.col_s = P.row_s + n_s;
  P.flag = P.col_s + n_s;
  P.slot = P.flag + n_s;
  P.pos = P.slot + n_s;
  structural_emit(ctx, a, P.S, P.row_s, P.col_s);
  product_inputs(ctx, a, bt, ProductTiles{n_s, P.row_s, P.col_s}, want_bits, true, P.S.tile_products, P.in, P.S.b);
}

// Features of every C row into feat (device, n_strips x kRowFeatures).
// in: the product's inputs, with set-bit counts. brow: n_strips of scratch.
void row_features_into(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, const Structural& S,
                       const ProductInputs& in, unsigned long long* brow, float* feat) {
  hipStream_t s = ctx->stream;
  const uint32_t n = S.n;
  if (!n) return;
  right_row_bits(ctx, bt, in, brow);
  row_features_kernel<<<grid_for(n, kWavesPerBlock, 65536), kBlock, 0, s>>>(
      n, a->offset_row.get(), a->col_idx.get(), in.a.head, brow, S.rows.cnt, S.rows.tp, feat);
  MG_LAUNCH_CHECK();
}

// Output slots from a prediction: per row min(structural, ceil(structural * clamp(y) *
// (1 + margin))); the total into *out, the unrounded prediction per row into pred.
__global__ void __launch_bounds__(kBlock) capacity_kernel(uint32_t n, const uint32_t* __restrict__ cnt,
                                                          const float* __restrict__ y, uint32_t y_stride,
                                                          float margin, float* __restrict__ pred,
                                                          unsigned long long* __restrict__ out) {
  uint64_t local = 0;
  for (uint32_t x = blockIdx.x * blockDim.x + threadIdx.x; x < n; x += gridDim.x * blockDim.x) {
    const float c = static_cast<float>(cnt[x]);
    const float f = fminf(fmaxf(y[static_cast<uint64_t>(x) * y_stride], 0.0f), 1.0f);
    const float pr = c * f;
    pred[x] = pr;
    const float cap = fminf(ceilf(pr * (1.0f + margin)), c);
    local += static_cast<uint64_t>(cap);
  }
  local = wave_sum(local);
  if (lane_id() == 0 && local) atomicAdd(out, static_cast<unsigned long long>(local));
}

// Numeric passes of a pruned product into *c (see mg_multiply_pruned for `capacity`).
void pruned_execute(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, PrunedPlan& P,
                    uint64_t capacity, mg_tiled_matrix* c, mg_pruned_stats& st) {
  hipStream_t s = ctx->stream;
  const Structural& S = P.S;
  const uint32_t n_s = static_cast<uint32_t>(S.n_c);
  st.structural_tiles = n_s;
  st.tile_products = S.tile_products;
  uint64_t n_num = 0;
  uint64_t cap = capacity == MG_PRUNED_STRUCTURAL ? n_s : std::min<uint64_t>(capacity, n_s);
  PrunedTiles tiles{n_s, S.n, P.flag, P.pos, P.row_s, P.col_s, S.rows.off_c, nullptr, nullptr, nullptr, 0};
  const auto place = [&] {
    place_pruned_kernel<<<grid_for(std::max<uint64_t>(n_s, S.n + 1ull), kWavesPerBlock * kPlaceTiles, 16384), kBlock, 0, s>>>(
        tiles, c->row_idx.get(), c->col_idx.get(), c->offset_row.get(), c->data.get());
    MG_LAUNCH_CHECK();
  };
  if (capacity == MG_PRUNED_EXACT || n_s == 0) {
    // Exact: flag pass, scan, then each non-empty tile written at its final position.
    ProductOut fo{};
    fo.flag = P.flag;
    run_product(ctx, P.in, kOutFlag, fo);
    exclusive_scan_u32(ctx, P.flag, P.pos, n_s);
    uint32_t n32 = 0;
    read_words(ctx, {P.pos + n_s, &n32, sizeof(n32)});
    n_num = n32;
    alloc_tiled_matrix(c, S.n, n32);
    if (n32) {
      ProductOut po{};
      po.data = c->data.get();
      po.pos = P.pos;
      run_product(ctx, P.in, kOutPos, po);
    }
    place();
    st.passes = 2;
    st.capacity = n32;
    st.scratch_bytes = 0;
  } else {
    // One pass into `cap` slots; the counter keeps counting past them, and the tiles that found none are
    // made in a second pass over their windows.
    st.capacity = cap;
    StreamBuf<uint64_t> scratch(cap * kTile, s), rest;
    MG_HIP(hipMemsetAsync(P.counter, 0, sizeof(unsigned long long), s));
    ProductOut ao{};
    ao.data = scratch.get();
    ao.flag = P.flag;
    ao.slot = P.slot;
    ao.counter = P.counter;
    ao.capacity = cap;
    run_product(ctx, P.in, kOutAppend, ao);
    // Row-major order: the tiles' places are the scan of their flags.
    exclusive_scan_u32(ctx, P.flag, P.pos, n_s);
    unsigned long long got = 0;
    read_words(ctx, {P.counter, &got, sizeof(got)});
    n_num = got;
    st.passes = got > cap ? 2 : 1;
    st.fallback = got > cap ? 1 : 0;
    st.scratch_bytes = std::max<uint64_t>(got, cap) * kTile * sizeof(uint64_t);
    if (got > cap) {
      rest.alloc((got - cap) * kTile, s);
      ao.data = rest.get();
      run_product(ctx, P.in, kOutRest, ao);
    }
    alloc_tiled_matrix(c, S.n, static_cast<uint32_t>(got));
    tiles.slot = P.slot;
    tiles.scratch = scratch.get();
    tiles.rest = rest.get();
    tiles.capacity = cap;
    place();
  }
  MG_HIP(hipStreamSynchronize(s));
  st.numeric_tiles = n_num;
  st.output_bytes = n_num * kTile * sizeof(uint64_t);
}

}  // namespace
}  // namespace mgamd

extern "C" int mg_multiply_pruned(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                  uint64_t capacity, mg_tiled_matrix** c_out, mg_pruned_stats* stats) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && c_out, "mg_multiply_pruned: NULL argument");
    *c_out = nullptr;
    DeviceGuard g(ctx->device);
    ScratchScope scratch(ctx);
    PrunedPlan P;
    pruned_prepare(ctx, a, bt, P, false, "mg_multiply_pruned");
    auto c = std::make_unique<mg_tiled_matrix>();
    c->device = ctx->device;
    mg_pruned_stats st{};
    pruned_execute(ctx, a, bt, P, capacity, c.get(), st);
    if (stats) *stats = st;
    *c_out = c.release();
  });
}

extern "C" int mg_multiply_pruned_model(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                        const mg_mlp* model, float margin, float* row_predicted,
                                        mg_tiled_matrix** c_out, mg_pruned_stats* stats) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && model && c_out, "mg_multiply_pruned_model: NULL argument");
    *c_out = nullptr;
    MG_REQUIRE(margin >= 0.0f && margin <= 16.0f, "mg_multiply_pruned_model: margin must be in [0, 16]");
    uint32_t n_in = 0, n_out = 0;
    mlp_dims(model, &n_in, &n_out);
    MG_REQUIRE(n_in == kRowFeatures && n_out >= 1,
               "mg_multiply_pruned_model: the model must take MG_ROW_FEATURES inputs");
    DeviceGuard g(ctx->device);
    ScratchScope scratch(ctx);
    hipStream_t s = ctx->stream;
    PrunedPlan P;
    pruned_prepare(ctx, a, bt, P, true, "mg_multiply_pruned_model");
    const uint32_t n = P.S.n;
    uint64_t capacity = MG_PRUNED_EXACT;
    if (P.S.n_c) {
      // u64: total, B's row bits; then the features, the model's outputs and the rows' predictions.
      const uint64_t feat_at = (1ull + n + 31) / 32 * 32;  // the model loads rows of 32 bytes
      StreamBuf<unsigned long long> mem(feat_at + (static_cast<uint64_t>(n) * (kRowFeatures + n_out + 1) + 1) / 2, s);
      unsigned long long* const total = mem.get();
      float* const feat = reinterpret_cast<float*>(total + feat_at);
      float* const y = feat + static_cast<uint64_t>(n) * kRowFeatures;
      float* const pred = y + static_cast<uint64_t>(n) * n_out;
      row_features_into(ctx, a, bt, P.S, P.in, total + 1, feat);
      if (mg_mlp_forward(ctx, model, feat, n, y) != MG_OK)
        fail(MG_ERR_INTERNAL, std::string("mg_multiply_pruned_model: ") + mg_last_error());
      MG_HIP(hipMemsetAsync(total, 0, sizeof(unsigned long long), s));
      capacity_kernel<<<grid_for(n, kBlock, 1024), kBlock, 0, s>>>(n, P.S.rows.cnt, y, n_out, margin, pred, total);
      MG_LAUNCH_CHECK();
      unsigned long long h = 0;
      if (row_predicted) MG_HIP(hipMemcpyAsync(row_predicted, pred, sizeof(float) * n, hipMemcpyDeviceToHost, s));
      read_words(ctx, {total, &h, sizeof(h)});
      capacity = std::max<unsigned long long>(1, h);
    } else if (row_predicted && n) {
      std::fill(row_predicted, row_predicted + n, 0.0f);
    }
    auto c = std::make_unique<mg_tiled_matrix>();
    c->device = ctx->device;
    mg_pruned_stats st{};
    pruned_execute(ctx, a, bt, P, capacity, c.get(), st);
    if (stats) *stats = st;
    *c_out = c.release();
  });
}

extern "C" int mg_multiply_row_features(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                        float* features, uint32_t* structural, uint64_t* tile_products) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && features, "mg_multiply_row_features: NULL argument");
    DeviceGuard g(ctx->device);
    ScratchScope scratch(ctx);
    hipStream_t s = ctx->stream;
    Structural S;
    structural_pass(ctx, a, bt, S, "mg_multiply_row_features");
    const uint32_t n = S.n;
    StreamBuf<float> feat(static_cast<uint64_t>(n) * kRowFeatures, s);
    ProductInputs in;
    product_inputs(ctx, a, bt, ProductTiles{}, true, false, S.tile_products, in, S.b);
    StreamBuf<unsigned long long> brow(n, s);
    row_features_into(ctx, a, bt, S, in, brow.get(), feat.get());
    if (n) {
      MG_HIP(hipMemcpyAsync(features, feat.get(), sizeof(float) * n * kRowFeatures, hipMemcpyDeviceToHost, s));
      if (structural)
        MG_HIP(hipMemcpyAsync(structural, S.rows.cnt, sizeof(uint32_t) * n, hipMemcpyDeviceToHost, s));
    }
    MG_HIP(hipStreamSynchronize(s));
    if (tile_products) *tile_products = S.tile_products;
  });
}

extern "C" int mg_multiply_numeric_noalloc(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                           mg_tiled_matrix* c) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && c, "mg_multiply_numeric_noalloc: NULL argument");
    MG_REQUIRE(a->n_strips == bt->n_strips && c->n_strips == a->n_strips,
               "mg_multiply_numeric_noalloc: operands differ in n_strips");
    ++c->version;
    const size_t words = payload_words(a, bt);
    if (words * sizeof(uint64_t) > kNoAllocScratchBytes)
      invalid("mg_multiply_numeric_noalloc: " + std::to_string(a->n_nz_tile) + " + " +
              std::to_string(bt->n_nz_tile) + " operand tiles need " + std::to_string(words * sizeof(uint64_t)) +
              " bytes of payload scratch, more than the static " + std::to_string(kNoAllocScratchBytes) +
              " (at most " + std::to_string(kNoAllocMaxTiles) + " tiles in A and Bt together)");
    DeviceGuard g(ctx->device);
    if (c->n_nz_tile == 0) return;
    // The device address of this device's copy of `scratch`, looked up when the context was
    // created; the kernels write every payload word they read, so nothing is cleared.
    WidePayload* pl = reinterpret_cast<WidePayload*>(noalloc_scratch(ctx->device));
    launch_payloads(ctx->stream, a, bt, pl);
    fill_tiles_payload_kernel<<<grid_for(c->n_nz_tile, kWavesPerBlock, 65536), kBlock, 0, ctx->stream>>>(
        c->n_nz_tile, a->offset_row.get(), bt->offset_row.get(), c->row_idx.get(), c->col_idx.get(), a->col_idx.get(),
        bt->col_idx.get(), a->data.get(), bt->data.get(), pl, pl + a->n_nz_tile, c->data.get());
    MG_LAUNCH_CHECK();
  });
}

extern "C" int mg_multiply_numeric_dense(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                                         mg_tiled_matrix* c, uint32_t min_bits, uint64_t* dense_products) {
  return guarded([&] {
    MG_REQUIRE(ctx && a && bt && c, "mg_multiply_numeric_dense: NULL argument");
    MG_REQUIRE(a->n_strips == bt->n_strips && c->n_strips == a->n_strips,
               "mg_multiply_numeric_dense: operands differ in n_strips");
    DeviceGuard g(ctx->device);
    ScratchScope scratch(ctx);
    ++c->version;
    ProductInputs in;
    product_inputs(ctx, a, bt, ProductTiles{c->n_nz_tile, c->row_idx.get(), c->col_idx.get()}, true, true, c->product_pairs, in);
    const uint64_t recorded = run_product_dense(ctx, a, bt, in, min_bits, c->data.get());
    // The caller may read C, or write A, from any stream once this returns.
    MG_HIP(hipStreamSynchronize(ctx->stream));
    if (dense_products) *dense_products = recorded;
  });
}
