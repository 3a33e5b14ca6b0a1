// Numeric pass of the handle-level tile products (mg_product.hip), used by the entry points of
// mg_spgemm.hip.
#pragma once

#include "mg_internal.hpp"

namespace mgamd {

// What a product reads of a tile instead of its 512 bytes: the columns in use (the inner indices j
// through which it meets the other operand's tiles), and its non-zero column words (bit r of
// column word j = bit j of row r) at words[off], in ascending j; off = kNoWords: not stored.
struct TileHead {
  uint64_t mask;
  uint32_t off;
  uint32_t bits;  // set bits (0 where the caller does not ask for them)
};
static_assert(sizeof(TileHead) == 16, "loaded as one 16-byte word");
constexpr uint32_t kNoWords = 0xFFFFFFFFu;

// Left operand A: heads in tile order.
struct LeftOperand {
  const TileHead* head;
  const uint64_t* words;
  const uint64_t* data;
  const uint32_t* off;  // A's row pointer
  const uint32_t* col;
};

// Word of B's bitmap: which of 64 strips y have a tile B(t, y), and the position of the first.
struct BitmapWord {
  uint64_t bits;
  uint32_t at, pad;
};
// Right operand B, from Bt's tiles (y, t). For product_kernel by its tile rows t: positions
// off[t] .. off[t + 1] - 1 are the tiles B(t, y) in ascending y, found through the bitmap. For
// tile_product_kernel: position = tile of Bt, found in Bt's own rows.
struct RightOperand {
  const TileHead* head;   // by position
  const uint64_t* words;
  const uint64_t* data;   // Bt's tiles
  const uint32_t* tile;   // position -> tile of Bt
  const BitmapWord* bm;   // null: by tiles of Bt
  const uint32_t* off;
  const uint32_t* bt_off;
  const uint32_t* bt_col;
};
constexpr uint32_t kBitmapStrips = 16384;

// The bitmap of B and its row pointer (grids up to kBitmapStrips).
struct RightIndex {
  const BitmapWord* bm = nullptr;
  const uint32_t* off = nullptr;
};
// Of a prepared operand from its handle, else made in mem.
RightIndex right_index(mg_context* ctx, const mg_tiled_matrix* bt, StreamBuf<uint64_t>& mem);

// Structural pass of C = A * B over bitmaps: per tile row x of C its strips in c_bits (n_strips rows of
// 64-bit words; rows without tiles of A are not written), their count cnt, and the tile products tp; then
// C's row pointer and the totals (tile products, tiles of the B rows that A refers to, C tiles).
struct SymbolicRows {
  uint64_t* c_bits;
  uint32_t* cnt;
  unsigned long long* tp;
  uint32_t* off_c;            // n_strips + 1
  uint32_t* ref;              // n_strips, scratch
  unsigned long long* sums;   // 3
};
void symbolic_rows(mg_context* ctx, const mg_tiled_matrix* a, const RightIndex& b, const SymbolicRows& S);
// Row and column of every tile of C, row-major.
void symbolic_emit(mg_context* ctx, uint32_t n_strips, const SymbolicRows& S, uint32_t* row_c, uint32_t* col_c);

// The n_c tiles of C, row-major.
struct ProductTiles {
  uint32_t n_c;
  const uint32_t* row;
  const uint32_t* col;
};

// Tiles of C for one workgroup: those of tile row x in the strips y0 .. y0 + kWindow - 1 below `end`,
// from tile `first` on; A's row x is tiles a0 .. a1 - 1.
struct Window {
  uint32_t first, x, y0, end, a0, a1, pad[2];
};
static_assert(sizeof(Window) == 32, "laid out in u64 words");

// Inputs of C = A * B. All of it lies in the context's scratch (ctx_scratch: the next call on the
// context overwrites it) or in prepared operands.
struct ProductInputs {
  uint32_t n_strips = 0;
  ProductTiles c{};
  LeftOperand a{};
  RightOperand b{};
  uint64_t pairs = 0;         // tile pairs that meet, or an estimate
  Window* windows = nullptr;  // *n_windows of them
  uint32_t* n_windows = nullptr;
};

// Stream-ordered, no synchronisation; no allocation if the context's scratch is large enough.
// want_bits: TileHead::bits; want_words: false leaves the column words out (heads only). pairs: the tile
// pairs that meet, 0 if not known (only the choice of kernel depends on it). known: B's index if it is
// made already.
void product_inputs(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt, const ProductTiles& c,
                    bool want_bits, bool want_words, uint64_t pairs, ProductInputs& P, const RightIndex& known = {});
// Operand kept with its handle (mg_tiled_matrix_prepare_operand): all but the payloads.
bool prepared(const mg_tiled_matrix* m);
// used_columns: columns in use of all tiles, which is the number of column words.
void prepare_operand(mg_context* ctx, mg_tiled_matrix* m, uint64_t used_columns);

// Where a finished C tile goes: ORed into data at its index (kOutStruct), or, for a pruned product,
// only if it is non-zero: into the next slot of data, whether and which in flag and slot
// (kOutAppend; slots past capacity are counted but not written), the same tiles whose slots of an
// earlier kOutAppend were past capacity (kOutRest, slot - capacity), flagged in flag (kOutFlag, no
// data written), or written at pos[i] (kOutPos).
enum : int { kOutStruct = 0, kOutAppend = 1, kOutFlag = 2, kOutPos = 3, kOutRest = 4 };
struct ProductOut {
  uint64_t* data = nullptr;
  uint32_t* flag = nullptr;  // per structural tile
  uint32_t* slot = nullptr;
  const uint32_t* pos = nullptr;
  unsigned long long* counter = nullptr;
  uint64_t capacity = 0;
};

void run_product(mg_context* ctx, const ProductInputs& P, int out_mode, const ProductOut& out);
// kOutStruct with the pairs of tiles that both hold at least min_bits set bits on the matrix cores;
// returns their number. It waits for the count; the contraction may still run when it returns. P needs
// TileHead::bits.
uint64_t run_product_dense(mg_context* ctx, const mg_tiled_matrix* a, const mg_tiled_matrix* bt,
                           const ProductInputs& P, uint32_t min_bits, uint64_t* data_c);
// Set bits of every row t of B into out[t] (P needs TileHead::bits).
void right_row_bits(mg_context* ctx, const mg_tiled_matrix* bt, const ProductInputs& P, unsigned long long* out);

}  // namespace mgamd
