// Internal definitions shared by the HIP translation units of libmatrixgraph_amd.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <memory>
#include <new>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "matrixgraph_amd.h"
#include "mg_block_cache.hpp"

namespace mgamd {

// ---------------------------------------------------------------------------
// Errors: every C entry point runs its body under guarded(), which maps the
// exceptions below to status codes and records the message for mg_last_error().
// ---------------------------------------------------------------------------
struct Failure : std::runtime_error {
  int code;
  Failure(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void set_last_error(const std::string& msg);

[[noreturn]] inline void fail(int code, const std::string& msg) { throw Failure(code, msg); }
[[noreturn]] inline void invalid(const std::string& msg) { throw Failure(MG_ERR_INVALID, msg); }

inline void hip_check(hipError_t e, const char* what, const char* file, int line) {
  if (e == hipSuccess) return;
  (void)hipGetLastError();  // clear the sticky launch error so later calls report their own
  const int code = (e == hipErrorOutOfMemory) ? MG_ERR_OOM : MG_ERR_HIP;
  throw Failure(code, std::string(what) + ": " + hipGetErrorString(e) + " (" + file + ":" +
                          std::to_string(line) + ")");
}
#define MG_HIP(call) ::mgamd::hip_check((call), #call, __FILE__, __LINE__)
#define MG_LAUNCH_CHECK() ::mgamd::hip_check(hipGetLastError(), "kernel launch", __FILE__, __LINE__)

template <class F>
int guarded(F&& f) {
  try {
    f();
    return MG_OK;
  } catch (const Failure& e) {
    set_last_error(e.what());
    return e.code;
  } catch (const std::bad_alloc&) {
    set_last_error("host allocation failed");
    return MG_ERR_OOM;
  } catch (const std::exception& e) {
    set_last_error(e.what());
    return MG_ERR_INTERNAL;
  } catch (...) {
    set_last_error("unknown failure");
    return MG_ERR_INTERNAL;
  }
}

#define MG_REQUIRE(cond, msg) \
  do {                        \
    if (!(cond)) ::mgamd::invalid(msg); \
  } while (0)

// ---------------------------------------------------------------------------
// Device memory of objects (mg_context.hip): hipMalloc blocks that cached_free keeps for the next
// cached_alloc of about their size instead of giving them back to the driver. A result matrix of
// 64 MB costs ~25 us to allocate and ~300 us to free there, one of 2 GB 330 and 590 us, and a
// program that makes and drops such results faster than the driver clears freed memory waits in
// hipMalloc for up to a second; a kept block costs a few microseconds.
//  - cached_free waits for all work on the device, as hipFree does, so a kept block is idle whichever
//    streams used it. Inside a FreeScope the frees share one wait.
//  - Kept: at most 1/64 of the device's memory, oldest blocks out first, none above half of that;
//    all of it is given back when the device's last context is destroyed, and, with what the
//    temporaries' pool does not use, when an allocation here or from the pool finds no memory, which is
//    then tried again. Without a context alive blocks go straight to hipFree.
//  - Safe from any thread. In a stream capture that forbids hipFree, cached_free does what hipFree
//    does (nothing is kept).
// ---------------------------------------------------------------------------
void* cached_alloc(size_t bytes);  // on the current device; throws Failure
// The driver's answer where the block goes back to it; hipErrorInvalidValue for a block that was freed
// before and is kept.
hipError_t cached_free(void* p) noexcept;
// A temporary from the device's default pool, in stream order (hipFreeAsync gives it back); throws Failure.
void* pool_alloc(size_t bytes, hipStream_t stream);
void cache_add_context(int device, size_t device_bytes);
void cache_drop_context(int device) noexcept;

// Device buffer (RAII, move-only). Allocation is explicit; freeing happens in
// the destructor. Only setup paths allocate; timed hop loops reuse buffers.
template <class T>
class DevBuf {
 public:
  DevBuf() = default;
  explicit DevBuf(size_t n) { alloc(n); }
  ~DevBuf() { release(); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p_(o.p_), n_(o.n_) { o.p_ = nullptr; o.n_ = 0; }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) { release(); p_ = o.p_; n_ = o.n_; o.p_ = nullptr; o.n_ = 0; }
    return *this;
  }
  void alloc(size_t n) {
    release();
    if (n == 0) return;
    p_ = static_cast<T*>(cached_alloc(n * sizeof(T)));
    n_ = n;
  }
  void release() {
    if (p_) (void)cached_free(p_);
    p_ = nullptr;
    n_ = 0;
  }
  T* get() const { return p_; }
  size_t size() const { return n_; }
  size_t bytes() const { return n_ * sizeof(T); }

 private:
  T* p_ = nullptr;
  size_t n_ = 0;
};

// Stream-ordered temporary from the device's default memory pool: hipMallocAsync and
// hipFreeAsync on one stream (the caller's context stream). Kernels queued on that stream
// before the buffer goes out of scope finish before its memory is reused, so a call can
// return without synchronising just to free its temporaries. mg_context_create keeps freed
// memory in the pool (release threshold: never), so repeated calls reuse it instead of
// going back to the driver. Counterpart of DeviceOwnedBuffer::Init (device_buffer.cuh:92-106)
// for temporaries; long-lived results keep DevBuf.
template <class T>
class StreamBuf {
 public:
  StreamBuf() = default;
  StreamBuf(size_t n, hipStream_t s) { alloc(n, s); }
  ~StreamBuf() { release(); }
  // At least one element, so get() is never null.
  void alloc(size_t n, hipStream_t s) {
    release();
    s_ = s;
    if (n == 0) n = 1;
    p_ = static_cast<T*>(pool_alloc(n * sizeof(T), s_));
    n_ = n;
  }
  void release() {
    if (p_) (void)hipFreeAsync(p_, s_);
    p_ = nullptr;
    n_ = 0;
  }
  StreamBuf(const StreamBuf&) = delete;
  StreamBuf& operator=(const StreamBuf&) = delete;
  StreamBuf(StreamBuf&& o) noexcept : p_(o.p_), n_(o.n_), s_(o.s_) { o.p_ = nullptr; o.n_ = 0; }
  T* get() const { return p_; }
  size_t size() const { return n_; }
  size_t bytes() const { return n_ * sizeof(T); }

 private:
  T* p_ = nullptr;
  size_t n_ = 0;
  hipStream_t s_ = nullptr;
};

// Pinned host staging buffer (hipHostMalloc; never hipHostRegister).
template <class T>
class PinnedBuf {
 public:
  PinnedBuf() = default;
  explicit PinnedBuf(size_t n) { alloc(n); }
  ~PinnedBuf() { if (p_) (void)hipHostFree(p_); }
  PinnedBuf(const PinnedBuf&) = delete;
  PinnedBuf& operator=(const PinnedBuf&) = delete;
  void alloc(size_t n) {
    if (p_) (void)hipHostFree(p_);
    p_ = nullptr;
    if (n == 0) return;
    MG_HIP(hipHostMalloc(reinterpret_cast<void**>(&p_), n * sizeof(T), hipHostMallocDefault));
  }
  T* get() const { return p_; }

 private:
  T* p_ = nullptr;
};

// Scoped device switch: restores the caller's current device.
struct DeviceGuard {
  int prev = 0;
  explicit DeviceGuard(int dev) {
    MG_HIP(hipGetDevice(&prev));
    if (prev != dev) MG_HIP(hipSetDevice(dev));
  }
  ~DeviceGuard() { (void)hipSetDevice(prev); }
};

}  // namespace mgamd

// ---------------------------------------------------------------------------
// Handle definitions (opaque to C callers).
// ---------------------------------------------------------------------------
struct mg_context {
  int device = 0;
  int n_cu = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  mgamd::DevBuf<unsigned long long> counters;  // small scratch for reductions (host-synchronised calls)
  hipEvent_t timer[2] = {nullptr, nullptr};    // mg_context_timer_start / _stop
  // Per-call device temporaries of asynchronous calls on `stream` (calls on one context run
  // in stream order, so the next call may reuse them); grown by ctx_scratch, stream-ordered. At most
  // scratch_limit bytes stay from one call to the next (ScratchScope).
  mgamd::StreamBuf<uint64_t> scratch;
  size_t scratch_limit = 0;  // 1/64 of the device's memory, as for kept blocks
  int scratch_users = 0;     // ScratchScopes
  mgamd::PinnedBuf<uint32_t> mail;  // read_words
};

struct mg_tiled_matrix {
  int device = 0;
  uint32_t n_strips = 0;
  uint32_t n_nz_tile = 0;
  uint32_t tile_size = 64;
  mgamd::DevBuf<uint32_t> offset_row;  // n_strips + 1
  mgamd::DevBuf<uint32_t> row_idx;     // n_nz_tile
  mgamd::DevBuf<uint32_t> col_idx;     // n_nz_tile
  mgamd::DevBuf<uint64_t> data;        // 64 * n_nz_tile
  // Tile pairs that meet in the product whose symbolic pass made this matrix (0: none did).
  uint64_t product_pairs = 0;
  // Bumped by every library call that writes this matrix's tiles (the numeric passes into C).
  uint64_t version = 0;
  // mg_tiled_matrix_prepare_operand, valid while prep_version == version: payloads (16 B a tile, the
  // allocation-free pass) and the inputs of mg_product.hpp: heads by tile and by position of B,
  // column words, bitmap; ranks, row offsets and tiles by position.
  mgamd::DevBuf<uint64_t> prep_payload;
  mgamd::DevBuf<uint64_t> prep_head;
  mgamd::DevBuf<uint64_t> prep_right_head;
  mgamd::DevBuf<uint64_t> prep_words;
  mgamd::DevBuf<uint64_t> prep_bitmap;
  mgamd::DevBuf<uint32_t> prep_index;
  mgamd::DevBuf<uint32_t> prep_weight;  // per tile row: columns in use of its tiles
  uint64_t prep_version = ~0ull;
};

struct mg_edge_list {
  int device = 0;
  uint32_t n_vertices = 0;
  uint64_t n_edges = 0;
  mgamd::DevBuf<uint64_t> keys;  // (src << 32) | dst, ascending, unique
};

namespace mgamd {

// At least n words of ctx->scratch; growing it first waits for the work queued on the
// context's stream, which may still read the old buffer.
inline uint64_t* ctx_scratch(mg_context* ctx, size_t n) {
  // The old buffer is freed in stream order: work already queued that reads it finishes first.
  if (ctx->scratch.size() < n) ctx->scratch.alloc(n, ctx->stream);
  return ctx->scratch.get();
}

// Around an entry point that uses ctx_scratch: once the outermost is left, a scratch above the limit is
// freed, in stream order. Not inside a capture, whose graph goes on using it.
struct ScratchScope {
  mg_context* ctx;
  explicit ScratchScope(mg_context* c) : ctx(c) { ++ctx->scratch_users; }
  ~ScratchScope() {
    if (--ctx->scratch_users || ctx->scratch.bytes() <= ctx->scratch_limit) return;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &capture) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    if (capture == hipStreamCaptureStatusNone) ctx->scratch.release();
  }
  ScratchScope(const ScratchScope&) = delete;
  ScratchScope& operator=(const ScratchScope&) = delete;
};

// Static payload scratch of mg_multiply_numeric_noalloc (mg_spgemm.hip): 32 MiB per device,
// 16 bytes per tile of both operands plus 16 (kNoAllocMaxTiles tiles in A and Bt together).
constexpr size_t kNoAllocScratchBytes = 32ull << 20;
constexpr uint64_t kNoAllocMaxTiles = kNoAllocScratchBytes / 16 - 1;
constexpr int kMaxDevices = 64;
// Looks up this device's address of the static scratch (device current); once per device.
void noalloc_scratch_resolve(int device);
// The address looked up by noalloc_scratch_resolve for `device`.
void* noalloc_scratch(int device);

// Input and output widths of a cost-model MLP (mg_mlp.hip).
void mlp_dims(const mg_mlp* p, uint32_t* n_in, uint32_t* n_out);

// Helpers implemented in mg_matrix.hip / mg_graph.hip, shared across units.
void alloc_tiled_matrix(mg_tiled_matrix* m, uint32_t n_strips, uint32_t n_nz_tile);
uint64_t device_popcount(mg_context* ctx, const uint64_t* data, uint64_t n_words);
// Sum of n u32 values, in 64 bits (for totals that a u32 scan would wrap).
uint64_t device_sum_u32(mg_context* ctx, const uint32_t* data, uint64_t n);
// Reads a few words of device memory (4-byte aligned, kMailWords together) into host memory once the
// stream gets there; waits for it. A kernel writes them to pinned memory: half the time of a copy.
struct DeviceWords {
  const void* from;
  void* to;
  uint32_t bytes;
};
constexpr uint32_t kMailWords = 64;
void read_words(mg_context* ctx, DeviceWords a, DeviceWords b = {nullptr, nullptr, 0});
// Exclusive scan of n u32 counts into out[0..n] (out[n] = total), on ctx->stream.
void exclusive_scan_u32(mg_context* ctx, const uint32_t* in, uint32_t* out, uint32_t n);
void exclusive_scan_u32_on(hipStream_t st, const uint32_t* in, uint32_t* out, uint32_t n);
// Sorts n < 2^31 keys by their bits [begin_bit, end_bit), stable; returns where they are, keys or alt. temp:
// sort_u64_bytes of scratch.
size_t sort_u64_bytes(uint64_t n, int begin_bit, int end_bit);
uint64_t* sort_u64(hipStream_t st, uint64_t* keys, uint64_t* alt, uint64_t n, int begin_bit, int end_bit, void* temp,
                   size_t temp_bytes);
// v[0 .. n] = exclusive scan of v[0 .. n) (v[n]: total), 16-byte aligned; one workgroup: for a few thousand.
void scan_in_place(hipStream_t st, uint32_t* v, uint32_t n);

inline unsigned grid_for(uint64_t work, unsigned per_block, unsigned cap = 1u << 20) {
  uint64_t g = (work + per_block - 1) / per_block;
  if (g == 0) g = 1;
  if (g > cap) g = cap;
  return static_cast<unsigned>(g);
}

}  // namespace mgamd
