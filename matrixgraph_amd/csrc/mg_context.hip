// Context lifecycle, error reporting and host-only helpers of the C-ABI.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <unordered_map>
#include <unordered_set>

#include "mg_device.hpp"
#include "mg_internal.hpp"

namespace mgamd {
namespace {
thread_local std::string g_last_error;
}
void set_last_error(const std::string& msg) { g_last_error = msg; }

// --- kept device memory ------------------------------------------------------------
namespace {

struct Kept {
  void* ptr;
  uint64_t age;
};
// Blocks of one device.
struct DeviceCache {
  int contexts = 0;
  size_t limit = 0;  // bytes kept at most
  size_t bytes = 0;  // kept now
  uint64_t next_age = 0;
  std::multimap<size_t, Kept> kept;  // by size
};
struct Live {
  size_t bytes;
  int device;
};
struct Cache {
  std::mutex mu;
  std::unordered_map<void*, Live> live;  // blocks handed out
  std::unordered_map<int, DeviceCache> devices;
};
// Never destroyed: objects may outlive static destruction, and the driver reclaims the memory.
Cache& cache() {
  static Cache* const c = new Cache();
  return *c;
}

thread_local int g_free_depth = 0;       // FreeScopes of this thread
thread_local bool g_free_waited = false;  // the outermost scope has waited already

// hipFree of a fresh block: waits for all work on the current device under hipFree's own rules (a
// hipDeviceSynchronize would also break captures that hipFree leaves alone).
bool wait_as_free() {
  void* p = nullptr;
  if (hipMalloc(&p, 256) != hipSuccess || hipFree(p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}

void flush_device(int device) noexcept {
  std::multimap<size_t, Kept> out;
  {
    std::lock_guard<std::mutex> lock(cache().mu);
    auto it = cache().devices.find(device);
    if (it == cache().devices.end()) return;
    out.swap(it->second.kept);
    it->second.bytes = 0;
  }
  for (auto& b : out) (void)hipFree(b.second.ptr);
}

}  // namespace

FreeScope::FreeScope() {
  if (g_free_depth++ == 0) g_free_waited = false;
}
FreeScope::~FreeScope() { --g_free_depth; }

void cache_add_context(int device, size_t device_bytes) {
  std::lock_guard<std::mutex> lock(cache().mu);
  DeviceCache& d = cache().devices[device];
  ++d.contexts;
  d.limit = device_bytes / 64;
}

void cache_drop_context(int device) noexcept {
  bool last = false;
  {
    std::lock_guard<std::mutex> lock(cache().mu);
    last = --cache().devices[device].contexts == 0;
  }
  if (!last) return;
  flush_device(device);
  hipMemPool_t pool = nullptr;  // and the temporaries' pool (StreamBuf)
  if (hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess) (void)hipMemPoolTrimTo(pool, 0);
  (void)hipGetLastError();
}

void* cached_alloc(size_t bytes) {
  bytes = (bytes + 511) / 512 * 512;
  int device = 0;
  MG_HIP(hipGetDevice(&device));
  {
    std::lock_guard<std::mutex> lock(cache().mu);
    DeviceCache& d = cache().devices[device];
    auto it = d.kept.lower_bound(bytes);
    if (it != d.kept.end() && it->first <= bytes + bytes / 8) {
      void* const p = it->second.ptr;
      cache().live[p] = Live{it->first, device};
      d.bytes -= it->first;
      d.kept.erase(it);
      return p;
    }
  }
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    flush_device(device);
    e = hipMalloc(&p, bytes);
  }
  MG_HIP(e);
  try {
    std::lock_guard<std::mutex> lock(cache().mu);
    cache().live[p] = Live{bytes, device};
  } catch (...) {
    (void)hipFree(p);
    throw;
  }
  return p;
}

void cached_free(void* p) noexcept {
  if (!p) return;
  Live l{0, -1};
  bool keep = false;
  {
    std::lock_guard<std::mutex> lock(cache().mu);
    auto it = cache().live.find(p);
    if (it != cache().live.end()) {
      l = it->second;
      cache().live.erase(it);
      auto d = cache().devices.find(l.device);
      keep = d != cache().devices.end() && d->second.contexts > 0 && l.bytes <= d->second.limit / 2;
    }
  }
  int current = -1;
  if (keep && (hipGetDevice(&current) != hipSuccess || current != l.device)) keep = false;
  if (keep && !(g_free_depth > 0 && g_free_waited)) {
    keep = wait_as_free();
    if (keep && g_free_depth > 0) g_free_waited = true;
  }
  if (keep) {
    try {
      std::lock_guard<std::mutex> lock(cache().mu);
      DeviceCache& d = cache().devices[l.device];
      keep = d.contexts > 0;  // the last context may have gone since
      if (keep) {
        d.kept.emplace(l.bytes, Kept{p, d.next_age++});
        d.bytes += l.bytes;
      }
    } catch (...) {
      keep = false;
    }
  }
  if (!keep) {
    (void)hipFree(p);
    return;
  }
  // Over the limit: the oldest blocks go back to the driver.
  for (;;) {
    void* old = nullptr;
    {
      std::lock_guard<std::mutex> lock(cache().mu);
      DeviceCache& d = cache().devices[l.device];
      if (d.bytes <= d.limit || d.kept.empty()) return;
      auto oldest = d.kept.begin();
      for (auto it = d.kept.begin(); it != d.kept.end(); ++it)
        if (it->second.age < oldest->second.age) oldest = it;
      old = oldest->second.ptr;
      d.bytes -= oldest->first;
      d.kept.erase(oldest);
    }
    (void)hipFree(old);
  }
}

}  // namespace mgamd

using namespace mgamd;

extern "C" const char* mg_version(void) { return "matrixgraph_amd 0.1.0 (gfx950)"; }

extern "C" const char* mg_last_error(void) { return g_last_error.c_str(); }

extern "C" int mg_context_create(int device, mg_context** out) {
  return guarded([&] {
    MG_REQUIRE(out != nullptr, "mg_context_create: out is NULL");
    *out = nullptr;
    if (device < 0) {
      // Same role as MATRIXGRAPH_CUDA_DEVICE in core/go_api/matrixgraph_go_api.cu:23-36.
      const char* env = std::getenv("MATRIXGRAPH_HIP_DEVICE");
      device = env ? std::atoi(env) : 0;
    }
    int n_dev = 0;
    MG_HIP(hipGetDeviceCount(&n_dev));
    if (device >= n_dev)
      invalid("mg_context_create: device " + std::to_string(device) + " not present (" +
              std::to_string(n_dev) + " devices)");
    DeviceGuard g(device);
    noalloc_scratch_resolve(device);
    {
      // Temporaries come from the device's default pool (StreamBuf); keep freed memory there.
      hipMemPool_t pool = nullptr;
      MG_HIP(hipDeviceGetDefaultMemPool(&pool, device));
      uint64_t keep = ~0ull;
      MG_HIP(hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep));
    }
    hipDeviceProp_t prop;
    MG_HIP(hipGetDeviceProperties(&prop, device));
    auto* ctx = new mg_context();
    ctx->device = device;
    ctx->n_cu = prop.multiProcessorCount;
    hipError_t e = hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
      delete ctx;
      MG_HIP(e);
    }
    ctx->stream = ctx->own_stream;
    cache_add_context(device, prop.totalGlobalMem);
    try {
      ctx->counters.alloc(64);
      ctx->mail.alloc(kMailWords);
    } catch (...) {
      cache_drop_context(device);
      (void)hipStreamDestroy(ctx->own_stream);
      delete ctx;
      throw;
    }
    *out = ctx;
  });
}

extern "C" int mg_context_destroy(mg_context* ctx) {
  return guarded([&] {
    if (!ctx) return;
    DeviceGuard g(ctx->device);
    ctx->scratch.release();  // stream-ordered: before the stream goes away
    (void)hipStreamSynchronize(ctx->stream);
    ctx->counters.release();
    for (hipEvent_t& e : ctx->timer)
      if (e) (void)hipEventDestroy(e);
    if (ctx->own_stream) (void)hipStreamDestroy(ctx->own_stream);
    cache_drop_context(ctx->device);
    delete ctx;
  });
}

extern "C" int mg_context_set_stream(mg_context* ctx, void* stream) {
  return guarded([&] {
    MG_REQUIRE(ctx != nullptr, "mg_context_set_stream: ctx is NULL");
    const hipStream_t next = stream ? static_cast<hipStream_t>(stream) : ctx->own_stream;
    if (next != ctx->stream) {
      // Work queued on the previous stream may still read the context's scratch, which the
      // next call (ordered on the new stream only) may overwrite or regrow.
      DeviceGuard g(ctx->device);
      ctx->scratch.release();  // freed on the stream that used it; the next call allocates on the new one
      MG_HIP(hipStreamSynchronize(ctx->stream));
    }
    ctx->stream = next;
  });
}

extern "C" int mg_context_synchronize(mg_context* ctx) {
  return guarded([&] {
    MG_REQUIRE(ctx != nullptr, "mg_context_synchronize: ctx is NULL");
    DeviceGuard g(ctx->device);
    MG_HIP(hipStreamSynchronize(ctx->stream));
  });
}

extern "C" int mg_context_device(const mg_context* ctx, int* device, int* n_compute_units) {
  return guarded([&] {
    MG_REQUIRE(ctx != nullptr, "mg_context_device: ctx is NULL");
    if (device) *device = ctx->device;
    if (n_compute_units) *n_compute_units = ctx->n_cu;
  });
}

// Floyd's algorithm (Bentley & Floyd, "Programming pearls: a sample of
// brilliance", CACM 1987): for j = n-count .. n-1 draw r in [0, j]; take r unless
// already taken, else take j. Draw i uses SplitMix64 counter i of the
// "sources" stream; r = (draw >> 11) % (j+1).
extern "C" int mg_sample_sources(uint32_t n_vertices, uint32_t count, uint64_t seed, uint32_t* out) {
  return guarded([&] {
    MG_REQUIRE(out != nullptr || count == 0, "mg_sample_sources: out is NULL");
    MG_REQUIRE(count <= n_vertices, "mg_sample_sources: count exceeds n_vertices");
    const uint64_t key = stream_key(seed, kTagSources);
    std::unordered_set<uint32_t> taken;
    taken.reserve(count * 2 + 1);
    uint32_t k = 0;
    for (uint64_t j = static_cast<uint64_t>(n_vertices) - count; j < n_vertices; ++j, ++k) {
      const uint64_t r = (sm64_at(key, k) >> 11) % (j + 1);
      const uint32_t pick = taken.count(static_cast<uint32_t>(r)) ? static_cast<uint32_t>(j)
                                                                   : static_cast<uint32_t>(r);
      taken.insert(pick);
      out[k] = pick;
    }
  });
}

extern "C" int mg_context_stream(const mg_context* ctx, void** stream) {
  return guarded([&] {
    MG_REQUIRE(ctx && stream, "mg_context_stream: NULL argument");
    *stream = ctx->stream;
  });
}

extern "C" int mg_buffer_alloc(mg_context* ctx, size_t bytes, void** dptr) {
  return guarded([&] {
    MG_REQUIRE(ctx && dptr, "mg_buffer_alloc: NULL argument");
    *dptr = nullptr;
    DeviceGuard g(ctx->device);
    void* p = cached_alloc(bytes ? bytes : 1);
    hipError_t e = hipMemsetAsync(p, 0, bytes ? bytes : 1, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
      cached_free(p);
      MG_HIP(e);
    }
    *dptr = p;
  });
}

extern "C" int mg_buffer_free(mg_context* ctx, void* dptr) {
  return guarded([&] {
    MG_REQUIRE(ctx != nullptr, "mg_buffer_free: NULL ctx");
    if (!dptr) return;
    DeviceGuard g(ctx->device);
    MG_HIP(hipStreamSynchronize(ctx->stream));
    cached_free(dptr);
  });
}

extern "C" int mg_buffer_upload(mg_context* ctx, void* dptr, const void* host, size_t bytes) {
  return guarded([&] {
    MG_REQUIRE(ctx && dptr && (host || bytes == 0), "mg_buffer_upload: NULL argument");
    DeviceGuard g(ctx->device);
    if (bytes) MG_HIP(hipMemcpyAsync(dptr, host, bytes, hipMemcpyHostToDevice, ctx->stream));
    MG_HIP(hipStreamSynchronize(ctx->stream));
  });
}

extern "C" int mg_buffer_download(mg_context* ctx, void* host, const void* dptr, size_t bytes) {
  return guarded([&] {
    MG_REQUIRE(ctx && dptr && (host || bytes == 0), "mg_buffer_download: NULL argument");
    DeviceGuard g(ctx->device);
    if (bytes) MG_HIP(hipMemcpyAsync(host, dptr, bytes, hipMemcpyDeviceToHost, ctx->stream));
    MG_HIP(hipStreamSynchronize(ctx->stream));
  });
}

extern "C" int mg_buffer_copy(mg_context* ctx, void* dst, const void* src, size_t bytes) {
  return guarded([&] {
    MG_REQUIRE(ctx && dst && src, "mg_buffer_copy: NULL argument");
    DeviceGuard g(ctx->device);
    if (bytes) MG_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
  });
}

extern "C" int mg_context_timer_start(mg_context* ctx) {
  return guarded([&] {
    MG_REQUIRE(ctx != nullptr, "mg_context_timer_start: ctx is NULL");
    DeviceGuard g(ctx->device);
    for (hipEvent_t& e : ctx->timer)
      if (!e) MG_HIP(hipEventCreate(&e));
    MG_HIP(hipEventRecord(ctx->timer[0], ctx->stream));
  });
}

extern "C" int mg_context_timer_stop(mg_context* ctx, double* ms) {
  return guarded([&] {
    MG_REQUIRE(ctx && ms, "mg_context_timer_stop: NULL argument");
    MG_REQUIRE(ctx->timer[0] && ctx->timer[1], "mg_context_timer_stop: timer not started");
    DeviceGuard g(ctx->device);
    MG_HIP(hipEventRecord(ctx->timer[1], ctx->stream));
    MG_HIP(hipEventSynchronize(ctx->timer[1]));
    float t = 0;
    MG_HIP(hipEventElapsedTime(&t, ctx->timer[0], ctx->timer[1]));
    *ms = t;
  });
}
