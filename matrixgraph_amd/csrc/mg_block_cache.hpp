// Device memory blocks kept between objects (cached_alloc and cached_free of mg_internal.hpp say what
// for). The driver's calls come from D, so that a host test can run the bookkeeping against a driver of
// its own:
//   Status, kOk, kOutOfMemory, kInvalid;
//   malloc(void**, bytes), free(void*), current_device(int*): Status;
//   Stream, pool_malloc(void**, bytes, Stream): Status, from the temporaries' pool;
//   wait(): waits as free does, false if that failed; settle(Stream): waits for the stream, false if it
//   may not (a capture); trim(device): the pool gives back what it does not use.
#pragma once

#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>

namespace mgamd {

// Frees of this thread inside a FreeScope share one wait.
inline thread_local int g_free_depth = 0;        // scopes of this thread
inline thread_local bool g_free_waited = false;  // the outermost scope has waited already
struct FreeScope {
  FreeScope() {
    if (g_free_depth++ == 0) g_free_waited = false;
  }
  ~FreeScope() { --g_free_depth; }
  FreeScope(const FreeScope&) = delete;
  FreeScope& operator=(const FreeScope&) = delete;
};

template <class D>
class BlockCache {
 public:
  using Status = typename D::Status;

  void add_context(int device, size_t device_bytes) {
    std::lock_guard<std::mutex> lock(mu_);
    Device& d = devices_[device];
    ++d.contexts;
    d.limit = device_bytes / 64;
  }

  void drop_context(int device) noexcept {
    {
      std::lock_guard<std::mutex> lock(mu_);
      if (--devices_[device].contexts) return;
    }
    give_back(device);
  }

  // A kept block of at least `bytes`, and at most an eighth more, or a fresh one. On the current device.
  Status alloc(size_t bytes, void** out) {
    *out = nullptr;
    if (bytes > SIZE_MAX - 511) return D::kOutOfMemory;  // rounding up would wrap to nothing
    bytes = (bytes + 511) / 512 * 512;
    int device = 0;
    Status e = D::current_device(&device);
    if (e != D::kOk) return e;
    {
      std::lock_guard<std::mutex> lock(mu_);
      Device& d = devices_[device];
      auto it = d.kept.lower_bound(bytes);
      if (it != d.kept.end() && it->first <= bytes + bytes / 8) {
        void* const p = it->second.ptr;
        live_[p] = Live{it->first, device};
        d.bytes -= it->first;
        d.kept.erase(it);
        *out = p;
        return D::kOk;
      }
    }
    void* p = nullptr;
    e = D::malloc(&p, bytes);
    if (e == D::kOutOfMemory) {
      (void)D::wait();  // frees that are queued on streams
      give_back(device);
      e = D::malloc(&p, bytes);
    }
    if (e != D::kOk) return e;
    try {
      std::lock_guard<std::mutex> lock(mu_);
      live_[p] = Live{bytes, device};
    } catch (...) {
      (void)D::free(p);
      throw;
    }
    *out = p;
    return D::kOk;
  }

  // Keeps the block or gives it to the driver, whose answer is returned: a pointer that alloc has not
  // handed out is the driver's to judge, except a kept block, which is refused (freed twice): the
  // driver would take it back while it may still be handed out.
  Status free(void* p) noexcept {
    if (!p) return D::kOk;
    Live l{0, -1};
    bool keep = false;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = live_.find(p);
      if (it == live_.end()) {
        for (const auto& d : devices_)
          for (const auto& b : d.second.kept)
            if (b.second.ptr == p) return D::kInvalid;
      } else {
        l = it->second;
        live_.erase(it);
        const auto d = devices_.find(l.device);
        keep = d != devices_.end() && d->second.contexts > 0 && l.bytes <= d->second.limit / 2;
      }
    }
    int current = -1;
    if (keep && (D::current_device(&current) != D::kOk || current != l.device)) keep = false;
    if (keep && !(g_free_depth > 0 && g_free_waited)) {
      keep = D::wait();
      if (keep && g_free_depth > 0) g_free_waited = true;
    }
    if (keep) {
      try {
        std::lock_guard<std::mutex> lock(mu_);
        Device& d = devices_[l.device];
        keep = d.contexts > 0;  // the last context may have gone since
        if (keep) {
          d.kept.emplace(l.bytes, Kept{p, d.next_age++});
          d.bytes += l.bytes;
        }
      } catch (...) {
        keep = false;
      }
    }
    if (!keep) return D::free(p);
    // Over the limit: the oldest blocks go back to the driver.
    for (;;) {
      void* old = nullptr;
      {
        std::lock_guard<std::mutex> lock(mu_);
        Device& d = devices_[l.device];
        if (d.bytes <= d.limit || d.kept.empty()) return D::kOk;
        auto oldest = d.kept.begin();
        for (auto it = d.kept.begin(); it != d.kept.end(); ++it)
          if (it->second.age < oldest->second.age) oldest = it;
        old = oldest->second.ptr;
        d.bytes -= oldest->first;
        d.kept.erase(oldest);
      }
      (void)D::free(old);
    }
  }

  // A temporary from the pool, on the current device.
  Status pool_alloc(size_t bytes, typename D::Stream stream, void** out) {
    *out = nullptr;
    Status e = D::pool_malloc(out, bytes, stream);
    if (e != D::kOutOfMemory) return e;
    int device = 0;
    if (!D::settle(stream) || D::current_device(&device) != D::kOk) return e;
    give_back(device);
    return D::pool_malloc(out, bytes, stream);
  }

  // What the library holds on the device without using it, back to the driver.
  void give_back(int device) noexcept {
    flush(device);
    D::trim(device);
  }

  // Every kept block of the device back to the driver.
  void flush(int device) noexcept {
    std::multimap<size_t, Kept> out;
    {
      std::lock_guard<std::mutex> lock(mu_);
      auto it = devices_.find(device);
      if (it == devices_.end()) return;
      out.swap(it->second.kept);
      it->second.bytes = 0;
    }
    for (auto& b : out) (void)D::free(b.second.ptr);
  }

 private:
  struct Kept {
    void* ptr;
    uint64_t age;
  };
  struct Device {
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
  std::mutex mu_;
  std::unordered_map<void*, Live> live_;  // blocks handed out
  std::unordered_map<int, Device> devices_;
};

}  // namespace mgamd
