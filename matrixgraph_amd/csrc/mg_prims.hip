// Setup-path primitives: scans and sorts (hipCUB), popcount reduction.
// None of these run inside a walk hop; they build indices and inputs.
#include <cstring>

#include <hipcub/hipcub.hpp>

#include "mg_device.hpp"
#include "mg_internal.hpp"

namespace mgamd {

namespace {

__global__ void __launch_bounds__(256) popcount_kernel(const uint64_t* __restrict__ data, uint64_t n,
                                                       unsigned long long* __restrict__ out) {
  uint64_t local = 0;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
    local += __popcll(data[i]);
  local = wave_sum(local);
  if (lane_id() == 0 && local) atomicAdd(out, static_cast<unsigned long long>(local));
}

__global__ void __launch_bounds__(256) sum_u32_kernel(const uint32_t* __restrict__ data, uint64_t n,
                                                      unsigned long long* __restrict__ out) {
  uint64_t local = 0;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) local += data[i];
  local = wave_sum(local);
  if (lane_id() == 0 && local) atomicAdd(out, static_cast<unsigned long long>(local));
}

__global__ void __launch_bounds__(kWave) read_words_kernel(const uint32_t* a, uint32_t n_a, const uint32_t* b,
                                                           uint32_t n_b, uint32_t* __restrict__ mail) {
  const uint32_t i = threadIdx.x;
  if (i < n_a) mail[i] = a[i];
  if (i >= n_a && i < n_a + n_b) mail[i] = b[i - n_a];
}

}  // namespace

void read_words(mg_context* ctx, DeviceWords a, DeviceWords b) {
  const uint32_t n_a = a.bytes / 4, n_b = b.bytes / 4;
  if (a.bytes % 4 || b.bytes % 4 || n_a + n_b > kMailWords) fail(MG_ERR_INTERNAL, "read_words: size");
  read_words_kernel<<<1, kWave, 0, ctx->stream>>>(static_cast<const uint32_t*>(a.from), n_a,
                                                  static_cast<const uint32_t*>(b.from), n_b, ctx->mail.get());
  MG_LAUNCH_CHECK();
  MG_HIP(hipStreamSynchronize(ctx->stream));
  std::memcpy(a.to, ctx->mail.get(), a.bytes);
  if (b.bytes) std::memcpy(b.to, ctx->mail.get() + n_a, b.bytes);
}

uint64_t device_popcount(mg_context* ctx, const uint64_t* data, uint64_t n_words) {
  unsigned long long* d = ctx->counters.get();
  MG_HIP(hipMemsetAsync(d, 0, sizeof(unsigned long long), ctx->stream));
  if (n_words) {
    popcount_kernel<<<grid_for(n_words, 256 * 16, 8192), 256, 0, ctx->stream>>>(data, n_words, d);
    MG_LAUNCH_CHECK();
  }
  unsigned long long h = 0;
  read_words(ctx, {d, &h, sizeof(h)});
  return h;
}

uint64_t device_sum_u32(mg_context* ctx, const uint32_t* data, uint64_t n) {
  unsigned long long* d = ctx->counters.get();
  MG_HIP(hipMemsetAsync(d, 0, sizeof(unsigned long long), ctx->stream));
  if (n) {
    sum_u32_kernel<<<grid_for(n, 256 * 16, 8192), 256, 0, ctx->stream>>>(data, n, d);
    MG_LAUNCH_CHECK();
  }
  unsigned long long h = 0;
  read_words(ctx, {d, &h, sizeof(h)});
  return h;
}

void exclusive_scan_u32_on(hipStream_t st, const uint32_t* in, uint32_t* out, uint32_t n) {
  // out[0..n-1] = exclusive prefix, out[n] = total: scan n+1 items with a zero appended
  // is avoided by scanning n items then adding the last count on device.
  size_t temp_bytes = 0;
  MG_HIP(hipcub::DeviceScan::InclusiveSum(nullptr, temp_bytes, in, out + 1, n, st));
  StreamBuf<uint8_t> temp(temp_bytes, st);
  MG_HIP(hipMemsetAsync(out, 0, sizeof(uint32_t), st));
  if (n) MG_HIP(hipcub::DeviceScan::InclusiveSum(temp.get(), temp_bytes, in, out + 1, n, st));
}

void exclusive_scan_u32(mg_context* ctx, const uint32_t* in, uint32_t* out, uint32_t n) {
  exclusive_scan_u32_on(ctx->stream, in, out, n);
}

size_t sort_u64_bytes(uint64_t n, int begin_bit, int end_bit) {
  size_t bytes = 0;
  hipcub::DoubleBuffer<uint64_t> db(nullptr, nullptr);
  MG_HIP(hipcub::DeviceRadixSort::SortKeys(nullptr, bytes, db, static_cast<int>(n), begin_bit, end_bit));
  return bytes;
}

uint64_t* sort_u64(hipStream_t st, uint64_t* keys, uint64_t* alt, uint64_t n, int begin_bit, int end_bit, void* temp,
                   size_t temp_bytes) {
  hipcub::DoubleBuffer<uint64_t> db(keys, alt);
  MG_HIP(hipcub::DeviceRadixSort::SortKeys(temp, temp_bytes, db, static_cast<int>(n), begin_bit, end_bit, st));
  return db.Current();
}

// One workgroup. A thread's entries in 16-byte loads, all in flight (one load at a time: 111 us for
// 65536 entries).
constexpr uint32_t kScanBlock = 1024;
static __global__ void __launch_bounds__(kScanBlock) scan_in_place_kernel(uint32_t* __restrict__ v, uint32_t n) {
  __shared__ uint32_t s_sum[kScanBlock / kWave];
  const uint32_t per = (n + 4 * kScanBlock - 1) / (4 * kScanBlock) * 4;
  const uint32_t lo = min(n, threadIdx.x * per), hi = min(n, lo + per);
  uint32_t sum = 0;
#pragma unroll 8
  for (uint32_t i = lo; i + 4 <= hi; i += 4) {
    const uint4 q = *reinterpret_cast<const uint4*>(v + i);
    sum += q.x + q.y + q.z + q.w;
  }
  for (uint32_t i = lo + (hi - lo) / 4 * 4; i < hi; ++i) sum += v[i];
  uint32_t incl = sum;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t o = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), d, kWave));
    if (lane_id() >= static_cast<uint32_t>(d)) incl += o;
  }
  if (lane_id() == kWave - 1) s_sum[threadIdx.x / kWave] = incl;
  __syncthreads();
  uint32_t at = incl - sum;
  for (uint32_t w = 0; w < threadIdx.x / kWave; ++w) at += s_sum[w];
#pragma unroll 8
  for (uint32_t i = lo; i + 4 <= hi; i += 4) {
    const uint4 q = *reinterpret_cast<const uint4*>(v + i);
    *reinterpret_cast<uint4*>(v + i) = make_uint4(at, at + q.x, at + q.x + q.y, at + q.x + q.y + q.z);
    at += q.x + q.y + q.z + q.w;
  }
  for (uint32_t i = lo + (hi - lo) / 4 * 4; i < hi; ++i) {
    const uint32_t c = v[i];
    v[i] = at;
    at += c;
  }
  if (threadIdx.x == kScanBlock - 1) v[n] = at;
}

void scan_in_place(hipStream_t st, uint32_t* v, uint32_t n) {
  scan_in_place_kernel<<<1, kScanBlock, 0, st>>>(v, n);
  MG_LAUNCH_CHECK();
}

}  // namespace mgamd
