// Reads of device state by the host: positions, orientations, the apply state.
//
// A copy into ordinary memory goes through the runtime's own staging (10 GB/s),
// as 32 bytes per body and side into fresh arrays that were cleared, copied from
// component by component and given back.  Here a kernel packs the components
// that are asked for straight into pinned memory, a chunk at a time, and the
// host copies each chunk to the caller while the next one arrives.
// Measured: a read of the positions of 1,000,188 spheres 18.4 and 2.9 ms, of
// the 256 replicas of a batch (4.1 million bodies) 32.5 and 16.0, of 1,024 disks 47
// and 17 us; an apply of 1,024 disks with its positions 190 and 117 us (three reads).
// Chunks of 0.5 MiB are as good, of 128 KiB 1.6 times slower.  Bound by the
// host's copy into pages it touches for the first time (12 GB/s).
#include "host.hpp"

namespace hmc {

// Words first .. first + n of the concatenation of two arrays of `rows` rows of
// `width` words, each row at the head of `stride` words in the source.
__global__ void __launch_bounds__(256) k_pack(const unsigned long long* a, const unsigned long long* b, uint32_t stride,
                                              uint32_t width, uint64_t rows, uint64_t first, uint32_t n,
                                              unsigned long long* out) {
  const uint64_t per = rows * width;
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
    uint64_t e = first + i;
    const unsigned long long* src = a;
    if (e >= per) {
      e -= per;
      src = b;
    }
    out[i] = src[e / width * stride + e % width];
  }
}

// The apply state, with the accepted moves summed over their counters.
__global__ void __launch_bounds__(kAccSlots) k_pack_state(const ApplyState* st, const unsigned long long* acc_slots,
                                                          ApplyState* out) {
  __shared__ unsigned long long sum;
  if (threadIdx.x == 0) sum = 0;
  __syncthreads();
  const unsigned long long v = acc_slots[threadIdx.x];
  if (v) atomicAdd(&sum, v);
  constexpr uint32_t words = sizeof(ApplyState) / 8;
  static_assert(sizeof(ApplyState) % 8 == 0 && words <= kAccSlots, "one word per thread");
  if (threadIdx.x < words) ((unsigned long long*)out)[threadIdx.x] = ((const unsigned long long*)st)[threadIdx.x];
  __syncthreads();
  if (threadIdx.x == 0) out->accepted_total = sum;
}

hipError_t Readback::init(uint64_t largest) {
  chunk = (std::min<uint64_t>(kChunkWords, std::max<uint64_t>(largest, sizeof(ApplyState) / 8)) + 511) / 512 * 512;
  hipError_t e = hipHostMalloc((void**)&host, 2 * chunk * 8);
  if (e == hipSuccess) e = hipHostGetDevicePointer((void**)&dev, host, 0);
  for (hipEvent_t& v : done)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
  return e;
}

Readback::~Readback() {
  for (hipEvent_t v : done)
    if (v) (void)hipEventDestroy(v);
  if (host) (void)hipHostFree(host);
}

hipError_t Readback::state(const ApplyState* st, const unsigned long long* acc_slots, ApplyState* out, hipStream_t s) {
  std::lock_guard<std::mutex> lock(use);
  k_pack_state<<<1, kAccSlots, 0, s>>>(st, acc_slots, (ApplyState*)dev);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e == hipSuccess) std::memcpy(out, host, sizeof(ApplyState));
  return e;
}

// (the wait of an earlier chunk's copy is the host's own program order: chunk k
// is launched into the half that chunk k - 2 was copied from)
hipError_t Readback::read(const void* a, const void* b, uint32_t stride, uint32_t width, uint64_t rows, void* out_a,
                          void* out_b, hipStream_t s) {
  std::lock_guard<std::mutex> lock(use);
  if (!out_a) {
    a = b;
    out_a = out_b;
    out_b = nullptr;
  }
  const uint64_t per = rows * width, total = out_b ? 2 * per : (out_a ? per : 0), chunks = (total + chunk - 1) / chunk;
  auto launch = [&](uint64_t k) {
    const uint32_t n = (uint32_t)std::min<uint64_t>(chunk, total - k * chunk);
    k_pack<<<std::min<uint32_t>(grid_for(n, 256), 1024), 256, 0, s>>>(
        (const unsigned long long*)a, (const unsigned long long*)b, stride, width, rows, k * chunk, n,
        dev + (k & 1) * chunk);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? hipEventRecord(done[k & 1], s) : e;
  };
  hipError_t e = chunks ? launch(0) : hipStreamSynchronize(s);
  for (uint64_t k = 0; k < chunks && e == hipSuccess; ++k) {
    if (k + 1 < chunks) e = launch(k + 1);
    if (e == hipSuccess) e = hipEventSynchronize(done[k & 1]);
    if (e != hipSuccess) break;
    const uint64_t w0 = k * chunk, w1 = std::min<uint64_t>(w0 + chunk, total), mid = std::min(std::max(per, w0), w1);
    const unsigned long long* src = host + (k & 1) * chunk;
    std::memcpy((unsigned long long*)out_a + w0, src, (mid - w0) * 8);
    if (w1 > mid) std::memcpy((unsigned long long*)out_b + (mid - per), src + (mid - w0), (w1 - mid) * 8);
  }
  // (a failure leaves nothing in flight into the pinned memory)
  if (e != hipSuccess) (void)hipStreamSynchronize(s);
  return e;
}

}  // namespace hmc
