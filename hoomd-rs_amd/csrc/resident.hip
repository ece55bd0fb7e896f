// Launches of the persistent applies, whose workgroups wait for one another and
// so must all be resident together.
//
// Their number fits the device by the occupancy API and by a probe with the
// kernel itself, so nothing that ends by itself can keep them out for good; only
// two such launches at once could, each holding what the other waits for.  A
// cooperative launch excludes that by waiting on the host for the stream before
// and after it: 20 us per launch, of the 71 of an apply of 16,384 disks.  Here
// they are ordinary launches, and one on another stream than the device's last
// first waits, on the device, for that stream's work.
// Measured us per apply, cooperative and so: 16,384 disks 70.8 and 50.7, 4,000
// spheres 164 and 144, 1,000,188 253 and 234, 131,072 overlap-penalty bodies 274
// and 252, 524,288 LJ bodies 1460 and 1429.
#include <map>

#include "host.hpp"

namespace hmc {

namespace {
struct Gate {
  hipStream_t last = nullptr;  // the stream of the device's last persistent launch
  hipEvent_t ev = nullptr;     // (made at the first change of streams)
};
std::mutex gates_use;
std::map<int, Gate>& gates() {
  static std::map<int, Gate>* g = new std::map<int, Gate>;  // (outlives every context)
  return *g;
}
}  // namespace

hipError_t launch_resident(int device, const void* fn, uint32_t blocks, uint32_t threads, void** args, size_t lds,
                           hipStream_t s) {
  std::lock_guard<std::mutex> lock(gates_use);
  Gate& g = gates()[device];
  hipError_t e = hipSuccess;
  if (g.last && g.last != s) {
    if (!g.ev) e = hipEventCreateWithFlags(&g.ev, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(g.ev, g.last);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, g.ev, 0);
    if (e != hipSuccess) return e;
  }
  e = hipLaunchKernel(fn, dim3(blocks), dim3(threads), args, lds, s);
  if (e == hipSuccess) g.last = s;
  return e;
}

void forget_resident(int device, hipStream_t s) {
  std::lock_guard<std::mutex> lock(gates_use);
  auto it = gates().find(device);
  if (it == gates().end() || it->second.last != s) return;
  if (it->second.ev) (void)hipEventDestroy(it->second.ev);
  gates().erase(it);
}

bool resident_order(int device) {
  std::lock_guard<std::mutex> lock(gates_use);
  auto it = gates().find(device);
  return it != gates().end() && it->second.last;
}

}  // namespace hmc
