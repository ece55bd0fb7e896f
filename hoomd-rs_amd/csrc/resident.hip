// Launches of the persistent applies, whose workgroups wait for one another and
// so must all be resident together.
//
// Their number fits the device by the occupancy API and by a probe with the
// kernel itself, so nothing that ends by itself can keep them out for good; only
// two such launches at once could, each holding what the other waits for.  A
// cooperative launch excludes that by waiting on the host for the stream before
// and after it: 20 us per launch, of the 71 of an apply of 16,384 disks.  Here
// they are ordinary launches, and
//  - in a process, one on another stream than the device's last first waits, on the
//    device, for that stream's work;
//  - between processes, a stream is in flight from its first persistent launch until
//    the host has waited for it, and while a process has streams in flight it holds
//    the device's lock (a record lock of the driver's device file: every process that
//    can use the device can open it).  One that launches many applies looks every
//    kLooks launches whether another waits, and then lets its work end and queues
//    behind it.  Four system calls per call of the library, 0.3 us of the 74 of an apply
//    of 1,024 disks.
// Measured us per apply, cooperative and so: 16,384 disks 70.8 and 50.7, 4,000
// spheres 164 and 144, 1,000,188 253 and 234, 131,072 overlap-penalty bodies 274
// and 252, 524,288 LJ bodies 1460 and 1429.
#include <algorithm>
#include <condition_variable>
#include <cstdio>

#include "host.hpp"
#include "turnstile.hpp"

namespace hmc {

namespace {
constexpr int kDevices = 64;
constexpr uint32_t kLooks = 16;
struct Gate {
  std::mutex use;
  std::condition_variable change;
  Turnstile turn;
  int usable = -1;                     // the lock: not opened yet, no, yes
  bool entering = false;               // a thread waits for the lock
  std::vector<hipStream_t> in_flight;  // holding the lock while there are any
  uint32_t launches = 0;
  hipStream_t last = nullptr;  // the stream of the last persistent launch
  hipEvent_t ev = nullptr;     // (made at the first change of streams)
};
Gate* gate_of(int device) {
  static Gate* g = new (std::nothrow) Gate[kDevices];  // (outlives every context)
  return g && device >= 0 && device < kDevices ? g + device : nullptr;
}

bool open_lock(Gate& g, int device) {
  if (g.usable < 0) {
    char id[32] = {};
    unsigned domain = 0, bus = 0, dev = 0, fn = 0;
    g.usable = hipDeviceGetPCIBusId(id, sizeof id, device) == hipSuccess &&
                       std::sscanf(id, "%x:%x:%x.%x", &domain, &bus, &dev, &fn) >= 3 &&
                       g.turn.open("/dev/kfd", ((uint64_t)domain << 16) | (bus << 8) | (dev << 3) | fn)
                   ? 1
                   : 0;
  }
  return g.usable == 1;
}

void drop(Gate& g, hipStream_t s) {
  auto it = std::find(g.in_flight.begin(), g.in_flight.end(), s);
  if (it == g.in_flight.end()) return;
  g.in_flight.erase(it);
  if (g.in_flight.empty()) g.turn.leave();
  g.change.notify_all();
}

// Stream s in flight, once it is this process's turn.
hipError_t join(Gate& g, std::unique_lock<std::mutex>& lock, hipStream_t s) {
  if (std::find(g.in_flight.begin(), g.in_flight.end(), s) != g.in_flight.end()) {
    if (++g.launches % kLooks != 0 || !g.turn.wanted()) return hipSuccess;
    lock.unlock();
    const hipError_t e = hipStreamSynchronize(s);
    lock.lock();
    if (e != hipSuccess) return e;
    drop(g, s);
  }
  for (;;) {
    if (g.entering || (!g.in_flight.empty() && g.turn.wanted())) {
      g.change.wait(lock);  // (the streams in flight leave at their next look, or at their ends)
    } else if (!g.in_flight.empty()) {
      break;
    } else {
      g.entering = true;
      lock.unlock();
      const bool got = g.turn.enter();
      lock.lock();
      g.entering = false;
      g.change.notify_all();
      if (!got) return hipErrorNotSupported;
      break;
    }
  }
  g.in_flight.push_back(s);
  return hipSuccess;
}
}  // namespace

hipError_t launch_resident(int device, const void* fn, uint32_t blocks, uint32_t threads, void** args, size_t lds,
                           hipStream_t s) {
  Gate* g = gate_of(device);
  if (!g) return hipErrorInvalidDevice;
  std::unique_lock<std::mutex> lock(g->use);
  if (!open_lock(*g, device)) return hipErrorNotSupported;
  hipError_t e = join(*g, lock, s);
  if (e == hipSuccess && g->last && g->last != s) {
    if (!g->ev) e = hipEventCreateWithFlags(&g->ev, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(g->ev, g->last);
    if (e == hipSuccess) e = hipStreamWaitEvent(s, g->ev, 0);
  }
  if (e == hipSuccess) e = hipLaunchKernel(fn, dim3(blocks), dim3(threads), args, lds, s);
  if (e == hipSuccess) g->last = s;
  return e;
}

void settled_resident(int device, hipStream_t s) {
  Gate* g = gate_of(device);
  if (!g) return;
  std::lock_guard<std::mutex> lock(g->use);
  drop(*g, s);
}

ResidentCall::~ResidentCall() {
  Gate* g = gate_of(device);
  if (!g) return;
  std::unique_lock<std::mutex> lock(g->use);
  if (std::find(g->in_flight.begin(), g->in_flight.end(), s) == g->in_flight.end()) return;
  lock.unlock();
  (void)hipStreamSynchronize(s);
  lock.lock();
  drop(*g, s);
}

void forget_resident(int device, hipStream_t s) {
  Gate* g = gate_of(device);
  if (!g) return;
  std::lock_guard<std::mutex> lock(g->use);
  drop(*g, s);
  if (g->last != s) return;
  if (g->ev) (void)hipEventDestroy(g->ev);
  g->ev = nullptr;
  g->last = nullptr;
}

bool resident_order(int device) {
  Gate* g = gate_of(device);
  if (!g) return false;
  std::lock_guard<std::mutex> lock(g->use);
  return g->last != nullptr;
}

}  // namespace hmc

extern "C" int hmc_debug_turn(const char* path, uint64_t key, int op) {
  static Turnstile* t = nullptr;
  if (op == 0) {
    delete t;
    t = new (std::nothrow) Turnstile;
    return t && t->open(path, key) ? 1 : 0;
  }
  if (!t) return 0;
  if (op == 1) return t->enter() ? 1 : 0;
  if (op == 2) t->leave();
  return op == 3 && t->wanted() ? 1 : 0;
}
