// Copies between pageable host arrays and the device.
//
// The runtime moves pageable memory through its own staging with one thread; a fresh host
// array also takes its page faults in that thread. Here the copy is cut into chunks that
// pass through pinned slots, one chunk crossing the link (move_kernel) while the pool's threads
// copy others between the slots and the caller's array.
//
// Bound: the link (57 GB/s each way from pinned memory) and the threads' page faults. Measured,
// runtime and here (GB/s): down 5 MiB 17.6 and 39, 20 MiB 17.6 and 42, 200 MiB 17.5 and 48.6; down
// into a fresh array of 200 MiB 10.5 and 19.7; up 8 MiB 34.5 and 43, 64 MiB 29.2 and 47.9. Copies of up
// to 4 MiB stay with the runtime: what is gained goes into waking the threads there (a lone
// 0.6 MiB download took 50 µs and 130).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <vector>

#include "host.h"
#include "hostpool.h"

namespace vh {
namespace {

constexpr size_t kChunk = (size_t)2 << 20;   // bytes per slot
constexpr size_t kPiece = (size_t)128 << 10; // bytes per thread at a time
constexpr int kSlots = 16;                   // pinned slots of the process (32 MiB)
constexpr int kSlotsPerCopy = 4;
constexpr int kMoveWgs = 32;                 // workgroups of move_kernel
// Copies of at most this many bytes go to the runtime.
constexpr size_t kDirect = (size_t)4 << 20;

// A slot's event belongs to the device it was made on.
struct Slot {
  char* mem = nullptr;
  hipEvent_t ev = nullptr;
  int device = -1;
};

// Slots are taken by a copy and given back at its end; a copy that finds none waits for one.
class SlotPool {
 public:
  std::vector<Slot> take(int want, int device) {
    std::vector<Slot> got;
    try {
      got.reserve(want);
      std::lock_guard<std::mutex> lk(mu_);
      free_.reserve(kSlots);
    } catch (const std::bad_alloc&) {
      return {};
    }
    std::unique_lock<std::mutex> lk(mu_);
    for (;;) {
      while ((int)got.size() < want && !free_.empty()) {
        got.push_back(free_.back());
        free_.pop_back();
      }
      while ((int)got.size() < want && made_ < kSlots) {
        void* p = nullptr;
        if (hipHostMalloc(&p, kChunk, hipHostMallocPortable) != hipSuccess) {
          (void)hipGetLastError();
          break;
        }
        ++made_;
        got.push_back(Slot{(char*)p, nullptr, -1});
      }
      if (!got.empty() || made_ == 0) break;
      cv_.wait(lk);
    }
    lk.unlock();
    for (size_t i = 0; i < got.size(); ++i) {
      Slot& s = got[i];
      if (s.device == device) continue;
      if (s.ev) (void)hipEventDestroy(s.ev);
      s.ev = nullptr;
      s.device = -1;
      if (hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) == hipSuccess) s.device = device;
    }
    return got;
  }
  void give_back(const std::vector<Slot>& slots) {
    std::lock_guard<std::mutex> lk(mu_);
    for (const Slot& s : slots) free_.push_back(s);
    cv_.notify_all();
  }

 private:
  std::mutex mu_;
  std::condition_variable cv_;
  std::vector<Slot> free_;
  int made_ = 0;
};
SlotPool& slot_pool() {
  static SlotPool* p = new SlotPool();   // never destroyed: copies may run while the process ends
  return *p;
}

void copy_pieces(char* dst, const char* src, size_t n) {
  try {
    HostPool::run_copies((int)((n + kPiece - 1) / kPiece), [&](int i) {
      const size_t o = (size_t)i * kPiece;
      memcpy(dst + o, src + o, std::min(kPiece, n - o));
    });
  } catch (const std::exception&) {   // the pool could not take the job (out of memory)
    memcpy(dst, src, n);
  }
}

// Ordinary host memory: what the runtime knows nothing of. Pinned, managed and device memory
// given as the host side is the runtime's to copy (a CPU copy could not read the last).
bool is_pageable(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// n bytes between a pinned slot and the device, 16 bytes per lane and pass (both 16-byte aligned).
// A kernel and not the runtime's copy, since that runs on an engine which the driver also
// clears freed device memory with: for some ms after a large free (a rollout's 860 MB) its
// downloads took 942 µs per 10 MiB against 266 at rest, the kernel's 234 and 232. Bound: the link;
// µs per 10 MiB by workgroups, down and up: 8: 247, 450; 16: 235, 252; 32: 232, 227; 128: 234, 236;
// 512: 226, 292.
typedef unsigned U4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) move_kernel(const char* __restrict__ src, char* __restrict__ dst, size_t n) {
  const size_t nv = n / 16, lane = (size_t)blockIdx.x * 256 + threadIdx.x;
  for (size_t i = lane; i < nv; i += (size_t)gridDim.x * 256)
    __builtin_nontemporal_store(__builtin_nontemporal_load((const U4*)src + i), (U4*)dst + i);
  if (lane < n % 16) dst[nv * 16 + lane] = src[nv * 16 + lane];
}

// Whether move_kernel may touch the bytes at p: an allocation of the device that holds them
// all, 16-byte aligned. Everything else, errors included, is left to the runtime.
bool kernel_moves(const void* p, size_t bytes, int device) {
  hipPointerAttribute_t a{};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if ((uintptr_t)p % 16 == 0 && hipPointerGetAttributes(&a, p) == hipSuccess && a.type == hipMemoryTypeDevice &&
      a.device == device && hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) == hipSuccess)
    return (size_t)((const char*)p - (const char*)base) + bytes <= size;
  (void)hipGetLastError();
  return false;
}

hipError_t staged(char* dst, const char* src, size_t bytes, bool up, hipStream_t s, int device,
                  const std::vector<Slot>& slots) {
  const size_t n = (bytes + kChunk - 1) / kChunk, ns = slots.size();
  const bool kernel = kernel_moves(up ? dst : src, bytes, device);
  auto len = [&](size_t c) { return std::min(kChunk, bytes - c * kChunk); };
  // chunk c across the link
  auto issue = [&](size_t c) {
    const Slot& sl = slots[c % ns];
    char* to = up ? dst + c * kChunk : sl.mem;
    const char* from = up ? sl.mem : src + c * kChunk;
    size_t count = len(c);
    void* args[] = {&from, &to, &count};
    hipError_t r = kernel ? hipLaunchKernel((const void*)move_kernel, dim3(kMoveWgs), dim3(256), args, 0, s)
                          : hipMemcpyAsync(to, from, count, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
    return r == hipSuccess ? hipEventRecord(sl.ev, s) : r;
  };
  hipError_t e = hipSuccess;
  if (up) {
    for (size_t c = 0; c < n && e == hipSuccess; ++c) {
      const Slot& sl = slots[c % ns];
      if (c >= ns) e = hipEventSynchronize(sl.ev);
      if (e != hipSuccess) break;
      copy_pieces(sl.mem, src + c * kChunk, len(c));
      e = issue(c);
    }
  } else {
    for (size_t c = 0; c < std::min(n, ns) && e == hipSuccess; ++c) e = issue(c);
    for (size_t c = 0; c < n && e == hipSuccess; ++c) {
      e = hipEventSynchronize(slots[c % ns].ev);
      if (e != hipSuccess) break;
      copy_pieces(dst + c * kChunk, slots[c % ns].mem, len(c));
      if (c + ns < n) e = issue(c + ns);
    }
  }
  const hipError_t es = hipStreamSynchronize(s);   // the slots are free again, whatever happened
  return e == hipSuccess ? es : e;
}

// The copy through the slots, complete on return; false where it is left to the runtime.
bool through_slots(void* dst, const void* src, size_t bytes, bool up, hipStream_t s, hipError_t* e) {
  int device = 0, stream_device = 0;
  if (bytes <= kDirect || HostPool::threads() <= 1 || hipGetDevice(&device) != hipSuccess) return false;
  // the slots' events are the current device's: a stream of another takes the plain copy
  if (!s || hipStreamGetDevice(s, &stream_device) != hipSuccess) stream_device = device;
  if (stream_device != device || !is_pageable(up ? src : dst)) return false;
  const size_t chunks = (bytes + kChunk - 1) / kChunk;
  std::vector<Slot> slots = slot_pool().take((int)std::min<size_t>(kSlotsPerCopy, chunks), device);
  bool usable = !slots.empty();
  for (const Slot& sl : slots) usable = usable && sl.device == device;
  if (usable) *e = staged((char*)dst, (const char*)src, bytes, up, s, device, slots);
  slot_pool().give_back(slots);
  return usable;
}

hipError_t host_copy(void* dst, const void* src, size_t bytes, bool up, hipStream_t s) {
  if (bytes == 0) return hipStreamSynchronize(s);
  hipError_t e = hipSuccess;
  if (through_slots(dst, src, bytes, up, s, &e)) return e;
  const hipMemcpyKind kind = up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  if (!s) return hipMemcpy(dst, src, bytes, kind);   // 1 KiB down 13 µs; queued and waited for, 22
  e = hipMemcpyAsync(dst, src, bytes, kind, s);
  const hipError_t es = hipStreamSynchronize(s);
  return e == hipSuccess ? es : e;
}

}  // namespace

hipError_t enqueue_up(void* dev, const void* host, size_t bytes, hipStream_t s) {
  hipError_t e = hipSuccess;
  return through_slots(dev, host, bytes, true, s, &e) ? e : hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
}
hipError_t copy_up(void* dev, const void* host, size_t bytes, hipStream_t s) { return host_copy(dev, host, bytes, true, s); }
hipError_t copy_down(void* host, const void* dev, size_t bytes, hipStream_t s) {
  return host_copy(host, dev, bytes, false, s);
}

}  // namespace vh
