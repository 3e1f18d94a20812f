// ckt_hostring.h -- pinned slots through which records stream between the
// caller's (pageable) memory and kernels that read or write them over PCIe.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstring>
#include <initializer_list>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "ckt_internal.h"

namespace ckt {

// While a kernel reads or writes one slot over the bus, host threads copy
// others: one core copies about 10 GB/s to or from pageable memory, the bus
// carries about 50.  One transfer at a time (the caller's lock).  Slots are
// allocated as large as they are first needed, kept, and freed with the ring:
// 16 of at most 2 MiB, two for each of eight threads, and three for transfers
// that one slot holds.  Where no pinned memory can be had a slot is device
// memory of the same size, filled and read with synchronous copies: slower, but
// a circuit can still be loaded and stored.
class HostRing {
 public:
  HostRing() = default;
  HostRing(const HostRing&) = delete;
  HostRing& operator=(const HostRing&) = delete;
  ~HostRing() {
    for (Slot& sl : slots_) {
      if (sl.busy) (void)hipEventSynchronize(sl.ev);
      (void)release(sl);
      if (sl.ev) (void)hipEventDestroy(sl.ev);
    }
  }

  // Copies `count` records of `size` bytes from `src` into slots and calls
  // launch(slot, first, n), which enqueues on `s` the kernel that reads them.
  // Returns once every launch is made (`src` is free then); a slot's kernel is
  // waited for where the slot is used again.
  template <class Launch>
  int in(const void* src, size_t size, uint32_t count, int device, hipStream_t s, Launch launch) {
    const Plan p(size, count);
    Slot* const own = slots_for(p);
    return team(p.workers, device, [&](int t) -> int {
      int side = 0;
      for (uint32_t c = (uint32_t)t; c < p.chunks; c += (uint32_t)p.workers, side ^= 1) {
        const uint32_t first = c * p.per, n = std::min(p.per, count - first);
        Slot& sl = own[2 * t + side];
        if (int st = acquire(sl, n * size)) return st;
        if (int st = write(sl, 0, (const char*)src + (size_t)first * size, n * size, s)) return st;
        if (hipError_t e = launch(sl.p, first, n)) return hip_fail(e, "reading records");
        if (int st = mark(sl, s)) return st;
      }
      return CKT_OK;
    });
  }

  // A part of a slot and the host memory it is copied from or to.
  struct Source {
    size_t at;
    const void* p;
    size_t bytes;
  };
  struct Sink {
    size_t at;
    void* p;
    size_t bytes;
  };

  // One slot of `bytes` (kSlotBytes at most): `parts` are copied into it, and
  // launch(slot) enqueues the kernel that reads it.
  template <class Launch>
  int put(size_t bytes, hipStream_t s, std::initializer_list<Source> parts, Launch launch) {
    Slot& sl = *small_slot();
    if (int st = acquire(sl, bytes)) return st;
    for (const Source& x : parts)
      if (int st = write(sl, x.at, x.p, x.bytes, s)) return st;
    if (hipError_t e = launch(sl.p)) return hip_fail(e, "reading records");
    return mark(sl, s);
  }

  // One slot of `bytes` (kSlotBytes at most): launch(slot) enqueues the kernel
  // that writes it, and `parts` are copied from it when that has run.
  template <class Launch>
  int get(size_t bytes, hipStream_t s, Launch launch, std::initializer_list<Sink> parts) {
    Slot& sl = *small_slot();
    if (int st = acquire(sl, bytes)) return st;
    if (hipError_t e = launch(sl.p)) return hip_fail(e, "writing records");
    if (int st = mark(sl, s)) return st;
    if (int st = wait(sl)) return st;
    for (const Sink& x : parts)
      if (int st = read(sl, x.at, x.p, x.bytes, s)) return st;
    return CKT_OK;
  }

  // `bytes` (kSlotBytes at most) of pinned memory until the next call here, or
  // NULL if there is none.
  void* pinned(size_t bytes) {
    Slot& sl = *small_slot();
    return acquire(sl, bytes) == CKT_OK && sl.pinned ? sl.p : nullptr;
  }

  // Calls launch(slot, first, n) for the kernels that write records into
  // slots on `s`, and copies each slot to `dst` when its kernel has run.
  // Returns when all records are there.
  template <class Launch>
  int out(void* dst, size_t size, uint32_t count, int device, hipStream_t s, Launch launch) {
    const Plan p(size, count);
    Slot* const own = slots_for(p);
    return team(p.workers, device, [&](int t) -> int {
      auto begin = [&](uint32_t c, int side) -> int {
        if (c >= p.chunks) return CKT_OK;
        const uint32_t first = c * p.per, n = std::min(p.per, count - first);
        Slot& sl = own[2 * t + side];
        if (int st = acquire(sl, n * size)) return st;
        if (hipError_t e = launch(sl.p, first, n)) return hip_fail(e, "writing records");
        return mark(sl, s);
      };
      int side = 0;
      int st = begin((uint32_t)t, side);
      for (uint32_t c = (uint32_t)t; !st && c < p.chunks; c += (uint32_t)p.workers, side ^= 1) {
        if ((st = begin(c + (uint32_t)p.workers, side ^ 1))) break;
        Slot& sl = own[2 * t + side];
        if ((st = wait(sl))) break;
        const uint32_t first = c * p.per, n = std::min(p.per, count - first);
        st = read(sl, 0, (char*)dst + (size_t)first * size, n * size, s);
      }
      return st;
    });
  }

  static constexpr size_t kSlotBytes = 2u << 20;

 private:
  static constexpr int kWorkers = 8, kSlots = 2 * kWorkers, kSmall = 3;
  struct Slot {
    void* p = nullptr;
    size_t cap = 0;
    hipEvent_t ev = nullptr;
    bool busy = false;    // ev is recorded and not yet waited for
    bool pinned = false;  // host memory, else device memory
  };
  Slot slots_[kSlots + kSmall];
  int next_ = 0;

  // A transfer's chunks (whole records, a multiple of four) and workers.
  struct Plan {
    uint32_t per, chunks;
    int workers;
    Plan(size_t size, uint32_t count)
        : per((uint32_t)(kSlotBytes / size) & ~3u),
          chunks((uint32_t)(((uint64_t)count + per - 1) / per)),
          workers((int)std::min<uint32_t>(chunks, kWorkers)) {}
  };

  // Slots 2 t and 2 t + 1 of the result are worker t's.  A transfer of one
  // chunk gets one of a few slots of its own in turn, so that it does not wait
  // for the kernel of the transfer just before it, and a program that only
  // makes small transfers pins few of them.
  Slot* slots_for(const Plan& p) { return p.chunks > 1 ? slots_ : small_slot(); }
  Slot* small_slot() {
    next_ = (next_ + 1) % kSmall;
    return slots_ + kSlots + next_;
  }

  static int wait(Slot& sl) {
    if (!sl.busy) return CKT_OK;
    CKT_HIP(hipEventSynchronize(sl.ev));
    sl.busy = false;
    return CKT_OK;
  }
  // The slot, free and of at least `bytes`.
  static int acquire(Slot& sl, size_t bytes) {
    if (int st = wait(sl)) return st;
    if (!sl.ev) CKT_HIP(hipEventCreateWithFlags(&sl.ev, hipEventDisableTiming));
    if (bytes > sl.cap) {
      CKT_HIP(release(sl));
      const size_t cap = std::min(kSlotBytes, std::max<size_t>(2 * bytes, 64u << 10));
      sl.pinned = hipHostMalloc(&sl.p, cap, hipHostMallocDefault) == hipSuccess;
      if (!sl.pinned) {
        (void)hipGetLastError();
        sl.p = nullptr;
        CKT_HIP(hipMalloc(&sl.p, cap));
      }
      sl.cap = cap;
    }
    return CKT_OK;
  }
  static hipError_t release(Slot& sl) {
    void* p = sl.p;
    sl.p = nullptr;
    sl.cap = 0;
    if (!p) return hipSuccess;
    return sl.pinned ? hipHostFree(p) : hipFree(p);
  }
  static int write(const Slot& sl, size_t at, const void* src, size_t bytes, hipStream_t s) {
    return move(sl, (char*)sl.p + at, src, bytes, hipMemcpyHostToDevice, s);
  }
  static int read(const Slot& sl, size_t at, void* dst, size_t bytes, hipStream_t s) {
    return move(sl, dst, (const char*)sl.p + at, bytes, hipMemcpyDeviceToHost, s);
  }
  static int move(const Slot& sl, void* dst, const void* src, size_t bytes, hipMemcpyKind kind,
                  hipStream_t s) {
    if (!bytes) return CKT_OK;
    if (sl.pinned) {
      std::memcpy(dst, src, bytes);
      return CKT_OK;
    }
    CKT_HIP(hipMemcpyAsync(dst, src, bytes, kind, s));
    CKT_HIP(hipStreamSynchronize(s));
    return CKT_OK;
  }
  static int mark(Slot& sl, hipStream_t s) {
    CKT_HIP(hipEventRecord(sl.ev, s));
    sl.busy = true;
    return CKT_OK;
  }

  // work(t) for t in [0, workers): the first on this thread, the others on
  // threads of their own (or here too where none can be started).  Returns the
  // first failure, with its message as this thread's.
  template <class Work>
  static int team(int workers, int device, Work work) {
    if (workers <= 0) return CKT_OK;
    int rc[kWorkers] = {0};
    std::string err[kWorkers];
    std::thread th[kWorkers];
    auto one = [&](int t) {
      const hipError_t e = hipSetDevice(device);
      rc[t] = e != hipSuccess ? hip_fail(e, "hipSetDevice") : work(t);
      if (rc[t]) err[t] = ckt_last_error();
    };
    for (int t = 1; t < workers; t++) {
      try {
        th[t] = std::thread(one, t);
      } catch (const std::system_error&) {
      }
    }
    one(0);
    for (int t = 1; t < workers; t++) {
      if (th[t].joinable()) th[t].join();
      else one(t);
    }
    for (int t = 0; t < workers; t++)
      if (rc[t]) return fail(rc[t], err[t]);
    return CKT_OK;
  }
};

}  // namespace ckt
