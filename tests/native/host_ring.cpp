// HostRing (ckt_hostring.h) against a HIP runtime of a few functions in host
// memory, with and without pinned memory.  Built for the host and run by
// tests/test_load_limits.py; exits non-zero on a failure, after printing it.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "ckt_hostring.h"

static std::atomic<int> g_pinned{0}, g_device{0};  // allocations alive
static bool g_no_pinned = false;

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (g_no_pinned) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  g_pinned++;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  g_pinned--;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  g_device++;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::free(p);
  g_device--;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = (hipEvent_t)1;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
const char* ckt_last_error() { return "failed"; }
}
namespace ckt {
int fail(int status, const std::string&) { return status; }
int hip_fail(hipError_t, const char*) { return CKT_ERR_HIP; }
}  // namespace ckt

static int fails = 0;
static void expect(bool ok, const char* what, unsigned n) {
  if (ok) return;
  std::printf("FAIL %s, %u records, pinned memory %s\n", what, n, g_no_pinned ? "refused" : "there");
  fails++;
}

// `count` records of 16 bytes there and back, then as one slot in two parts.
static void round_trip(unsigned count) {
  std::vector<unsigned> src(4 * (size_t)count), dev(src.size()), back(src.size(), 0);
  for (size_t i = 0; i < src.size(); i++) src[i] = (unsigned)(i * 2654435761u);
  ckt::HostRing ring;
  for (int again = 0; again < 2; again++) {
    std::fill(dev.begin(), dev.end(), 0u);
    std::fill(back.begin(), back.end(), 0u);
    expect(ring.in(src.data(), 16, count, 0, nullptr, [&](void* slot, unsigned first, unsigned n) {
      std::memcpy(dev.data() + 4 * (size_t)first, slot, 16 * (size_t)n);
      return hipSuccess;
    }) == CKT_OK && dev == src, "in", count);
    expect(ring.out(back.data(), 16, count, 0, nullptr, [&](void* slot, unsigned first, unsigned n) {
      std::memcpy(slot, dev.data() + 4 * (size_t)first, 16 * (size_t)n);
      return hipSuccess;
    }) == CKT_OK && back == src, "out", count);
    const size_t bytes = 16 * (size_t)count, half = bytes / 32 * 16;
    if (bytes > ckt::HostRing::kSlotBytes) continue;
    std::fill(dev.begin(), dev.end(), 0u);
    std::fill(back.begin(), back.end(), 0u);
    char *s = (char*)src.data(), *b = (char*)back.data();
    expect(ring.put(bytes, nullptr, {{0, s, half}, {half, s + half, bytes - half}, {0, nullptr, 0}},
                    [&](void* slot) {
                      std::memcpy(dev.data(), slot, bytes);
                      return hipSuccess;
                    }) == CKT_OK && dev == src, "put", count);
    expect(ring.get(bytes, nullptr,
                    [&](void* slot) {
                      std::memcpy(slot, dev.data(), bytes);
                      return hipSuccess;
                    },
                    {{0, b, half}, {half, b + half, bytes - half}}) == CKT_OK && back == src,
           "get", count);
  }
}

int main() {
  for (bool none : {false, true}) {
    g_no_pinned = none;
    for (unsigned n : {1u, 3u, 4096u, 131072u, 131073u, 2500001u}) round_trip(n);
  }
  expect(g_pinned == 0 && g_device == 0, "every slot freed", 0);
  if (fails) return 1;
  std::printf("host ring: ok\n");
}
