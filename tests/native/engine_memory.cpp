// The engine's device memory (ckt_engine.cpp) against a HIP runtime of a few
// functions in host memory that counts device allocations: what a load holds at
// once, and the scratch kept between builds.  Kernels do nothing here.  Built for
// the host and run by tests/test_load_limits.py; exits non-zero on a failure,
// after printing it.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>

#include "ckt_engine.h"
#include "ckt_records.h"

using namespace ckt;

static std::map<void*, size_t> g_alive;
static size_t g_now, g_peak, g_capacity;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (g_now + n > g_capacity) return hipErrorOutOfMemory;
  *p = std::malloc(n);
  g_alive[*p] = n;
  g_now += n;
  g_peak = std::max(g_peak, g_now);
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  if (!g_alive.count(p)) std::abort();
  g_now -= g_alive[p];
  g_alive.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  return *s = (hipStream_t)1, hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t*, int) { return hipErrorNotSupported; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
const char* ckt_last_error() { return ""; }
int ckt_device_info(int, int* is950, int* cus, size_t* lds, size_t* hbm) {
  *is950 = 1, *cus = 256, *lds = 160 << 10, *hbm = 1u << 30;
  return CKT_OK;
}
}

namespace ckt {
int fail(int status, const std::string&) { return status; }
int hip_fail(hipError_t e, const char*) {
  return e == hipErrorOutOfMemory ? CKT_ERR_NO_MEMORY : CKT_ERR_HIP;
}
size_t scratch_of(uint32_t W) { return 32 * (size_t)W; }
int index_scratch(uint32_t, uint32_t W, void*, IndexScratch*, size_t* bytes) {
  return *bytes = scratch_of(W), CKT_OK;
}
size_t devgen_scratch_bytes(uint32_t, uint32_t W) { return scratch_of(W); }
int devgen_enqueue(const ckt_gen_params_t* p, const SlabLayout&, void*, void*, hipStream_t,
                   std::vector<ckt_piece_t>& pieces) {
  pieces.assign(1, ckt_piece_t{0, (uint32_t)p->wires_per_piece, 0, (uint32_t)p->nodes_per_piece});
  return CKT_OK;
}
int index_sort(const DevCircuit&, const IndexScratch&, hipStream_t) { return CKT_OK; }
hipError_t launch_index_rows(const DevCircuit&, const IndexScratch&, const LoadFaults*,
                             LoadFaults* host, hipStream_t) {
  return *host = LoadFaults{~0ull, ~0ull, ~0ull}, hipSuccess;
}
hipError_t launch_fill_u32(uint32_t*, uint32_t, size_t, hipStream_t) { return hipSuccess; }
hipError_t launch_clear_faults(LoadFaults*, hipStream_t) { return hipSuccess; }
hipError_t launch_unpack_rest(const void*, const LoadRest&, const DevCircuit&, uint32_t*,
                              LoadFaults*, hipStream_t) {
  return hipSuccess;
}
hipError_t launch_unpack_nodes(const ckt_node_t*, uint32_t, uint32_t, const DevCircuit&,
                               hipStream_t) {
  return hipSuccess;
}
hipError_t launch_unpack_wires(const ckt_wire_t*, uint32_t, uint32_t, const DevCircuit&,
                               const IndexScratch&, LoadFaults*, hipStream_t) {
  return hipSuccess;
}
hipError_t launch_unpack_locator(const int32_t*, uint32_t, uint32_t, const DevCircuit&,
                                 hipStream_t) {
  return hipSuccess;
}
hipError_t launch_copy_words(uint32_t*, const uint32_t*, uint32_t, hipStream_t) {
  return hipSuccess;
}
hipError_t launch_derive_locator(const DevCircuit&, hipStream_t) { return hipSuccess; }
hipError_t launch_check_pieces(const PieceIndex&, uint32_t, const DevCircuit&, LoadFaults*,
                               hipStream_t) {
  return hipSuccess;
}
}  // namespace ckt

static int fails = 0;
static void expect(bool ok, const char* what, uint64_t a, uint64_t b) {
  if (ok) return;
  std::printf("FAIL %s: %llu, %llu\n", what, (unsigned long long)a, (unsigned long long)b);
  fails++;
}

constexpr uint32_t N = 500, W = 40000;  // enough for a load on the device
constexpr size_t kFixed = 4096;  // the engine's counters
static const size_t kSlab = SlabLayout::make(N, W, 1).total;
static const size_t kScratch = scratch_of(W) + 4096;

struct Records {
  std::vector<ckt_node_t> nodes{N};
  std::vector<ckt_wire_t> wires{W};
  ckt_piece_t piece{0, W, 0, N};
};

static int add(Engine& e, uint32_t* id, const uint32_t* replaced = nullptr) {
  static const Records r;
  return e.add_records(r.nodes.data(), N, r.wires.data(), W, nullptr, &r.piece, 1, 0, replaced, id);
}
static int generate(Engine& e, uint32_t* id) {
  ckt_gen_params_t g{};
  g.num_pieces = 1, g.nodes_per_piece = N, g.wires_per_piece = W, g.pct_wire_in_piece = 100;
  return e.add_generated_on_device(&g, 0, id);
}

int main() {
  uint32_t id = 0;
  // A load holds no more than the budget at once, whatever room it leaves.
  for (size_t extra : {(size_t)0, kScratch / 2, kScratch, 4 * kScratch}) {
    for (bool replace : {false, true}) {
      g_capacity = ~(size_t)0;
      const size_t budget = (replace ? 2 : 1) * kSlab + extra;
      Engine e;
      expect(e.init(0, budget) == CKT_OK, "init", 0, 0);
      if (replace) expect(add(e, &id) == CKT_OK, "first load", budget, 0);
      g_peak = g_now;
      const uint32_t old = id;
      const int st = add(e, &id, replace ? &old : nullptr);
      expect(st == CKT_OK, "load", budget, (uint64_t)st);
      expect(e.count() == 1, "circuits", e.count(), 1);
      expect(g_peak <= budget + kFixed, "peak of a load, budget", g_peak, budget);
    }
    expect(g_now == 0, "everything freed", g_now, 0);
  }
  // Scratch kept between builds leaves as many circuits their room as there is.
  for (bool gen : {false, true}) {
    g_capacity = ~(size_t)0;
    const size_t budget = 256 * kScratch + kSlab / 2, want = budget / kSlab;
    Engine e;
    expect(e.init(0, budget) == CKT_OK, "init", 0, 0);
    size_t n = 0;
    int st = CKT_OK;
    while (!(st = gen ? generate(e, &id) : add(e, &id))) {
      n++;
      expect(g_now <= budget + kFixed, "kept, budget", g_now, budget);
      if (n == 3) expect(g_now >= 3 * kSlab + scratch_of(W), "scratch is kept", g_now, 3 * kSlab);
    }
    expect(st == CKT_ERR_BUDGET && n == want, "circuits in the budget", n, want);
  }
  // Where device memory runs out, a circuit gets the place of idle scratch.
  {
    g_capacity = ~(size_t)0;
    Engine e;
    expect(e.init(0, 1u << 30) == CKT_OK, "init", 0, 0);
    expect(add(e, &id) == CKT_OK, "load", 0, 0);
    expect(g_now > kSlab + scratch_of(W), "scratch is kept", g_now, kSlab);
    g_capacity = g_now - scratch_of(W) + kSlab;
    const int st = add(e, &id);
    expect(st == CKT_OK && e.count() == 2, "load into the scratch's place", (uint64_t)st, e.count());
  }
  expect(g_now == 0, "everything freed", g_now, 0);
  if (fails) return 1;
  std::printf("engine memory: ok\n");
}
