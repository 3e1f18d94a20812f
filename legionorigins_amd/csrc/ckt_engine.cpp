// ckt_engine.cpp -- device-resident circuits, tile lists and task launches.
#include "ckt_engine.h"
#include "ckt_index.h"
#include "ckt_records.h"

#include <algorithm>
#include <cstring>
#include <numeric>
#include <string>

namespace ckt {

static size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

SlabLayout SlabLayout::make(uint32_t N, uint32_t W, uint32_t P) {
  SlabLayout L{};
  L.ws = (uint32_t)align_up(std::max<uint32_t>(W, 1), 64);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off = align_up(off + bytes, 256);
    return o;
  };
  const size_t ws = L.ws, n = std::max<uint32_t>(N, 1), w = std::max<uint32_t>(W, 1);
  L.cur = take(ws * 4 * kSeg);
  L.vol = take(ws * 4 * (kSeg - 1));
  L.ind = take(ws * 4);
  L.res = take(ws * 4);
  L.wcap = take(ws * 4);
  L.in_ptr = take(ws * 4);
  L.out_ptr = take(ws * 4);
  L.in_loc = take(ws);
  L.out_loc = take(ws);
  L.charge = take(n * 4);
  L.voltage = take(n * 4);
  L.ncap = take(n * 4);
  L.leak = take(n * 4);
  L.locator = take(n);
  L.csr_row = take((n + 1) * 4);
  L.csr_ent = take(2 * w * 4);
  L.pieces = take(std::max<uint32_t>(P, 1) * sizeof(ckt_piece_t));
  L.total = off;
  return L;
}

void SlabImage::reset(uint32_t n, uint32_t w, uint32_t p) {
  N = n;
  W = w;
  P = p;
  lay = SlabLayout::make(n, w, p);
  bytes.assign(lay.total, 0);
  pieces.assign(p, ckt_piece_t{0, 0, 0, 0});
}

// Validates the loaded circuit and builds the node -> (wire, end) index in
// global (wire, in-before-out) order.
static int finalize_image(SlabImage& img) {
  const uint32_t N = img.N, W = img.W;
  const SlabLayout& L = img.lay;
  const uint32_t* in_ptr = img.at<uint32_t>(L.in_ptr);
  const uint32_t* out_ptr = img.at<uint32_t>(L.out_ptr);
  const uint8_t* in_loc = img.at<uint8_t>(L.in_loc);
  const uint8_t* out_loc = img.at<uint8_t>(L.out_loc);
  const uint8_t* loc = img.at<uint8_t>(L.locator);
  for (uint32_t w = 0; w < W; w++) {
    if (in_ptr[w] >= N || out_ptr[w] >= N)
      return fail(CKT_ERR_OUT_OF_RANGE, "wire " + std::to_string(w) + " points past the last node");
    if (in_loc[w] > 2 || out_loc[w] > 2)
      return fail(CKT_ERR_INVALID_ARG, "wire " + std::to_string(w) + " has an invalid PointerLocation");
  }
  for (uint32_t k = 0; k < img.P; k++) {
    const ckt_piece_t& p = img.pieces[k];
    if ((uint64_t)p.first_wire + p.num_wires > W || (uint64_t)p.first_node + p.num_nodes > N)
      return fail(CKT_ERR_OUT_OF_RANGE, "piece " + std::to_string(k) + " exceeds the circuit");
    // A private node belongs to one piece's region (circuit.cc:1261): only
    // that piece's wires may reach it.
    for (uint32_t w = p.first_wire; w < p.first_wire + p.num_wires; w++) {
      const uint32_t ends[2] = {in_ptr[w], out_ptr[w]};
      for (uint32_t e : ends)
        if (e - p.first_node >= p.num_nodes && loc[e])
          return fail(CKT_ERR_INVALID_ARG, "wire " + std::to_string(w) + " of piece " +
                                               std::to_string(k) +
                                               " reaches a private node of another piece");
    }
  }
  uint32_t* row = img.at<uint32_t>(L.csr_row);
  uint32_t* ent = img.at<uint32_t>(L.csr_ent);
  std::fill(row, row + N + 1, 0u);
  for (uint32_t w = 0; w < W; w++) {
    row[in_ptr[w] + 1]++;
    row[out_ptr[w] + 1]++;
  }
  for (uint32_t i = 0; i < N; i++) row[i + 1] += row[i];
  std::vector<uint32_t> pos(row, row + N);
  for (uint32_t w = 0; w < W; w++) {
    ent[pos[in_ptr[w]]++] = w << 1;
    ent[pos[out_ptr[w]]++] = (w << 1) | 1u;
  }
  std::memcpy(img.at<ckt_piece_t>(L.pieces), img.pieces.data(), img.P * sizeof(ckt_piece_t));
  return CKT_OK;
}

int image_from_aos(SlabImage& img, const ckt_node_t* nodes, uint32_t N, const ckt_wire_t* wires,
                   uint32_t W, const int32_t* locator, const ckt_piece_t* pieces, uint32_t P) {
  if ((N && !nodes) || (W && !wires) || (P && !pieces))
    return fail(CKT_ERR_INVALID_ARG, "load: null array");
  if (N == 0 || P == 0) return fail(CKT_ERR_INVALID_ARG, "load: need at least one node and one piece");
  if (N >= kMaxElements || W >= kMaxElements)
    return fail(CKT_ERR_OUT_OF_RANGE, "load: more than 2^30 nodes or wires");
  img.reset(N, W, P);
  const SlabLayout& L = img.lay;
  const size_t ws = L.ws;
  float* cur = img.at<float>(L.cur);
  float* vol = img.at<float>(L.vol);
  float *ind = img.at<float>(L.ind), *res = img.at<float>(L.res), *wcap = img.at<float>(L.wcap);
  uint32_t *in_ptr = img.at<uint32_t>(L.in_ptr), *out_ptr = img.at<uint32_t>(L.out_ptr);
  uint8_t *in_loc = img.at<uint8_t>(L.in_loc), *out_loc = img.at<uint8_t>(L.out_loc);
  // A block of records at a time, array by array: the arrays lie a multiple of
  // the wire stride apart, and where that is a power of two, 26 of them written in
  // turn push each other out of the cache (4096 wires took 376 us, 4097 took 64).
  constexpr uint32_t kBlock = 64;
  for (uint32_t first = 0; first < W; first += kBlock) {
    const ckt_wire_t* x = wires + first;
    const uint32_t n = std::min(kBlock, W - first);
    for (int s = 0; s < kSeg; s++)
      for (uint32_t k = 0; k < n; k++) cur[s * ws + first + k] = x[k].current[s];
    for (int s = 0; s < kSeg - 1; s++)
      for (uint32_t k = 0; k < n; k++) vol[s * ws + first + k] = x[k].voltage[s];
    for (uint32_t k = 0; k < n; k++) ind[first + k] = x[k].inductance;
    for (uint32_t k = 0; k < n; k++) res[first + k] = x[k].resistance;
    for (uint32_t k = 0; k < n; k++) wcap[first + k] = x[k].capacitance;
    for (uint32_t k = 0; k < n; k++) in_ptr[first + k] = x[k].in_ptr;
    for (uint32_t k = 0; k < n; k++) out_ptr[first + k] = x[k].out_ptr;
    for (uint32_t k = 0; k < n; k++) {
      if ((uint32_t)x[k].in_loc > 2 || (uint32_t)x[k].out_loc > 2)
        return fail(CKT_ERR_INVALID_ARG,
                    "wire " + std::to_string(first + k) + " has an invalid PointerLocation");
      in_loc[first + k] = (uint8_t)x[k].in_loc;
      out_loc[first + k] = (uint8_t)x[k].out_loc;
    }
  }
  float *charge = img.at<float>(L.charge), *voltage = img.at<float>(L.voltage);
  float *ncap = img.at<float>(L.ncap), *leak = img.at<float>(L.leak);
  uint8_t* loc = img.at<uint8_t>(L.locator);
  for (uint32_t i = 0; i < N; i++) {
    charge[i] = nodes[i].charge;
    voltage[i] = nodes[i].voltage;
    ncap[i] = nodes[i].capacitance;
    leak[i] = nodes[i].leakage;
    loc[i] = 1;
  }
  if (locator) {
    for (uint32_t i = 0; i < N; i++) loc[i] = locator[i] ? 1 : 0;
  } else {
    // Without a locator, a node is shared when any wire names it as a
    // shared or ghost end.
    for (uint32_t w = 0; w < W; w++) {
      if (in_loc[w] != CKT_PRIVATE_PTR && in_ptr[w] < N) loc[in_ptr[w]] = 0;
      if (out_loc[w] != CKT_PRIVATE_PTR && out_ptr[w] < N) loc[out_ptr[w]] = 0;
    }
  }
  std::copy(pieces, pieces + P, img.pieces.begin());
  return finalize_image(img);
}

namespace {
struct ImageSink final : GenSink {
  SlabImage* img;
  size_t ws;
  float *voltage, *ncap, *leak, *ind, *res, *wcap;
  uint32_t *in_ptr, *out_ptr;
  uint8_t *in_loc, *out_loc, *loc;
  explicit ImageSink(SlabImage* im) : img(im) {
    const SlabLayout& L = im->lay;
    ws = L.ws;
    voltage = im->at<float>(L.voltage);
    ncap = im->at<float>(L.ncap);
    leak = im->at<float>(L.leak);
    ind = im->at<float>(L.ind);
    res = im->at<float>(L.res);
    wcap = im->at<float>(L.wcap);
    in_ptr = im->at<uint32_t>(L.in_ptr);
    out_ptr = im->at<uint32_t>(L.out_ptr);
    in_loc = im->at<uint8_t>(L.in_loc);
    out_loc = im->at<uint8_t>(L.out_loc);
    loc = im->at<uint8_t>(L.locator);
  }
  void node(uint32_t i, float v, float c, float l) override {
    voltage[i] = v;
    ncap[i] = c;
    leak[i] = l;
  }
  void wire(uint32_t w, uint32_t in, uint32_t out, float L, float R, float C) override {
    in_ptr[w] = in;
    out_ptr[w] = out;
    ind[w] = L;
    res[w] = R;
    wcap[w] = C;
  }
  void ends(uint32_t w, uint32_t* in, uint32_t* out) override {
    *in = in_ptr[w];
    *out = out_ptr[w];
  }
  void locations(uint32_t w, int32_t a, int32_t b) override {
    in_loc[w] = (uint8_t)a;
    out_loc[w] = (uint8_t)b;
  }
  void locator(uint32_t i, int32_t v) override { loc[i] = (uint8_t)v; }
  void piece(uint32_t n, const ckt_piece_t& p) override { img->pieces[n] = p; }
};
}  // namespace

int image_from_gen(SlabImage& img, const ckt_gen_params_t* params) {
  uint32_t N, W, P;
  int st = gen_validate(params, &N, &W, &P);
  if (st) return st;
  img.reset(N, W, P);
  ImageSink sink(&img);
  if ((st = gen_run(params, sink))) return st;
  return finalize_image(img);
}

// ---------------------------------------------------------------------------

static uint64_t fnv(uint64_t h, const void* data, size_t n) {
  const uint8_t* p = (const uint8_t*)data;
  for (size_t i = 0; i < n; i++) {
    h ^= p[i];
    h *= 1099511628211ull;
  }
  return h;
}

static uint64_t piece_key(const ckt_piece_t& p) {
  return fnv(1469598103934665603ull, &p, sizeof(p));
}

// Build scratch up to this share of the budget is kept with the engine for the
// next build, within the budget beside the circuits; other scratch is allocated
// and freed by each build.  A circuit's scratch is about a quarter of its slab,
// nearly all of it for the index's sort (64 x 65536 wires 170 MB), and
// allocating it costs such a build 0.3 ms of 1.3.  The default budget's share (1
// GB) is the scratch of 25 M wires.
constexpr uint64_t kKeepShare = 256;

// How a load goes, by the slab's size (us a load with its wait, nodes = wires / 4).
// Up to kHostLoadBytes the host unpacks and checks the records and the slab goes up
// whole: 700 wires 22 against 77 on the device, 1500 30 / 83, 3000 45 / 94, 6000 77 /
// 108, 9500 120 / 135, 11000 137 / 143; 13000 158 / 152, 14500 173 / 160.
constexpr size_t kHostLoadBytes = 1408 << 10;
// Slabs up to this size are stored with one copy of the slab and a pass on the
// host, record by record (300 wires 16 us against 20 to 25 for a launch that packs the
// records, on two cards; 500 18 / 20 to 25, 900 22 / 23 to 29; in a process's first 200
// stores or so 30, see Engine::add, but with a copy to pinned memory 21 at any time).
// From 1024 wires on strides are multiples of 4 KB, for which that pass is slow.
constexpr size_t kHostStoreBytes = 104 << 10;

Engine::~Engine() {
  if (device_ < 0) return;
  (void)hipSetDevice(device_);
  if (stream_) (void)hipStreamSynchronize(stream_);
  drop_caches();
  for (Circuit* c : slots_) {
    if (c->stream_ordered) (void)hipFreeAsync(c->slab, stream_);
    else (void)hipFree(c->slab);
    delete c;
  }
  if (stream_) (void)hipStreamSynchronize(stream_);
  slots_.clear();
  if (d_table_) (void)hipFree(d_table_);
  if (d_counters_) (void)hipFree(d_counters_);
  if (d_bad_) (void)hipFree(d_bad_);
  if (d_partial_) (void)hipFree(d_partial_);
  if (devgen_scratch_) (void)hipFree(devgen_scratch_);
  for (const PinnedChunk& c : staging_) (void)hipHostFree(c.p);
  for (auto& p : pending_) {
    (void)hipEventDestroy(p.a);
    (void)hipEventDestroy(p.b);
  }
  for (hipEvent_t e : event_pool_) (void)hipEventDestroy(e);
  if (stream_) (void)hipStreamDestroy(stream_);
}

int Engine::init(int device, uint64_t budget_bytes) {
  int is950 = 0;
  size_t lds = 0, hbm = 0;
  int st = ckt_device_info(device, &is950, &num_cus_, &lds, &hbm);
  if (st) return st;
  if (!is950) return fail(CKT_ERR_NO_DEVICE, "device is not gfx950; this library is built for gfx950 only");
  CKT_HIP(hipSetDevice(device));
  device_ = device;
  lds_limit_ = lds;
  budget_ = budget_bytes ? budget_bytes : (uint64_t)(0.9 * (double)hbm);
  CKT_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
  // Asynchronously generated circuits come from the device's default memory
  // pool; keep what they release for reuse instead of returning it at each
  // synchronisation.  Without pool support they use plain allocations.
  hipMemPool_t pool = nullptr;
  uint64_t keep = UINT64_MAX;
  pool_ok_ = hipDeviceGetDefaultMemPool(&pool, device) == hipSuccess &&
             hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep) == hipSuccess;
  (void)hipGetLastError();
  CKT_HIP(hipMalloc((void**)&d_counters_, 4 * sizeof(uint32_t)));
  CKT_HIP(hipMalloc((void**)&d_bad_, sizeof(unsigned long long)));
  CKT_HIP(launch_fill_u32(d_counters_, 0u, 4, stream_));
  CKT_HIP(hipStreamSynchronize(stream_));
  return CKT_OK;
}

int Engine::add(SlabImage& img, int32_t loops, uint32_t* id) {
  CKT_HIP(hipSetDevice(device_));
  if (budget_ && in_use_ + img.lay.total > budget_)
    return fail(CKT_ERR_BUDGET, "circuit needs " + std::to_string(img.lay.total) +
                                    " bytes; budget has " + std::to_string(budget_ - in_use_) + " left");
  int st = trim_scratch(img.lay.total);
  if (st) return st;
  void* slab = nullptr;
  hipError_t e = alloc_slab(img.lay.total, &slab);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc(circuit)");
  // From pinned memory where a slot holds it: the runtime's copy from pageable
  // memory is slow for its first 10 MB or so in a process (loads of 3000 wires 175
  // us, then 45; 9500 wires 320, then 130).
  const bool fits = img.lay.total <= HostRing::kSlotBytes;
  const void* from = img.bytes.data();
  if (void* slot = fits ? ring_.pinned(img.lay.total) : nullptr)
    from = std::memcpy(slot, from, img.lay.total);
  e = hipMemcpy(slab, from, img.lay.total, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(slab);
    return hip_fail(e, "hipMemcpy(circuit upload)");
  }
  attach(slab, img.lay, img.N, img.W, img.P, img.pieces, loops, id);
  return CKT_OK;
}

// Scratch of a load: what it found wrong, the piece table's workgroup numbers
// (PieceIndex::first_block, over wires) and the index build's scratch.
namespace {
struct RecordScratch {
  size_t first_block, index, bytes;  // bytes 0: the index's size query failed
  RecordScratch(uint32_t N, uint32_t W, uint32_t P)
      : first_block(align_up(sizeof(LoadFaults), 256)),
        index(align_up(first_block + 4 * ((size_t)P + 1), 256)) {
    size_t n = 0;
    bytes = index_scratch(N, W, nullptr, nullptr, &n) ? 0 : index + n;
  }
};
}  // namespace

int Engine::build_scratch(size_t need, bool keep, void** scratch, void** own) {
  *scratch = *own = nullptr;
  int st;
  if (need > devgen_scratch_cap_ && keep) {
    if ((st = drop_scratch())) return st;
    if (hipMalloc(&devgen_scratch_, need) == hipSuccess) devgen_scratch_cap_ = need;
    else devgen_scratch_ = nullptr;
  }
  if (need <= devgen_scratch_cap_) *scratch = devgen_scratch_;
  else if (hipMalloc(own, need) == hipSuccess) *scratch = *own;
  else *own = nullptr;
  (void)hipGetLastError();
  return CKT_OK;
}

int Engine::drop_scratch() {
  if (!devgen_scratch_) return CKT_OK;
  // Builds already enqueued use it.
  CKT_HIP(hipStreamSynchronize(stream_));
  CKT_HIP(hipFree(devgen_scratch_));
  devgen_scratch_ = nullptr;
  devgen_scratch_cap_ = 0;
  return CKT_OK;
}

int Engine::trim_scratch(uint64_t bytes) {
  if (!budget_ || in_use_ + bytes + devgen_scratch_cap_ <= budget_) return CKT_OK;
  return drop_scratch();
}

hipError_t Engine::alloc_slab(size_t bytes, void** slab) {
  hipError_t e = hipMalloc(slab, bytes);
  if (e != hipSuccess && devgen_scratch_) {  // it may fit in the scratch's place
    (void)hipGetLastError();
    if (drop_scratch() == CKT_OK) e = hipMalloc(slab, bytes);
  }
  if (e != hipSuccess) {
    *slab = nullptr;
    (void)hipGetLastError();  // not the next launch's
  }
  return e;
}

int Engine::build_records(const ckt_node_t* nodes, const ckt_wire_t* wires, const int32_t* locator,
                          const ckt_piece_t* pieces, const DevCircuit& c, void* scratch) {
  const uint32_t N = c.num_nodes, W = c.num_wires, P = c.num_pieces;
  const RecordScratch at(N, W, P);
  LoadFaults* faults = (LoadFaults*)scratch;
  uint32_t* d_blocks = (uint32_t*)((uint8_t*)scratch + at.first_block);
  int st;
  IndexScratch sc{};
  size_t index_bytes = 0;
  if ((st = index_scratch(N, W, (uint8_t*)scratch + at.index, &sc, &index_bytes))) return st;
  // Pieces up to the first one that exceeds the circuit are checked for
  // private nodes of other pieces that their wires reach.
  std::vector<uint32_t> blocks(1, 0u);
  uint32_t good = 0;
  if (!piece_check_blocks(pieces, P, N, W, &blocks, &good)) return CKT_ERR_UNSUPPORTED;
  const LoadRest rest(N, locator != nullptr, P, good + 1);
  if (rest.bytes <= HostRing::kSlotBytes) {
    if ((st = ring_.put(rest.bytes, stream_,
                        {{0, nodes, sizeof(ckt_node_t) * (size_t)N},
                         {rest.locator_at, locator, locator ? 4 * (size_t)N : 0},
                         {rest.pieces_at, pieces, sizeof(ckt_piece_t) * (size_t)P},
                         {rest.blocks_at, blocks.data(), 4 * blocks.size()}},
                        [&](void* slot) {
                          return launch_unpack_rest(slot, rest, c, d_blocks, faults, stream_);
                        })))
      return st;
  } else {
    CKT_HIP(launch_clear_faults(faults, stream_));
    if ((st = ring_.in(nodes, sizeof(ckt_node_t), N, device_, stream_,
                       [&](void* slot, uint32_t first, uint32_t n) {
                         return launch_unpack_nodes((const ckt_node_t*)slot, first, n, c, stream_);
                       })) ||
        (locator &&
         (st = ring_.in(locator, sizeof(int32_t), N, device_, stream_,
                        [&](void* slot, uint32_t first, uint32_t n) {
                          return launch_unpack_locator((const int32_t*)slot, first, n, c, stream_);
                        }))) ||
        (st = ring_.in(pieces, sizeof(ckt_piece_t), P, device_, stream_,
                       [&](void* slot, uint32_t first, uint32_t n) {
                         return launch_copy_words((uint32_t*)(c.pieces + first), (uint32_t*)slot,
                                                  4 * n, stream_);
                       })) ||
        (st = ring_.in(blocks.data(), sizeof(uint32_t), good + 1, device_, stream_,
                       [&](void* slot, uint32_t first, uint32_t n) {
                         return launch_copy_words(d_blocks + first, (uint32_t*)slot, n, stream_);
                       })))
      return st;
  }
  if ((st = ring_.in(wires, sizeof(ckt_wire_t), W, device_, stream_,
                     [&](void* slot, uint32_t first, uint32_t n) {
                       return launch_unpack_wires((const ckt_wire_t*)slot, first, n, c, sc, faults,
                                                  stream_);
                     })))
    return st;
  if (!locator) CKT_HIP(launch_derive_locator(c, stream_));
  const PieceIndex ix{c.pieces, d_blocks, good};
  CKT_HIP(launch_check_pieces(ix, blocks.back(), c, faults, stream_));
  LoadFaults f;
  if ((st = index_sort(c, sc, stream_)) ||
      (st = ring_.out(&f, sizeof(f), 1, device_, stream_, [&](void* slot, uint32_t, uint32_t) {
         return launch_index_rows(c, sc, faults, (LoadFaults*)slot, stream_);
       })))
    return st;
  // In the order in which a pass over wires, then pieces, meets them.
  if (~f.location)
    return fail(CKT_ERR_INVALID_ARG,
                "wire " + std::to_string(f.location) + " has an invalid PointerLocation");
  if (~f.pointer)
    return fail(CKT_ERR_OUT_OF_RANGE,
                "wire " + std::to_string(f.pointer) + " points past the last node");
  if (~f.foreign)
    return fail(CKT_ERR_INVALID_ARG, "wire " + std::to_string((uint32_t)f.foreign) + " of piece " +
                                         std::to_string(f.foreign >> 32) +
                                         " reaches a private node of another piece");
  if (good < P)
    return fail(CKT_ERR_OUT_OF_RANGE, "piece " + std::to_string(good) + " exceeds the circuit");
  return CKT_OK;
}

int Engine::add_records(const ckt_node_t* nodes, uint32_t N, const ckt_wire_t* wires, uint32_t W,
                        const int32_t* locator, const ckt_piece_t* pieces, uint32_t P,
                        int32_t loops, const uint32_t* replaced, uint32_t* id) {
  if ((N && !nodes) || (W && !wires) || (P && !pieces))
    return fail(CKT_ERR_INVALID_ARG, "load: null array");
  if (N == 0 || P == 0) return fail(CKT_ERR_INVALID_ARG, "load: need at least one node and one piece");
  if (N >= kMaxElements || W >= kMaxElements)
    return fail(CKT_ERR_OUT_OF_RANGE, "load: more than 2^30 nodes or wires");
  CKT_HIP(hipSetDevice(device_));
  int st;
  const SlabLayout lay = SlabLayout::make(N, W, P);
  // The device path holds the new circuit and its scratch beside the replaced
  // one.  Where the budget or the memory has no room for that, the records are
  // unpacked and checked on the host and the replaced circuit leaves first; so
  // are small circuits.
  void *slab = nullptr, *own = nullptr, *scratch = nullptr;
  const size_t need = RecordScratch(N, W, P).bytes, kept = devgen_scratch_cap_;
  const bool keep = need <= budget_ / kKeepShare;
  const uint64_t held = in_use_ + lay.total + (need <= kept ? kept : keep ? need : kept + need);
  bool fits = lay.total > kHostLoadBytes && need && (!budget_ || held <= budget_);
  if (fits && (st = build_scratch(need, keep, &scratch, &own))) return st;
  fits = fits && scratch && hipMalloc(&slab, lay.total) == hipSuccess;
  (void)hipGetLastError();
  if (fits) {
    st = build_records(nodes, wires, locator, pieces, device_view(slab, lay, N, W, P),
                       scratch);
    const hipError_t e = hipStreamSynchronize(stream_);
    if (!st && e != hipSuccess) st = hip_fail(e, "load");
    if (own) (void)hipFree(own);
    if (st) (void)hipFree(slab);
    if (st && st != CKT_ERR_UNSUPPORTED && st != CKT_ERR_NO_MEMORY) return st;
    if (!st && replaced && (st = remove(*replaced))) {
      (void)hipFree(slab);
      return st;
    }
    if (!st) {
      attach(slab, lay, N, W, P, std::vector<ckt_piece_t>(pieces, pieces + P), loops, id);
      return CKT_OK;
    }
    (void)hipGetLastError();
  } else if (own) {
    (void)hipFree(own);
  }
  SlabImage img;
  if ((st = image_from_aos(img, nodes, N, wires, W, locator, pieces, P))) return st;
  if (replaced && (st = remove(*replaced))) return st;
  return add(img, loops, id);
}

int Engine::add_generated_on_device(const ckt_gen_params_t* params, int32_t loops, uint32_t* id) {
  uint32_t N, W, P;
  int st = gen_validate(params, &N, &W, &P);
  if (st) return st;
  CKT_HIP(hipSetDevice(device_));
  const SlabLayout lay = SlabLayout::make(N, W, P);
  if (budget_ && in_use_ + lay.total > budget_)
    return fail(CKT_ERR_BUDGET, "circuit needs " + std::to_string(lay.total) +
                                    " bytes; budget has " + std::to_string(budget_ - in_use_) + " left");
  const size_t need = devgen_scratch_bytes(N, W);
  if (!need) return fail(CKT_ERR_HIP, "device generator scratch size query failed");
  if ((st = trim_scratch(lay.total))) return st;
  void* slab = nullptr;
  hipError_t e = alloc_slab(lay.total, &slab);
  if (e != hipSuccess) return hip_fail(e, "hipMalloc(circuit)");
  std::vector<ckt_piece_t> pieces;
  void *scratch = nullptr, *own = nullptr;
  const bool keep =
      need <= budget_ / kKeepShare && (!budget_ || in_use_ + lay.total + need <= budget_);
  if (!(st = build_scratch(need, keep, &scratch, &own)) && !scratch)
    st = fail(CKT_ERR_NO_MEMORY, "device generator: no memory for its scratch");
  if (!st) st = devgen_enqueue(params, lay, slab, scratch, stream_, pieces);
  e = hipStreamSynchronize(stream_);
  if (!st && e != hipSuccess) st = hip_fail(e, "device generator");
  if (own) (void)hipFree(own);
  if (st) {
    (void)hipFree(slab);
    return st;
  }
  attach(slab, lay, N, W, P, pieces, loops, id);
  return CKT_OK;
}

DevCircuit Engine::device_view(void* slab, const SlabLayout& L, uint32_t N, uint32_t W,
                               uint32_t P) {
  uint8_t* b = (uint8_t*)slab;
  DevCircuit d{};
  d.cur = (float*)(b + L.cur);
  d.vol = (float*)(b + L.vol);
  d.ind = (float*)(b + L.ind);
  d.res = (float*)(b + L.res);
  d.wcap = (float*)(b + L.wcap);
  d.in_ptr = (uint32_t*)(b + L.in_ptr);
  d.out_ptr = (uint32_t*)(b + L.out_ptr);
  d.in_loc = b + L.in_loc;
  d.out_loc = b + L.out_loc;
  d.charge = (float*)(b + L.charge);
  d.voltage = (float*)(b + L.voltage);
  d.ncap = (float*)(b + L.ncap);
  d.leak = (float*)(b + L.leak);
  d.locator = b + L.locator;
  d.csr_row = (uint32_t*)(b + L.csr_row);
  d.csr_ent = (uint32_t*)(b + L.csr_ent);
  d.pieces = (ckt_piece_t*)(b + L.pieces);
  d.num_wires = W;
  d.ws = L.ws;
  d.num_nodes = N;
  d.num_pieces = P;
  return d;
}

void Engine::attach(void* slab, const SlabLayout& L, uint32_t N, uint32_t W, uint32_t P,
                    const std::vector<ckt_piece_t>& pieces, int32_t loops, uint32_t* id,
                    bool stream_ordered) {
  Circuit* c = new Circuit();
  c->stream_ordered = stream_ordered;
  c->id = next_id_++;
  c->num_nodes = N;
  c->num_wires = W;
  c->num_pieces = P;
  c->lay = L;
  c->slab = slab;
  c->pieces = pieces;
  c->loops_left = loops;
  c->dev = device_view(slab, L, N, W, P);
  for (uint32_t k = 0; k < P; k++) c->piece_index.emplace(piece_key(pieces[k]), k);
  // Wires partitioned by the pieces -> the CSR modes apply; node ranges
  // disjoint -> the LDS-privatised reduction applies.
  {
    std::vector<ckt_piece_t> ps = pieces;
    std::sort(ps.begin(), ps.end(), [](const ckt_piece_t& a, const ckt_piece_t& x) {
      return a.first_wire < x.first_wire;
    });
    uint64_t at = 0;
    bool ok = true;
    for (auto& p : ps) {
      if (p.num_wires == 0) continue;
      if (p.first_wire != at) ok = false;
      at = (uint64_t)p.first_wire + p.num_wires;
    }
    c->csr_ok = ok && at == W;
    std::sort(ps.begin(), ps.end(), [](const ckt_piece_t& a, const ckt_piece_t& x) {
      return a.first_node < x.first_node;
    });
    uint64_t end = 0, covered = 0;
    ok = true;
    for (auto& p : ps) {
      if (p.num_nodes == 0) continue;
      if (p.first_node < end) ok = false;
      end = (uint64_t)p.first_node + p.num_nodes;
      covered += p.num_nodes;
    }
    c->lds_ok = ok;
    c->nodes_ok = ok && covered == N;
  }
  slots_.push_back(c);
  by_id_[c->id] = c;
  in_use_ += L.total;
  table_dirty_ = true;
  generation_++;
  if (id) *id = c->id;
}

int Engine::remove(uint32_t id) { return remove_many(&id, 1); }

// A slab from the stream's memory pool is released stream-ordered, after
// everything already queued on the stream, so removing only such circuits
// needs no synchronisation; any other slab is freed after one stream
// synchronisation for the whole set.  The device descriptor table is only
// rewritten by ensure_table, by a copy queued behind every launch already on
// the stream.  Cached tile
// lists and graphs are keyed by the engine generation, which changes here, so
// entries naming the removed circuits can never be looked up again; they stay
// until the cache's size bound evicts them (drop_caches waits for the stream
// first).
int Engine::remove_many(const uint32_t* ids, size_t n) {
  bool sync = false;
  for (size_t k = 0; k < n; k++) {
    auto it = by_id_.find(ids[k]);
    if (it == by_id_.end())
      return fail(CKT_ERR_NOT_FOUND, "no circuit with id " + std::to_string(ids[k]));
    if (!it->second->stream_ordered) sync = true;
  }
  if (n == 0) return CKT_OK;
  CKT_HIP(hipSetDevice(device_));
  if (sync) CKT_HIP(hipStreamSynchronize(stream_));
  for (size_t k = 0; k < n; k++) {
    auto it = by_id_.find(ids[k]);
    if (it == by_id_.end()) continue;  // listed twice
    Circuit* c = it->second;
    if (c->stream_ordered) CKT_HIP(hipFreeAsync(c->slab, stream_));
    else CKT_HIP(hipFree(c->slab));
    in_use_ -= c->lay.total;
    slots_.erase(std::find(slots_.begin(), slots_.end(), c));
    by_id_.erase(it);
    delete c;
  }
  table_dirty_ = true;
  generation_++;
  return CKT_OK;
}

Circuit* Engine::find(uint32_t id) {
  auto it = by_id_.find(id);
  return it == by_id_.end() ? nullptr : it->second;
}

int Engine::slot_of(uint32_t id) const {
  for (size_t i = 0; i < slots_.size(); i++)
    if (slots_[i]->id == id) return (int)i;
  return -1;
}

int Engine::ref_for(uint32_t slot, const ckt_piece_t& p, PieceRef* out) const {
  if (slot >= slots_.size()) return fail(CKT_ERR_NOT_FOUND, "no circuit in slot");
  const Circuit* c = slots_[slot];
  auto it = c->piece_index.find(piece_key(p));
  if (it == c->piece_index.end())
    return fail(CKT_ERR_OUT_OF_RANGE, "piece {first_wire " + std::to_string(p.first_wire) +
                                          ", first_node " + std::to_string(p.first_node) +
                                          "} is not a piece of the loaded circuit");
  out->slot = slot;
  out->piece = it->second;
  return CKT_OK;
}

void Engine::all_refs(std::vector<PieceRef>& refs, bool only_active) const {
  refs.clear();
  for (uint32_t s = 0; s < slots_.size(); s++) {
    if (only_active && slots_[s]->loops_left <= 0) continue;
    for (uint32_t k = 0; k < slots_[s]->num_pieces; k++) refs.push_back(PieceRef{s, k});
  }
}

// The records of the slab `b`, in host memory; either array may be NULL.
static void aos_from_slab(const uint8_t* b, const SlabLayout& L, ckt_node_t* nodes, uint32_t N,
                          ckt_wire_t* wires, uint32_t W) {
  auto real = [&](size_t off) { return (const float*)(b + off); };
  auto word = [&](size_t off) { return (const uint32_t*)(b + off); };
  for (uint32_t w = 0; wires && w < W; w++) {
    ckt_wire_t& x = wires[w];
    std::memset(&x, 0, sizeof(x));
    x.in_ptr = word(L.in_ptr)[w];
    x.out_ptr = word(L.out_ptr)[w];
    x.in_loc = b[L.in_loc + w];
    x.out_loc = b[L.out_loc + w];
    x.inductance = real(L.ind)[w];
    x.resistance = real(L.res)[w];
    x.capacitance = real(L.wcap)[w];
    for (int s = 0; s < kSeg; s++) x.current[s] = real(L.cur)[s * L.ws + w];
    for (int s = 0; s < kSeg - 1; s++) x.voltage[s] = real(L.vol)[s * L.ws + w];
  }
  for (uint32_t i = 0; nodes && i < N; i++)
    nodes[i] = ckt_node_t{real(L.charge)[i], real(L.voltage)[i], real(L.ncap)[i], real(L.leak)[i]};
}

// The records are put together on the device and written straight into
// pinned slots; waits for the stream, behind which the kernels are queued.  The
// smallest circuits' slabs are copied out whole instead.
int Engine::store(uint32_t id, ckt_node_t* nodes, ckt_wire_t* wires) {
  Circuit* c = find(id);
  if (!c) return fail(CKT_ERR_NOT_FOUND, "no circuit with id " + std::to_string(id));
  CKT_HIP(hipSetDevice(device_));
  int st;
  if (c->lay.total <= kHostStoreBytes) {
    std::vector<uint8_t> slab(c->lay.total);
    CKT_HIP(hipStreamSynchronize(stream_));
    CKT_HIP(hipMemcpy(slab.data(), c->slab, c->lay.total, hipMemcpyDeviceToHost));
    aos_from_slab(slab.data(), c->lay, nodes, c->num_nodes, wires, c->num_wires);
    return CKT_OK;
  }
  const size_t wire_bytes = sizeof(ckt_wire_t) * (size_t)c->num_wires,
               node_bytes = sizeof(ckt_node_t) * (size_t)c->num_nodes;
  if (wires && nodes && wire_bytes + node_bytes <= HostRing::kSlotBytes)
    return ring_.get(wire_bytes + node_bytes, stream_,
                     [&](void* slot) {
                       return launch_pack_all((ckt_wire_t*)slot,
                                              (ckt_node_t*)((uint8_t*)slot + wire_bytes), c->dev,
                                              stream_);
                     },
                     {{0, wires, wire_bytes}, {wire_bytes, nodes, node_bytes}});
  if (wires &&
      (st = ring_.out(wires, sizeof(ckt_wire_t), c->num_wires, device_, stream_,
                      [&](void* slot, uint32_t first, uint32_t n) {
                        return launch_pack_wires((ckt_wire_t*)slot, first, n, c->dev, stream_);
                      })))
    return st;
  if (nodes &&
      (st = ring_.out(nodes, sizeof(ckt_node_t), c->num_nodes, device_, stream_,
                      [&](void* slot, uint32_t first, uint32_t n) {
                        return launch_pack_nodes((ckt_node_t*)slot, first, n, c->dev, stream_);
                      })))
    return st;
  CKT_HIP(hipStreamSynchronize(stream_));
  return CKT_OK;
}

int Engine::store_topology(uint32_t id, int32_t* locator, uint32_t* csr_row, uint32_t* csr_ent) {
  Circuit* c = find(id);
  if (!c) return fail(CKT_ERR_NOT_FOUND, "no circuit with id " + std::to_string(id));
  CKT_HIP(hipSetDevice(device_));
  int st;
  auto words = [&](uint32_t* dst, const uint32_t* src, uint32_t count) {
    return ring_.out(dst, sizeof(uint32_t), count, device_, stream_,
                     [&](void* slot, uint32_t first, uint32_t n) {
                       return launch_copy_words((uint32_t*)slot, src + first, n, stream_);
                     });
  };
  if (locator &&
      (st = ring_.out(locator, sizeof(int32_t), c->num_nodes, device_, stream_,
                      [&](void* slot, uint32_t first, uint32_t n) {
                        return launch_pack_locator((int32_t*)slot, first, n, c->dev, stream_);
                      })))
    return st;
  if (csr_row && (st = words(csr_row, c->dev.csr_row, c->num_nodes + 1))) return st;
  if (csr_ent && (st = words(csr_ent, c->dev.csr_ent, 2 * c->num_wires))) return st;
  CKT_HIP(hipStreamSynchronize(stream_));
  return CKT_OK;
}

int Engine::copy_voltages_async(uint32_t id, float* dst) {
  Circuit* c = find(id);
  if (!c) return fail(CKT_ERR_NOT_FOUND, "no circuit with id " + std::to_string(id));
  CKT_HIP(hipMemcpyAsync(dst, c->dev.voltage, (size_t)c->num_nodes * 4, hipMemcpyDeviceToHost,
                         stream_));
  return CKT_OK;
}

int Engine::download_voltages(uint32_t id, std::vector<float>& v) {
  Circuit* c = find(id);
  if (!c) return fail(CKT_ERR_NOT_FOUND, "no circuit with id " + std::to_string(id));
  CKT_HIP(hipSetDevice(device_));
  CKT_HIP(hipStreamSynchronize(stream_));
  v.resize(c->num_nodes);
  CKT_HIP(hipMemcpy(v.data(), c->dev.voltage, (size_t)c->num_nodes * 4, hipMemcpyDeviceToHost));
  return CKT_OK;
}

// The table is rewritten by a copy queued on the stream: it runs after every
// launch already queued there (which read the old contents) and before every
// later one.  Graphs are keyed by the engine generation, which changes with
// the table, so no captured graph is replayed against a rewritten table.
// Only growing the buffer waits for the stream.
int Engine::ensure_table() {
  if (!table_dirty_) return CKT_OK;
  std::vector<DevCircuit> tab(slots_.size());
  for (size_t i = 0; i < slots_.size(); i++) tab[i] = slots_[i]->dev;
  if (tab.size() > table_cap_) {
    CKT_HIP(hipStreamSynchronize(stream_));
    if (d_table_) CKT_HIP(hipFree(d_table_));
    d_table_ = nullptr;
    table_cap_ = std::max<size_t>(tab.size(), 2 * table_cap_);
    CKT_HIP(hipMalloc((void**)&d_table_, table_cap_ * sizeof(DevCircuit)));
  }
  if (!tab.empty()) {
    void* staged = nullptr;
    int st = stage(tab.data(), tab.size() * sizeof(DevCircuit), &staged);
    if (st) return st;
    CKT_HIP(hipMemcpyAsync(d_table_, staged, tab.size() * sizeof(DevCircuit),
                           hipMemcpyHostToDevice, stream_));
  }
  table_dirty_ = false;
  return CKT_OK;
}

void Engine::drop_caches() {
  if (tile_cache_.empty() && graphs_.empty()) return;
  if (stream_) (void)hipStreamSynchronize(stream_);
  for (auto& kv : graphs_) (void)hipGraphExecDestroy(kv.second);
  graphs_.clear();
  for (auto& kv : tile_cache_) {
    if (kv.second.pooled) (void)hipFreeAsync(kv.second.p, stream_);
    else (void)hipFree(kv.second.p);
  }
  tile_cache_.clear();
}

// Tile lists are allocated from the stream's memory pool and filled by a
// copy from pinned staging queued on the stream, so building one for a new
// set of circuits does not wait for the launches already queued.
int Engine::upload_buf(uint64_t key, const void* data, size_t bytes, uint32_t n, DevBuf* out) {
  if (tile_cache_.size() >= 64) drop_caches();
  DevBuf b;
  b.n = n;
  b.pooled = pool_ok_;
  const size_t sz = std::max<size_t>(bytes, 16);
  CKT_HIP(b.pooled ? hipMallocAsync(&b.p, sz, stream_) : hipMalloc(&b.p, sz));
  if (bytes) {
    void* staged = nullptr;
    int st = stage(data, bytes, &staged);
    hipError_t e = st ? hipSuccess : hipMemcpyAsync(b.p, staged, bytes, hipMemcpyHostToDevice, stream_);
    if (st || e != hipSuccess) {
      if (b.pooled) (void)hipFreeAsync(b.p, stream_);
      else (void)hipFree(b.p);
      return st ? st : hip_fail(e, "hipMemcpyAsync(tiles)");
    }
  }
  tile_cache_[key] = b;
  *out = b;
  return CKT_OK;
}

enum TileKind { TK_WIRES = 1, TK_NODES = 2, TK_CSR = 3, TK_PIECES = 4, TK_CNC = 5 };
// update_voltages: 256 lanes x 8 nodes per tile.
constexpr int kUpvTile = 2048;
// Node bytes update_voltages moves per node (4 arrays read, 2 written) and the
// MI355X last-level cache (256 MB of Infinity Cache): a launch over more node
// bytes than that streams them with nontemporal accesses.
constexpr uint64_t kUpvBytesPerNode = 24;
constexpr uint64_t kLastLevelCacheBytes = 256ull << 20;

// Whether calc_new_currents with the early end moves its wires' state with
// ordinary accesses, so that the last-level cache holds it from loop to loop:
// where the state, the pointers and the index entries (104 bytes a wire) fit that
// cache but not twice the L2s (8 x 4 MB), else nontemporal (load_once).  Larger
// circuits push each other's lines out, and below the L2s the ordinary accesses
// push out what the loop's other launch reads.  Microseconds a SCALED loop,
// nontemporal / ordinary, 16384 wires to 4096 nodes or 65536 to 16384: 128k wires
// 15.7 / 15.7, 256k 19.3 / 20.3, 384k 27.3 / 27.8, 512k 36.0 / 36.9; 768k 45.8 /
// 41.2, 1024k 59.3 / 51.7, 2048k 109 / 89.5, 2304k 119 / 101; 2560k 132 / 144, 4096k
// 200 / 230.  FAST and RECIP alike; EXACT, whose launch its divisions bind, gains 2% there
// and stays nontemporal.
//   It takes loops in a row: on a state that is not in the cache yet the ordinary
// accesses are slower.  Whole calls with the voltages read back, on states that take
// turns, 1024k and 2048k wires, us: 1 loop 335 / 338 and 576 / 589, 2 loops 416 / 426
// and 679 / 693, 3 loops 486 / 486 and 796 / 772, 5 loops 631 / 600 and 1083 / 1055, 8 loops
// 831 / 772 and 1555 / 1425.
constexpr uint64_t kL2Bytes = 8 * (4ull << 20);
constexpr uint64_t kCncBytesPerWire = 104;
constexpr int kCachedLoops = 3;

static bool cnc_state_cached(uint64_t wires, int policy, int loops) {
  const uint64_t bytes = wires * kCncBytesPerWire;
  return loops >= kCachedLoops && policy != CKT_POLICY_EXACT && bytes > 2 * kL2Bytes &&
         bytes <= kLastLevelCacheBytes;
}

int Engine::tiles_for(int kind, const std::vector<PieceRef>& refs, int block, DevBuf* out) {
  uint64_t key = fnv(1469598103934665603ull, &kind, sizeof(kind));
  key = fnv(key, &block, sizeof(block));
  if (kind == TK_CNC) {
    const int sched[3] = {wires_per_lane_, tile_span_, tile_order_};
    key = fnv(key, sched, sizeof(sched));
  }
  key = fnv(key, &generation_, sizeof(generation_));
  key = fnv(key, refs.data(), refs.size() * sizeof(PieceRef));
  auto it = tile_cache_.find(key);
  if (it != tile_cache_.end()) {
    *out = it->second;
    return CKT_OK;
  }
  if (kind == TK_PIECES) {
    // `block` is the number of wire subranges per piece; each piece's rows of
    // partial sums follow the previous piece's.
    std::vector<PieceTile> t;
    t.reserve(refs.size());
    uint64_t off = 0;
    for (const PieceRef& r : refs) {
      t.push_back(PieceTile{r.slot, r.piece, (uint32_t)off, 0});
      off += (uint64_t)std::max(block, 1) * slots_[r.slot]->pieces[r.piece].num_nodes;
    }
    return upload_buf(key, t.data(), t.size() * sizeof(PieceTile), (uint32_t)t.size(), out);
  }
  std::vector<Tile> t;
  if (kind == TK_CSR) {
    std::vector<uint32_t> seen;
    for (const PieceRef& r : refs) {  // usually grouped by circuit
      if (!seen.empty() && seen.back() == r.slot) continue;
      if (std::find(seen.begin(), seen.end(), r.slot) == seen.end()) seen.push_back(r.slot);
    }
    for (uint32_t s : seen) {
      const uint32_t N = slots_[s]->num_nodes;
      for (uint32_t off = 0; off < N; off += (uint32_t)block)
        t.push_back(Tile{s, off, std::min<uint32_t>((uint32_t)block, N - off), 0});
    }
  } else if (kind == TK_CNC) {
    std::vector<Tile> pieces;
    pieces.reserve(refs.size());
    for (const PieceRef& r : refs) {
      const ckt_piece_t& p = slots_[r.slot]->pieces[r.piece];
      pieces.push_back(Tile{r.slot, p.first_wire, p.num_wires, r.piece});
    }
    t = cnc_schedule<Tile>(pieces, (uint32_t)block * (uint32_t)wires_per_lane_, tile_span_, tile_order_);
  } else {
    for (const PieceRef& r : refs) {
      const ckt_piece_t& p = slots_[r.slot]->pieces[r.piece];
      const uint32_t first = kind == TK_WIRES ? p.first_wire : p.first_node;
      const uint32_t num = kind == TK_WIRES ? p.num_wires : p.num_nodes;
      for (uint32_t off = 0; off < num; off += (uint32_t)block)
        t.push_back(Tile{r.slot, first + off, std::min<uint32_t>((uint32_t)block, num - off), r.piece});
    }
  }
  return upload_buf(key, t.data(), t.size() * sizeof(Tile), (uint32_t)t.size(), out);
}

int Engine::timed_begin(int task, hipEvent_t* a) {
  (void)task;
  *a = nullptr;
  if (!timing_) return CKT_OK;
  if (event_pool_.empty()) {
    hipEvent_t e;
    CKT_HIP(hipEventCreate(&e));
    event_pool_.push_back(e);
  }
  *a = event_pool_.back();
  event_pool_.pop_back();
  CKT_HIP(hipEventRecord(*a, stream_));
  return CKT_OK;
}

int Engine::timed_end(int task, hipEvent_t a) {
  if (!timing_ || !a) return CKT_OK;
  hipEvent_t b;
  if (event_pool_.empty()) {
    CKT_HIP(hipEventCreate(&b));
  } else {
    b = event_pool_.back();
    event_pool_.pop_back();
  }
  CKT_HIP(hipEventRecord(b, stream_));
  pending_.push_back(Pending{task, a, b});
  if (pending_.size() > 4096) {
    double ms;
    uint64_t n;
    return kernel_time(-1, &ms, &n);
  }
  return CKT_OK;
}

int Engine::kernel_time(int task, double* ms, uint64_t* launches) {
  if (!pending_.empty()) {  // events to read: they have to have happened
    CKT_HIP(hipSetDevice(device_));
    CKT_HIP(hipStreamSynchronize(stream_));
  }
  for (auto& p : pending_) {
    float t = 0.f;
    CKT_HIP(hipEventElapsedTime(&t, p.a, p.b));
    acc_ms_[p.task] += t;
    acc_n_[p.task]++;
    event_pool_.push_back(p.a);
    event_pool_.push_back(p.b);
  }
  pending_.clear();
  if (task >= 0 && task < CKT_NUM_TASK_IDS) {
    if (ms) *ms = acc_ms_[task];
    if (launches) *launches = acc_n_[task];
  }
  return CKT_OK;
}

void Engine::reset_timing() {
  double ms;
  uint64_t n;
  (void)kernel_time(-1, &ms, &n);
  for (int i = 0; i < CKT_NUM_TASK_IDS; i++) {
    acc_ms_[i] = 0;
    acc_n_[i] = 0;
  }
}

int Engine::cnc(const std::vector<PieceRef>& refs, int policy, bool fuse_dsc) {
  if (policy < CKT_POLICY_EXACT || policy > CKT_POLICY_SCALED)
    return fail(CKT_ERR_INVALID_ARG, "calc_new_currents: unknown policy");
  int st;
  if ((st = ensure_table())) return st;
  DevBuf t;
  const int block = cnc_block_for(policy);
  if ((st = tiles_for(TK_CNC, refs, block, &t))) return st;
  hipEvent_t a;
  if ((st = timed_begin(CKT_CALC_NEW_CURRENTS, &a))) return st;
  hipError_t e;
  // Launch shape unless set with OPT_CNC_BLOCK / OPT_PERSISTENT /
  // OPT_WAVES_PER_SIMD.  With the early end a launch is bound by the wires'
  // bytes, and a plain grid of 256-lane workgroups is best: on the 64 x 16384 x
  // 65536 circuit 157 us for SCALED, FAST and RECIP, and 183 to 358 for EXACT (stable
  // profile).  With ordinary instead of nontemporal accesses, where the shapes
  // were compared: 170 us for the first three (172-190 with 64, 128 or 512 lanes;
  // a tile queue 190-980), EXACT 239 (stable) and 169 (reference profile) against
  // 228-374 and 179-185.  With every step: on the same circuit a persistent tile
  // queue of 256-lane workgroups with 4 resident waves per SIMD beats the
  // plain grid by 6% for SCALED and 1-2% for FAST and RECIP.  For EXACT (71
  // VGPRs, at most 7 resident waves) a queue of 64-lane workgroups at 7 waves
  // per SIMD is 1-3% faster than the plain grid of 256-lane workgroups, which
  // it keeps when the workgroup size is set (a queue of 256-lane workgroups
  // is 1-4% slower than that grid).
  const bool persistent =
      persistent_ >= 0 ? persistent_ != 0
                       : all_steps_ && (policy != CKT_POLICY_EXACT || cnc_block_ < 0);
  uint64_t wires = 0;
  for (const PieceRef& r : refs) wires += slots_[r.slot]->pieces[r.piece].num_wires;
  const CncSteps how = all_steps_ ? kEveryStep
                       : cnc_state_cached(wires, policy, loops_in_a_row_) ? kEarlyEnd
                                                 : kEarlyEndStream;
  const int waves = waves_per_simd_ > 0 ? waves_per_simd_ : (policy == CKT_POLICY_EXACT ? 7 : 4);
  if (persistent) {
    const int waves_per_block = block / 64;
    int grid = num_cus_ * 4 * waves / waves_per_block;
    if (grid > (int)t.n) grid = (int)t.n;
    e = launch_cnc_persistent(policy, fuse_dsc, d_table_, (const Tile*)t.p, t.n, block, grid,
                              d_counters_, steps_, how, stream_);
  } else {
    e = launch_cnc(policy, fuse_dsc, d_table_, (const Tile*)t.p, t.n, block, steps_, how, stream_);
  }
  if (e != hipSuccess) return hip_fail(e, "calc_new_currents launch");
  return timed_end(CKT_CALC_NEW_CURRENTS, a);
}

// Every tile list one loop's launches use, built before the first launch.
// A synchronous upload issued while a kernel runs waits for CUs the kernel
// holds (for the whole of a calc_new_currents launch), and the host with it.
int Engine::prefetch_tiles(const std::vector<PieceRef>& refs, int policy, int mode) {
  int st;
  if (mode < CKT_REDUCE_ATOMIC || mode > CKT_REDUCE_CSR_KAHAN64)
    return fail(CKT_ERR_INVALID_ARG, "distribute_charge: unknown reduction mode");
  // room for every entry made here, so none is evicted before its launch
  if (tile_cache_.size() + 8 > 64) drop_caches();
  if ((st = ensure_table())) return st;
  DevBuf t;
  if ((st = tiles_for(TK_CNC, refs, cnc_block_for(policy), &t))) return st;
  const LoopForm form = loop_form(refs, mode);
  if (form == kFusedNodes) return tiles_for(TK_CSR, refs, 256, &t);
  if (mode == CKT_REDUCE_ATOMIC && form == kSeparate) {
    if ((st = tiles_for(TK_WIRES, refs, 256, &t))) return st;
    LdsPlan plan;
    if ((st = lds_plan(refs, &plan))) return st;
    if (plan.lds && (st = tiles_for(TK_PIECES, refs, (int)plan.splits, &t))) return st;
  }
  if (mode != CKT_REDUCE_ATOMIC) {
    if ((st = csr_nodes_ok(refs))) return st;
    if ((st = tiles_for(TK_CSR, refs, 256, &t))) return st;
  }
  return tiles_for(TK_NODES, refs, kUpvTile, &t);
}

int Engine::loop_once(const std::vector<PieceRef>& refs, int policy, int mode) {
  int st;
  if ((st = prefetch_tiles(refs, policy, mode))) return st;
  return launch_loop(refs, policy, mode);
}

int Engine::launch_loop(const std::vector<PieceRef>& refs, int policy, int mode) {
  int st;
  const LoopForm form = loop_form(refs, mode);
  if ((st = cnc(refs, policy, form == kFusedAtomic))) return st;
  if (form == kFusedNodes) return csr(refs, mode, true);
  if (form == kSeparate && (st = dsc(refs, mode))) return st;
  return upv(refs);
}

// The index form of distribute_charge leaves a node's whole charge in one
// lane's register, so update_voltages rides along wherever the launch covers
// every node of its circuits once.  ATOMIC's order of additions is unspecified,
// and with the early end the index is the faster way to it too, except in small
// launches (us a loop with the index / with the atomics in calc_new_currents /
// with the LDS reduction as its own launch: 64 x 65536 wires 230 / 417 / 234, 16 x
// 16384 21 / 34 / 29, 4 x 4096 11.9 / 10.7 / 18.7; the first of these is 201 now
// that calc_new_currents leaves the index its cached currents).  Where every step runs, the
// atomics hide behind the steps of other waves and stay fused.  OPT_FUSE_DSC names the
// form; where it does not, a named OPT_DSC_ATOMIC_IMPL, which is about launches of
// distribute_charge alone, leaves the loops the fused atomics.
constexpr uint64_t kIndexSumWires = 32768;

Engine::LoopForm Engine::loop_form(const std::vector<PieceRef>& refs, int mode) const {
  if (mode == CKT_REDUCE_ATOMIC) {
    if (fuse_dsc_ > 0 || (fuse_dsc_ < 0 && all_steps_)) return kFusedAtomic;
    if (fuse_dsc_ == 0) return kSeparate;
    if (dsc_atomic_impl_ != 0) return kFusedAtomic;
    uint64_t wires = 0;
    for (const PieceRef& r : refs) wires += slots_[r.slot]->pieces[r.piece].num_wires;
    if (wires < kIndexSumWires) return kFusedAtomic;
  }
  // every piece of every circuit named, each once (refs are grouped by slot,
  // as all_refs lists them)
  bool whole = true;
  for (size_t i = 0; whole && i < refs.size();) {
    const Circuit* c = slots_[refs[i].slot];
    whole = c->csr_ok && c->nodes_ok && refs.size() - i >= c->num_pieces;
    for (uint32_t k = 0; whole && k < c->num_pieces; k++)
      whole = refs[i + k].slot == refs[i].slot && refs[i + k].piece == k;
    i += c->num_pieces;
    whole = whole && (i >= refs.size() || refs[i].slot > refs[i - 1].slot);
  }
  if (whole) return kFusedNodes;
  return mode == CKT_REDUCE_ATOMIC ? kFusedAtomic : kSeparate;
}

int Engine::csr(const std::vector<PieceRef>& refs, int mode, bool update) {
  int st;
  DevBuf t;
  if ((st = tiles_for(TK_CSR, refs, 256, &t))) return st;
  hipEvent_t a;
  if ((st = timed_begin(CKT_DISTRIBUTE_CHARGE, &a))) return st;
  const hipError_t e = launch_dsc_csr(mode == CKT_REDUCE_CSR_KAHAN64, update, d_table_,
                                      (const Tile*)t.p, t.n, 256, stream_);
  if (e != hipSuccess) return hip_fail(e, "distribute_charge launch");
  return timed_end(CKT_DISTRIBUTE_CHARGE, a);
}

int Engine::csr_nodes_ok(const std::vector<PieceRef>& refs) const {
  std::map<uint32_t, std::vector<uint32_t>> per;
  for (const PieceRef& r : refs) per[r.slot].push_back(r.piece);
  for (auto& kv : per) {
    const Circuit* c = slots_[kv.first];
    if (!c->csr_ok)
      return fail(CKT_ERR_UNSUPPORTED, "CSR reduction needs pieces that partition the wires");
    std::vector<uint32_t>& v = kv.second;
    std::sort(v.begin(), v.end());
    if (v.size() != c->num_pieces || std::unique(v.begin(), v.end()) != v.end())
      return fail(CKT_ERR_UNSUPPORTED,
                  "CSR reduction runs over every piece of a circuit in one launch");
  }
  return CKT_OK;
}

int Engine::lds_plan(const std::vector<PieceRef>& refs, LdsPlan* plan) {
  LdsPlan p;
  p.lds = dsc_atomic_impl_ != 1 && !refs.empty();
  uint32_t min_wires = UINT32_MAX;
  uint64_t nodes = 0;
  for (const PieceRef& r : refs) {
    const Circuit* c = slots_[r.slot];
    const ckt_piece_t& pc = c->pieces[r.piece];
    p.lds = p.lds && c->lds_ok;
    p.max_nodes = std::max(p.max_nodes, pc.num_nodes);
    min_wires = std::min(min_wires, pc.num_wires);
    nodes += pc.num_nodes;
  }
  p.lds_bytes = dsc_lds_bytes(p.max_nodes);
  p.lds = p.lds && p.lds_bytes <= lds_limit_;
  if (p.lds) {
    // Two workgroups per CU, with no subrange under 2048 wires and at most 16
    // per piece.
    const uint64_t want = ((uint64_t)2 * num_cus_ + refs.size() - 1) / refs.size();
    const uint64_t by_size = std::max<uint32_t>(1, min_wires / 2048);
    p.splits = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>({want, by_size, 16}));
    if ((uint64_t)p.splits * nodes > 0xffffffffull) p.splits = 1;
    // Rows of partial sums even with one subrange: the second kernel's plain
    // read-add-write of every node replaces an atomic per shared node.
    p.partial_floats = (uint64_t)p.splits * nodes <= 0xffffffffull ? (uint64_t)p.splits * nodes : 0;
    if (p.partial_floats > partial_cap_) {
      CKT_HIP(hipStreamSynchronize(stream_));
      if (d_partial_) CKT_HIP(hipFree(d_partial_));
      d_partial_ = nullptr;
      partial_cap_ = 0;
      CKT_HIP(hipMalloc((void**)&d_partial_, p.partial_floats * sizeof(float)));
      partial_cap_ = p.partial_floats;
    }
  }
  *plan = p;
  return CKT_OK;
}

int Engine::dsc(const std::vector<PieceRef>& refs, int mode) {
  int st;
  if (mode < CKT_REDUCE_ATOMIC || mode > CKT_REDUCE_CSR_KAHAN64)
    return fail(CKT_ERR_INVALID_ARG, "distribute_charge: unknown reduction mode");
  if ((st = ensure_table())) return st;
  DevBuf t;
  hipError_t e;
  hipEvent_t a;
  if (mode == CKT_REDUCE_ATOMIC) {
    LdsPlan plan;
    if ((st = lds_plan(refs, &plan))) return st;
    if (dsc_atomic_impl_ == 2 && !plan.lds)
      return fail(CKT_ERR_UNSUPPORTED, "LDS reduction: a piece's node range does not fit in LDS");
    if (plan.lds) {
      if ((st = tiles_for(TK_PIECES, refs, (int)plan.splits, &t))) return st;
      if ((st = timed_begin(CKT_DISTRIBUTE_CHARGE, &a))) return st;
      e = launch_dsc_lds(d_table_, (const PieceTile*)t.p, t.n, plan.splits, plan.max_nodes,
                         plan.partial_floats ? d_partial_ : nullptr, plan.lds_bytes, stream_);
    } else {
      if ((st = tiles_for(TK_WIRES, refs, 256, &t))) return st;
      if ((st = timed_begin(CKT_DISTRIBUTE_CHARGE, &a))) return st;
      e = launch_dsc_atomic(d_table_, (const Tile*)t.p, t.n, 256, stream_);
    }
  } else {
    if ((st = csr_nodes_ok(refs))) return st;
    return csr(refs, mode, false);
  }
  if (e != hipSuccess) return hip_fail(e, "distribute_charge launch");
  return timed_end(CKT_DISTRIBUTE_CHARGE, a);
}

int Engine::upv(const std::vector<PieceRef>& refs) {
  int st;
  if ((st = ensure_table())) return st;
  DevBuf t;
  if ((st = tiles_for(TK_NODES, refs, kUpvTile, &t))) return st;
  hipEvent_t a;
  if ((st = timed_begin(CKT_UPDATE_VOLTAGES, &a))) return st;
  uint64_t nodes = 0;
  for (const PieceRef& r : refs) nodes += slots_[r.slot]->pieces[r.piece].num_nodes;
  const bool nontemporal = nodes * kUpvBytesPerNode > kLastLevelCacheBytes;
  hipError_t e = launch_upv(d_table_, (const Tile*)t.p, t.n, 256, nontemporal, stream_);
  if (e != hipSuccess) return hip_fail(e, "update_voltages launch");
  return timed_end(CKT_UPDATE_VOLTAGES, a);
}

int Engine::sanity(const std::vector<PieceRef>& refs, uint64_t* bad) {
  int st;
  if ((st = ensure_table())) return st;
  DevBuf t;
  if ((st = tiles_for(TK_WIRES, refs, 256, &t))) return st;
  CKT_HIP(hipMemsetAsync(d_bad_, 0, sizeof(*d_bad_), stream_));
  hipError_t e = launch_sanity(d_table_, (const Tile*)t.p, t.n, 256, d_bad_, stream_);
  if (e != hipSuccess) return hip_fail(e, "sanity_check_wires launch");
  unsigned long long h = 0;
  CKT_HIP(hipMemcpyAsync(&h, d_bad_, sizeof(h), hipMemcpyDeviceToHost, stream_));
  CKT_HIP(hipStreamSynchronize(stream_));
  if (bad) *bad = h;
  return CKT_OK;
}

int Engine::nop() {
  hipError_t e = launch_nop(stream_);
  if (e != hipSuccess) return hip_fail(e, "nop launch");
  return CKT_OK;
}

int Engine::sync() {
  CKT_HIP(hipSetDevice(device_));
  CKT_HIP(hipStreamSynchronize(stream_));
  // Every copy out of the staging chunks has run.
  staging_chunk_ = 0;
  staging_off_ = 0;
  return CKT_OK;
}

// Copies `bytes` into pinned staging memory (new chunks as needed, 1 MiB and
// then twice the last one: pinning 64 MiB at the first tile list took 203 us
// and freeing it 692, 1 MiB takes 80 and 47) and returns its address, valid until
// the next sync().
int Engine::stage(const void* src, size_t bytes, void** out) {
  while (staging_chunk_ < staging_.size() &&
         staging_off_ + bytes > staging_[staging_chunk_].cap) {
    staging_chunk_++;
    staging_off_ = 0;
  }
  if (staging_chunk_ == staging_.size()) {
    const size_t grown = staging_.empty() ? 1ull << 20 : 2 * staging_.back().cap;
    PinnedChunk c{nullptr, std::max(bytes, std::min<size_t>(grown, 64ull << 20))};
    CKT_HIP(hipHostMalloc(&c.p, c.cap, hipHostMallocDefault));
    staging_.push_back(c);
    staging_off_ = 0;
  }
  uint8_t* dst = (uint8_t*)staging_[staging_chunk_].p + staging_off_;
  std::memcpy(dst, src, bytes);
  staging_off_ = align_up(staging_off_ + bytes, 256);
  *out = dst;
  return CKT_OK;
}

int Engine::add_generated_async(const ckt_gen_params_t* params, int32_t loops, uint32_t* id) {
  uint32_t N, W, P;
  int st = gen_validate(params, &N, &W, &P);
  if (st) return st;
  CKT_HIP(hipSetDevice(device_));
  const SlabLayout lay = SlabLayout::make(N, W, P);
  if (budget_ && in_use_ + lay.total > budget_)
    return fail(CKT_ERR_BUDGET, "circuit needs " + std::to_string(lay.total) +
                                    " bytes; budget has " + std::to_string(budget_ - in_use_) + " left");
  const size_t need = devgen_scratch_bytes(N, W);
  if (need == 0) return fail(CKT_ERR_HIP, "device generator scratch size query failed");
  if (need > devgen_scratch_cap_) {
    // Builds already enqueued use the old scratch.
    CKT_HIP(hipStreamSynchronize(stream_));
    if (devgen_scratch_) CKT_HIP(hipFree(devgen_scratch_));
    devgen_scratch_ = nullptr;
    devgen_scratch_cap_ = 0;
    CKT_HIP(hipMalloc(&devgen_scratch_, need));
    devgen_scratch_cap_ = need;
  }
  // From the stream's memory pool: allocated and, at removal, released in
  // stream order, without waiting for the device.
  void* slab = nullptr;
  hipError_t e = pool_ok_ ? hipMallocAsync(&slab, lay.total, stream_) : hipMalloc(&slab, lay.total);
  if (e != hipSuccess) return hip_fail(e, "allocating a circuit");
  std::vector<ckt_piece_t> pieces;
  if ((st = devgen_enqueue(params, lay, slab, devgen_scratch_, stream_, pieces))) {
    (void)hipStreamSynchronize(stream_);
    if (pool_ok_) (void)hipFreeAsync(slab, stream_);
    else (void)hipFree(slab);
    (void)hipStreamSynchronize(stream_);
    return st;
  }
  attach(slab, lay, N, W, P, pieces, loops, id, pool_ok_);
  return CKT_OK;
}

int Engine::run_graph(const std::vector<PieceRef>& refs, int policy, int mode, int times) {
  int st;
  if ((st = ensure_table())) return st;
  uint64_t key = fnv(1469598103934665603ull, refs.data(), refs.size() * sizeof(PieceRef));
  const int64_t cfg[14] = {policy,           mode,       steps_,          cnc_block_,
                           persistent_,      waves_per_simd_, dsc_atomic_impl_, fuse_dsc_,
                           wires_per_lane_,  tile_span_, tile_order_,     all_steps_,
                           (int64_t)generation_, loops_in_a_row_ >= kCachedLoops};
  key = fnv(key, cfg, sizeof(cfg));
  // Every buffer the launches use is created before any capture (an allocation
  // during capture is not allowed).
  if ((st = prefetch_tiles(refs, policy, mode))) return st;
  const bool timing = timing_;  // no events are recorded in this form
  timing_ = false;
  st = replay_loops(key, refs, policy, mode, times);
  timing_ = timing;
  return st;
}

// A graph of one loop takes 4 to 6 us a loop longer than its launches, one of
// kGraphLoops as long as they do, and capturing one takes as long as several
// loops of a small circuit; so fewer loops than that are launched directly.
int Engine::replay_loops(uint64_t key, const std::vector<PieceRef>& refs, int policy, int mode,
                         int times) {
  int st;
  for (int i = 0; i < times % kGraphLoops; i++)
    if ((st = launch_loop(refs, policy, mode))) return st;
  if (times < kGraphLoops) return CKT_OK;
  auto it = graphs_.find(key);
  hipGraphExec_t exec = nullptr;
  if (it == graphs_.end()) {
    CKT_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
    st = CKT_OK;
    for (int i = 0; i < kGraphLoops && !st; i++) st = launch_loop(refs, policy, mode);
    hipGraph_t graph = nullptr;
    hipError_t e = hipStreamEndCapture(stream_, &graph);
    if (st) {
      if (graph) (void)hipGraphDestroy(graph);
      return st;
    }
    if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
    graphs_[key] = exec;
  } else {
    exec = it->second;
  }
  for (int i = 0; i < times / kGraphLoops; i++) CKT_HIP(hipGraphLaunch(exec, stream_));
  return CKT_OK;
}

int Engine::set_option(int opt, int64_t v) {
  switch (opt) {
    case OPT_STEPS:
      if (v < 0 || v > (1 << 30)) return fail(CKT_ERR_INVALID_ARG, "steps out of range");
      steps_ = (int)v;
      return CKT_OK;
    case OPT_CNC_BLOCK:
      if (v != -1 && v != 64 && v != 128 && v != 256 && v != 512)
        return fail(CKT_ERR_INVALID_ARG, "block must be 64, 128, 256, 512 or -1");
      cnc_block_ = (int)v;
      return CKT_OK;
    case OPT_PERSISTENT: persistent_ = v < 0 ? -1 : v ? 1 : 0; return CKT_OK;
    case OPT_WAVES_PER_SIMD:
      if (v > 8 || v == 0) return fail(CKT_ERR_INVALID_ARG, "waves per SIMD must be 1..8 or -1");
      waves_per_simd_ = v < 0 ? -1 : (int)v;
      return CKT_OK;
    case OPT_DSC_ATOMIC_IMPL:
      if (v < 0 || v > 2) return fail(CKT_ERR_INVALID_ARG, "atomic implementation must be 0, 1 or 2");
      dsc_atomic_impl_ = (int)v;
      return CKT_OK;
    case OPT_FUSE_DSC: fuse_dsc_ = v < 0 ? -1 : v ? 1 : 0; return CKT_OK;
    case OPT_WIRES_PER_LANE:
      if (v != 1 && v != 2 && v != 4) return fail(CKT_ERR_INVALID_ARG, "wires per lane must be 1, 2 or 4");
      wires_per_lane_ = (int)v;
      return CKT_OK;
    case OPT_TILE_SPAN:
      if (v < 0 || v > 1) return fail(CKT_ERR_INVALID_ARG, "tile span must be 0 or 1");
      tile_span_ = (int)v;
      return CKT_OK;
    case OPT_TILE_ORDER:
      if (v < 0 || v > 2) return fail(CKT_ERR_INVALID_ARG, "tile order must be 0, 1 or 2");
      tile_order_ = (int)v;
      return CKT_OK;
    case OPT_ALL_STEPS: all_steps_ = v ? 1 : 0; return CKT_OK;
    default: return fail(CKT_ERR_INVALID_ARG, "unknown option");
  }
}

int64_t Engine::option(int opt) const {
  switch (opt) {
    case OPT_STEPS: return steps_;
    case OPT_CNC_BLOCK: return cnc_block_;
    case OPT_PERSISTENT: return persistent_;
    case OPT_WAVES_PER_SIMD: return waves_per_simd_;
    case OPT_DSC_ATOMIC_IMPL: return dsc_atomic_impl_;
    case OPT_FUSE_DSC: return fuse_dsc_;
    case OPT_WIRES_PER_LANE: return wires_per_lane_;
    case OPT_TILE_SPAN: return tile_span_;
    case OPT_TILE_ORDER: return tile_order_;
    case OPT_ALL_STEPS: return all_steps_;
    default: return -1;
  }
}

}  // namespace ckt
