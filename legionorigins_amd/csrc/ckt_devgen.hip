// ckt_devgen.hip -- load_circuit (apps/circuit/circuit.cc:1071-1288) built
// directly in HBM.
//
// The reference draws from one drand48 stream in a fixed order: three draws
// per node, then per wire six (in-piece) or seven (cross-piece) draws.  A
// node's first draw is a fixed jump from the seed, so every node is drawn
// independently.  A wire's first draw depends on how many earlier wires were
// cross-piece; that chain is cut into spans of the draw sequence whose effect
// on it is known for each of the seven ways in which it can enter them
// (gen_spans, scan_spans), so that every span's wires are drawn independently
// too.  The device then marks shared nodes, derives the locations, and builds
// the node -> (wire, end) index with a stable radix sort.  The slab is
// bit-identical to the host generator's image (ckt_generator.cpp +
// finalize_image).  The library is compiled with -ffp-contract=off, so the
// double expressions round exactly as on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include <rocprim/block/block_radix_sort.hpp>
#include <rocprim/device/device_radix_sort.hpp>

#include "ckt_engine.h"
#include "ckt_records.h"

namespace ckt {

namespace {

constexpr uint64_t kMask48 = (1ull << 48) - 1;
constexpr uint64_t kA = 0x5DEECE66Dull, kC = 0xBull;

// s -> a*s + c (mod 2^48): a number of steps of the drand48 recurrence.
struct Jump {
  uint64_t a, c;
};

// Jumps of 3 * 2^k draws: node i starts 3*i draws after the seed.
struct NodeJumps {
  Jump j[32];
};

// Jumps of 2^k draws (a circuit of 2^30 nodes and wires takes under 2^34).
struct DrawJumps {
  Jump j[34];
};

__host__ __device__ __forceinline__ uint64_t apply(const Jump& j, uint64_t s) {
  return (j.a * s + j.c) & kMask48;
}

// `first` then `second`.
Jump then(const Jump& first, const Jump& second) {
  return Jump{(second.a * first.a) & kMask48, (second.a * first.c + second.c) & kMask48};
}

Jump jump(uint64_t n) {
  Jump result{1, 0}, step{kA, kC};
  while (n) {
    if (n & 1) result = then(result, step);
    step = then(step, step);
    n >>= 1;
  }
  return result;
}

// One drand48 draw: advance, then return the new state / 2^48 (exact).
__device__ __forceinline__ double draw(uint64_t& s) {
  s = (kA * s + kC) & kMask48;
  return (double)s * 0x1p-48;
}

// Nodes (circuit.cc:1109-1136); the doubles round to float on assignment.
__global__ __launch_bounds__(256) void gen_nodes(uint32_t N, uint64_t seed_state, NodeJumps t,
                                                 float* __restrict__ voltage,
                                                 float* __restrict__ ncap,
                                                 float* __restrict__ leak) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= N) return;
  uint64_t s = seed_state;
  for (uint32_t k = 0, m = i; m; k++, m >>= 1)
    if (m & 1) s = apply(t.j[k], s);
  voltage[i] = (float)(2 * draw(s) - 1);
  ncap[i] = (float)(draw(s) + 1);
  leak[i] = (float)((double)0.1f * draw(s));
}

// The index of a small circuit in one workgroup: entry and node packed into
// 32 bits and sorted by node in LDS (stable, so entries keep their order), then
// each entry that starts a new node fills the rows up to it.  One launch for
// the device-wide sort's eight and the rows': generating 4 x 1024 wires takes 77
// us instead of 85.
constexpr uint32_t kSmallLanes = 512, kSmallEach = 16, kSmallEntries = kSmallLanes * kSmallEach;
constexpr unsigned kEntryBits = 13;
static_assert(kSmallEntries == 1u << kEntryBits, "an entry fits its bits");

__global__ __launch_bounds__(kSmallLanes) void index_small(DevCircuit c, unsigned bits) {
  using Sort = rocprim::block_radix_sort<uint32_t, kSmallLanes, kSmallEach>;
  __shared__ typename Sort::storage_type storage;
  __shared__ uint32_t last[kSmallLanes];
  const uint32_t t = threadIdx.x, E = 2 * c.num_wires;
  uint32_t item[kSmallEach];
#pragma unroll
  for (uint32_t u = 0; u < kSmallEach; u++) {
    // Past the end: the largest node, after every real entry of it.
    const uint32_t e = t * kSmallEach + u;
    uint32_t n = c.num_nodes - 1;
    if (e < E) n = (e & 1u) ? c.out_ptr[e >> 1] : c.in_ptr[e >> 1];
    item[u] = n << kEntryBits | e;
  }
  Sort().sort(item, storage, kEntryBits, kEntryBits + bits);
  last[t] = item[kSmallEach - 1] >> kEntryBits;
  __syncthreads();
  // Row n is the number of entries of nodes below n: each entry writes the
  // rows after its predecessor's node, up to its own.
  uint32_t next = t ? last[t - 1] + 1 : 0u;
#pragma unroll
  for (uint32_t u = 0; u < kSmallEach; u++) {
    const uint32_t i = t * kSmallEach + u, n = item[u] >> kEntryBits;
    if (i < E) c.csr_ent[i] = item[u] & (kSmallEntries - 1);
    if (i < E)
      for (; next <= n; next++) c.csr_row[next] = i;
    if (i + 1 == E)
      for (; next <= c.num_nodes; next++) c.csr_row[next] = E;
  }
  if (E == 0)
    for (uint32_t n = t; n <= c.num_nodes; n += kSmallLanes) c.csr_row[n] = 0;
}

// The wires' draws, position 0 the first wire's first draw, are cut into spans
// of kSpan positions, each into kSubs sub-spans.  A wire that starts at
// position p starts the next wire at p + 6, or at p + 7 if it is cross-piece
// (its fifth draw, circuit.cc:1167).  So a chain enters a sub-span at one of its
// first seven positions, and for each of them the walk through it (about 21
// wires, one dependent LDS read each) gives where it enters the next one and how
// many wires it started.  For 4.2 M wires the spans take 69 us, their composition
// 61 and the wires 98, bound by the walks' latency and the draws' 64-bit
// multiplies; the whole circuit is built in 1.0 ms, where one host core's walk of
// the chain made it 26.
constexpr uint32_t kSpan = 1024, kSubs = 8, kSub = kSpan / kSubs, kEntries = 7;

struct SpanScratch {
  // whether a wire that starts here is cross-piece; a lane writes four as a word
  alignas(4) uint8_t cross[kSpan];
  uint16_t step[kSubs][kEntries + 1];     // count << 3 | entry into the next sub-span
};
static_assert(alignof(SpanScratch) >= 4, "word stores into cross");

// Fills `sp` for span b: lane t takes positions 4 t .. 4 t + 3.  With `states`,
// also each position's state (before its draw).
template <bool kStates>
__device__ __forceinline__ void walk_span(uint32_t b, uint64_t first_state, const DrawJumps& t,
                                          const Jump& j5, int32_t pct, SpanScratch& sp,
                                          uint64_t* states) {
  const uint32_t p0 = 4u * threadIdx.x;
  uint64_t s = first_state;
  uint64_t m = (uint64_t)b * kSpan + p0;
  for (uint32_t k = 0; m; k++, m >>= 1)
    if (m & 1) s = apply(t.j[k], s);
  if (kStates) {
    uint64_t x = s;
#pragma unroll
    for (uint32_t k = 0; k < 4; k++) {
      states[p0 + k] = x;
      x = (kA * x + kC) & kMask48;
    }
  }
  s = apply(j5, s);
  uint32_t four = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4; k++) {
    const double u = (double)s * 0x1p-48;
    four |= ((100 * u) < pct ? 0u : 1u) << (8 * k);
    s = (kA * s + kC) & kMask48;
  }
  *(uint32_t*)(sp.cross + p0) = four;
  __syncthreads();
  if (threadIdx.x < kSubs * 8 && (threadIdx.x & 7u) < kEntries) {
    const uint32_t sub = threadIdx.x >> 3, end = (sub + 1) * kSub;
    uint32_t p = sub * kSub + (threadIdx.x & 7u), n = 0;
    for (; p < end; n++) p += 6u + sp.cross[p];
    sp.step[sub][threadIdx.x & 7u] = (uint16_t)(n << 3 | (p - end));
  }
  __syncthreads();
}

// Each span's step for each entry, as in SpanScratch::step, eight to a span.
__global__ __launch_bounds__(256) void gen_spans(uint64_t first_state, DrawJumps t, Jump j5,
                                                 int32_t pct, uint16_t* __restrict__ steps) {
  __shared__ SpanScratch sp;
  walk_span<false>(blockIdx.x, first_state, t, j5, pct, sp, nullptr);
  if (threadIdx.x < kEntries) {
    uint32_t e = threadIdx.x, n = 0;
    for (uint32_t sub = 0; sub < kSubs; sub++) {
      const uint32_t v = sp.step[sub][e];
      n += v >> 3;
      e = v & 7u;
    }
    steps[(size_t)blockIdx.x * 8 + threadIdx.x] = (uint16_t)(n << 3 | e);
  }
}

// Where the chain that starts at position 0 enters each span and the wire it
// starts first there.  One workgroup: lane t composes the steps of its share of
// the spans, 32 lanes compose 32 lanes' shares each, one lane walks those 32, and
// the same again downwards.
__global__ __launch_bounds__(1024) void scan_spans(uint32_t spans, const uint16_t* __restrict__ steps,
                                                   uint2* __restrict__ starts) {
  __shared__ uint32_t count[1024][kEntries], group_count[32][kEntries];
  __shared__ uint8_t exit_to[1024][kEntries], group_exit[32][kEntries];
  __shared__ uint32_t enter[1024], first[1024], group_enter[32], group_first[32];
  const uint32_t t = threadIdx.x, share = (spans + 1023u) / 1024u;
  const uint32_t lo = t * share < spans ? t * share : spans;
  const uint32_t hi = lo + share < spans ? lo + share : spans;
  auto at = [](const uint4& v, uint32_t e) {  // entry e of a span's eight steps
    const uint32_t w = e < 4 ? (e < 2 ? v.x : v.y) : (e < 6 ? v.z : v.w);
    return (w >> (16u * (e & 1u))) & 0xffffu;
  };
  const uint4* spans4 = (const uint4*)steps;
  uint32_t e[kEntries], n[kEntries];
#pragma unroll
  for (uint32_t k = 0; k < kEntries; k++) e[k] = k, n[k] = 0;
  for (uint32_t b = lo; b < hi; b++) {
    const uint4 v = spans4[b];
#pragma unroll
    for (uint32_t k = 0; k < kEntries; k++) {
      const uint32_t x = at(v, e[k]);
      n[k] += x >> 3;
      e[k] = x & 7u;
    }
  }
#pragma unroll
  for (uint32_t k = 0; k < kEntries; k++) {
    count[t][k] = n[k];
    exit_to[t][k] = (uint8_t)e[k];
  }
  __syncthreads();
  if (t < 32 * 8 && (t & 7u) < kEntries) {
    const uint32_t g = t >> 3;
    uint32_t x = t & 7u, c = 0;
    for (uint32_t k = g * 32; k < g * 32 + 32; k++) {
      c += count[k][x];
      x = exit_to[k][x];
    }
    group_count[g][t & 7u] = c;
    group_exit[g][t & 7u] = (uint8_t)x;
  }
  __syncthreads();
  if (t == 0) {
    uint32_t x = 0, c = 0;
    for (uint32_t g = 0; g < 32; g++) {
      group_enter[g] = x;
      group_first[g] = c;
      c += group_count[g][x];
      x = group_exit[g][x];
    }
  }
  __syncthreads();
  if (t < 32) {
    uint32_t x = group_enter[t], c = group_first[t];
    for (uint32_t k = t * 32; k < t * 32 + 32; k++) {
      enter[k] = x;
      first[k] = c;
      c += count[k][x];
      x = exit_to[k][x];
    }
  }
  __syncthreads();
  uint32_t x = enter[t], c = first[t];
  for (uint32_t b = lo; b < hi; b++) {
    starts[b] = make_uint2(x, c);
    const uint32_t v = at(spans4[b], x);
    c += v >> 3;
    x = v & 7u;
  }
}

// The wires that start in span blockIdx.x (circuit.cc:1147-1193).  A
// cross-piece wire's out-node becomes shared.
__global__ __launch_bounds__(256) void gen_wires(uint32_t W, uint64_t first_state, DrawJumps t,
                                                 Jump j5, const uint2* __restrict__ starts,
                                                 uint32_t P, uint32_t npp, uint32_t wpp, int32_t pct,
                                                 int32_t stable, float* __restrict__ ind,
                                                 float* __restrict__ res, float* __restrict__ wcap,
                                                 uint32_t* __restrict__ in_ptr,
                                                 uint32_t* __restrict__ out_ptr, uint8_t* locator) {
  __shared__ SpanScratch sp;
  __shared__ uint64_t states[kSpan];
  __shared__ uint16_t at[kSpan / 6 + 2];
  __shared__ uint16_t sub_enter[kSubs], sub_first[kSubs + 1];
  const uint2 start = starts[blockIdx.x];
  if (start.y >= W) return;
  walk_span<true>(blockIdx.x, first_state, t, j5, pct, sp, states);
  if (threadIdx.x == 0) {
    uint32_t e = start.x, n = 0;
    for (uint32_t sub = 0; sub < kSubs; sub++) {
      sub_enter[sub] = (uint16_t)e;
      sub_first[sub] = (uint16_t)n;
      const uint32_t v = sp.step[sub][e];
      n += v >> 3;
      e = v & 7u;
    }
    sub_first[kSubs] = (uint16_t)n;
  }
  __syncthreads();
  if (threadIdx.x < kSubs) {
    const uint32_t sub = threadIdx.x, end = (sub + 1) * kSub;
    uint32_t k = sub_first[sub];
    for (uint32_t p = sub * kSub + sub_enter[sub]; p < end; p += 6u + sp.cross[p])
      at[k++] = (uint16_t)p;
  }
  __syncthreads();
  if (threadIdx.x >= sub_first[kSubs] || threadIdx.x >= W - start.y) return;
  const uint32_t w = start.y + threadIdx.x;
  const uint32_t n = w / wpp;
  const uint32_t base = n * npp;
  uint64_t s = states[at[threadIdx.x]];
  float R, L, C;
  if (stable) {  // the same draws; inductance x 1e-6, capacitance U(0.001, 0.011)
    R = (float)(draw(s) * 10 + 1);
    L = (float)((draw(s) * 0.01 + 0.1) * 1e-6);
    C = (float)(draw(s) * 0.01 + 0.001);
  } else {
    R = (float)(draw(s) * 10 + 1);
    L = (float)(draw(s) * 0.01 + 0.1);
    C = (float)(draw(s) * 0.1);
  }
  const uint32_t in = base + (uint32_t)(int)(draw(s) * (double)npp);
  uint32_t out;
  if ((100 * draw(s)) < pct) {
    out = base + (uint32_t)(int)(draw(s) * (double)npp);
  } else {
    int nn = (int)(draw(s) * (double)((int)P - 1));
    if (nn >= (int)n) nn++;
    if (nn >= (int)P) nn -= (int)P;  // one piece: the pick wraps to piece 0
    out = (uint32_t)nn * npp + (uint32_t)(int)(draw(s) * (double)npp);
    locator[out] = 0;  // every writer stores the same value
  }
  ind[w] = L;
  res[w] = R;
  wcap[w] = C;
  in_ptr[w] = in;
  out_ptr[w] = out;
}

// Locations (find_location, circuit.cc:1051-1069) and the index entries:
// entry 2w+e (end e of wire w) is keyed by that end's node.
__global__ __launch_bounds__(256) void gen_locations(uint32_t W, uint32_t npp, uint32_t wpp,
                                                     const uint32_t* __restrict__ in_ptr,
                                                     const uint32_t* __restrict__ out_ptr,
                                                     const uint8_t* __restrict__ locator,
                                                     uint8_t* __restrict__ in_loc,
                                                     uint8_t* __restrict__ out_loc,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ vals) {
  const uint32_t w = blockIdx.x * 256u + threadIdx.x;
  if (w >= W) return;
  const uint32_t lo = (w / wpp) * npp;
  const uint32_t a = in_ptr[w], b = out_ptr[w];
  in_loc[w] = a - lo < npp ? (locator[a] ? CKT_PRIVATE_PTR : CKT_SHARED_PTR) : CKT_GHOST_PTR;
  out_loc[w] = b - lo < npp ? (locator[b] ? CKT_PRIVATE_PTR : CKT_SHARED_PTR) : CKT_GHOST_PTR;
  keys[2 * w] = a;
  keys[2 * w + 1] = b;
  vals[2 * w] = w << 1;
  vals[2 * w + 1] = (w << 1) | 1u;
}

// csr_row[n] = the first of the E sorted entries whose node is at least n, by
// one binary search per row: 24 us for 8.4 M entries of 1 M nodes, where an
// atomic count per entry and a scan of the counts took 296.
__global__ __launch_bounds__(256) void index_rows(uint32_t N, uint32_t E,
                                                  const uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ row,
                                                  const LoadFaults* faults,
                                                  LoadFaults* host_faults) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n == 0 && faults) *host_faults = *faults;
  if (n > N) return;
  uint32_t lo = 0, hi = E;
  while (lo < hi) {
    const uint32_t mid = lo + ((hi - lo) >> 1);
    if (keys[mid] < n) lo = mid + 1;
    else hi = mid;
  }
  row[n] = lo;
}

__global__ __launch_bounds__(256) void fill_bytes(uint8_t* p, uint8_t v, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) p[i] = v;
}

// Piece n owns wires [n*wpp, (n+1)*wpp) and nodes [n*npp, (n+1)*npp)
// (circuit.cc:1092-1104,1140-1157).
__global__ __launch_bounds__(256) void gen_pieces(uint32_t P, uint32_t npp, uint32_t wpp,
                                                  ckt_piece_t* pieces) {
  const uint32_t n = blockIdx.x * 256u + threadIdx.x;
  if (n < P) pieces[n] = ckt_piece_t{n * wpp, wpp, n * npp, npp};
}

uint32_t grid_for(size_t n) { return (uint32_t)((n + 255) / 256); }

uint64_t seed_state_of(const ckt_gen_params_t* p) {
  return ((uint64_t)(uint32_t)p->random_seed << 16) | 0x330Eull;
}

// Slab arrays the kernels write.
struct SlabView {
  uint8_t* b;
  const SlabLayout& L;
  float* f(size_t off) const { return (float*)(b + off); }
  uint32_t* u(size_t off) const { return (uint32_t*)(b + off); }
};

// Zero the slab, mark every node private, draw the nodes, write the pieces.
int enqueue_nodes(const ckt_gen_params_t* p, uint32_t N, uint32_t P, const SlabView& v,
                  hipStream_t s) {
  CKT_HIP(launch_fill_u32((uint32_t*)v.b, 0u, v.L.total / 4, s));
  hipLaunchKernelGGL(fill_bytes, dim3(grid_for(N)), dim3(256), 0, s, v.b + v.L.locator,
                     (uint8_t)1, N);
  CKT_HIP(hipGetLastError());
  NodeJumps t{};
  for (int k = 0; k < 32; k++) t.j[k] = jump(3ull << k);
  hipLaunchKernelGGL(gen_nodes, dim3(grid_for(N)), dim3(256), 0, s, N, seed_state_of(p), t,
                     v.f(v.L.voltage), v.f(v.L.ncap), v.f(v.L.leak));
  CKT_HIP(hipGetLastError());
  hipLaunchKernelGGL(gen_pieces, dim3(grid_for(P)), dim3(256), 0, s, P,
                     (uint32_t)p->nodes_per_piece, (uint32_t)p->wires_per_piece,
                     (ckt_piece_t*)(v.b + v.L.pieces));
  CKT_HIP(hipGetLastError());
  return CKT_OK;
}

uint32_t span_count(uint32_t W) { return (uint32_t)((7ull * W + kSpan - 1) / kSpan); }

size_t align256(size_t x) { return (x + 255) / 256 * 256; }

// Scratch of the wires' draws: eight steps and a start per span.
size_t span_scratch_bytes(uint32_t W) {
  return align256((size_t)span_count(W) * 8 * sizeof(uint16_t)) +
         align256((size_t)span_count(W) * sizeof(uint2));
}

int enqueue_wires(const ckt_gen_params_t* p, uint32_t N, uint32_t W, uint32_t P, void* scratch,
                  const SlabView& v, hipStream_t s) {
  if (W == 0) return CKT_OK;
  const uint32_t spans = span_count(W);
  uint16_t* steps = (uint16_t*)scratch;
  uint2* starts = (uint2*)((uint8_t*)scratch + align256((size_t)spans * 8 * sizeof(uint16_t)));
  DrawJumps t{};
  for (int k = 0; k < 34; k++) t.j[k] = jump(1ull << k);
  const uint64_t first = apply(jump(3ull * N), seed_state_of(p));
  const Jump j5 = jump(5);
  const int32_t pct = p->pct_wire_in_piece;
  hipLaunchKernelGGL(gen_spans, dim3(spans), dim3(256), 0, s, first, t, j5, pct, steps);
  hipLaunchKernelGGL(scan_spans, dim3(1), dim3(1024), 0, s, spans, steps, starts);
  hipLaunchKernelGGL(gen_wires, dim3(spans), dim3(256), 0, s, W, first, t, j5, starts, P,
                     (uint32_t)p->nodes_per_piece, (uint32_t)p->wires_per_piece, pct,
                     (int32_t)(p->profile == CKT_PROFILE_STABLE), v.f(v.L.ind), v.f(v.L.res),
                     v.f(v.L.wcap), v.u(v.L.in_ptr), v.u(v.L.out_ptr), v.b + v.L.locator);
  CKT_HIP(hipGetLastError());
  return CKT_OK;
}

unsigned key_bits(uint32_t N) {
  unsigned bits = 1;
  while (bits < 32 && (1ull << bits) < N) bits++;
  return bits;
}

// Circuits of up to 4096 wires and 2^15 nodes (with many more nodes than entries
// the rows between them, written by one lane, would take longer than the launches
// saved).
bool index_is_small(uint32_t N, uint32_t W) {
  return 2ull * W <= kSmallEntries && N <= 1u << 15;
}

// Locations, then the index (from the entries, or for a small circuit from
// the pointers).
int enqueue_index(const ckt_gen_params_t* p, uint32_t N, uint32_t W, const SlabView& v,
                  const IndexScratch& sc, hipStream_t s) {
  if (W) {
    hipLaunchKernelGGL(gen_locations, dim3(grid_for(W)), dim3(256), 0, s, W,
                       (uint32_t)p->nodes_per_piece, (uint32_t)p->wires_per_piece,
                       v.u(v.L.in_ptr), v.u(v.L.out_ptr), v.b + v.L.locator, v.b + v.L.in_loc,
                       v.b + v.L.out_loc, sc.keys, sc.vals);
    CKT_HIP(hipGetLastError());
  }
  DevCircuit c{};
  c.num_nodes = N;
  c.num_wires = W;
  c.csr_row = v.u(v.L.csr_row);
  c.csr_ent = v.u(v.L.csr_ent);
  c.in_ptr = v.u(v.L.in_ptr);
  c.out_ptr = v.u(v.L.out_ptr);
  if (index_is_small(N, W)) {
    hipLaunchKernelGGL(index_small, dim3(1), dim3(kSmallLanes), 0, s, c, key_bits(N));
    CKT_HIP(hipGetLastError());
    return CKT_OK;
  }
  if (int st = index_sort(c, sc, s)) return st;
  CKT_HIP(launch_index_rows(c, sc, nullptr, nullptr, s));
  return CKT_OK;
}

}  // namespace

int index_scratch(uint32_t N, uint32_t W, void* base, IndexScratch* sc, size_t* bytes) {
  size_t sort_bytes = 0;
  if (W)
    CKT_HIP(rocprim::radix_sort_pairs(nullptr, sort_bytes, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                      (uint32_t*)nullptr, (uint32_t*)nullptr, (size_t)2 * W, 0,
                                      key_bits(N), (hipStream_t)0));
  const size_t e = align256((size_t)2 * W * sizeof(uint32_t));
  const size_t w = align256(std::max<size_t>(sort_bytes, 16));
  *bytes = 3 * e + w;
  if (base && sc) {
    uint8_t* b = (uint8_t*)base;
    sc->keys = (uint32_t*)b;
    sc->vals = (uint32_t*)(b + e);
    sc->keys_sorted = (uint32_t*)(b + 2 * e);
    sc->work = b + 3 * e;
    sc->sort_bytes = sort_bytes;
  }
  return CKT_OK;
}

int index_sort(const DevCircuit& c, const IndexScratch& sc, hipStream_t s) {
  size_t sort_bytes = sc.sort_bytes;
  if (c.num_wires)
    CKT_HIP(rocprim::radix_sort_pairs(sc.work, sort_bytes, sc.keys, sc.keys_sorted, sc.vals,
                                      c.csr_ent, (size_t)2 * c.num_wires, 0,
                                      key_bits(c.num_nodes), s));
  return CKT_OK;
}

hipError_t launch_index_rows(const DevCircuit& c, const IndexScratch& sc, const LoadFaults* faults,
                             LoadFaults* host_faults, hipStream_t s) {
  hipLaunchKernelGGL(index_rows, dim3(grid_for((size_t)c.num_nodes + 1)), dim3(256), 0, s,
                     c.num_nodes, 2 * c.num_wires, sc.keys_sorted, c.csr_row, faults, host_faults);
  return hipGetLastError();
}

size_t devgen_scratch_bytes(uint32_t N, uint32_t W) {
  size_t index = 0;
  return index_scratch(N, W, nullptr, nullptr, &index) ? 0 : span_scratch_bytes(W) + index;
}

int devgen_enqueue(const ckt_gen_params_t* p, const SlabLayout& L, void* slab, void* scratch,
                   hipStream_t s, std::vector<ckt_piece_t>& pieces) {
  uint32_t N, W, P;
  int st = gen_validate(p, &N, &W, &P);
  if (st) return st;
  const SlabView v{(uint8_t*)slab, L};
  if ((st = enqueue_nodes(p, N, P, v, s))) return st;
  if ((st = enqueue_wires(p, N, W, P, scratch, v, s))) return st;
  size_t bytes = 0;
  IndexScratch sc{};
  if ((st = index_scratch(N, W, (uint8_t*)scratch + span_scratch_bytes(W), &sc, &bytes))) return st;
  if ((st = enqueue_index(p, N, W, v, sc, s))) return st;
  pieces.resize(P);
  for (uint32_t n = 0; n < P; n++)
    pieces[n] = ckt_piece_t{n * (uint32_t)p->wires_per_piece, (uint32_t)p->wires_per_piece,
                            n * (uint32_t)p->nodes_per_piece, (uint32_t)p->nodes_per_piece};
  return CKT_OK;
}

}  // namespace ckt
