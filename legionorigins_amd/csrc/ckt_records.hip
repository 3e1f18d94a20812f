// ckt_records.hip -- kernels between reference-layout records in pinned host
// memory and the structure-of-arrays slab.
//
// Bound by PCIe (about 50 GB/s each way): the kernels read and write the
// records in place over the bus, 16 contiguous bytes per lane, and exchange
// rows and columns in LDS, so that the slab side is coalesced too and neither
// a second copy of the records in HBM nor a pass over them on the host is
// needed.  Measured: 2 MiB of wire records in 40 us either way (52 GB/s); a
// circuit of 4.2 M wires and 1 M nodes loads in 13.0 ms and stores in 12.6 (0.77
// without its wires), where a pass over the records on one host thread and one
// copy of the whole slab took 470 and 175 (111).
#include <hip/hip_runtime.h>

#include "ckt_index.h"
#include "ckt_records.h"

namespace ckt {

namespace {

constexpr uint32_t kTile = 256;             // wires per workgroup
constexpr uint32_t kWords = 32;             // words of a wire record
constexpr uint32_t kRow = kTile + 1;        // LDS row stride, off the bank period
static_assert(sizeof(ckt_wire_t) == 4 * kWords, "wire record layout");

// Word offsets in a wire record (ckt_wire_t).
constexpr uint32_t kInPtr = 0, kOutPtr = 1, kInLoc = 2, kOutLoc = 3, kInd = 4, kRes = 5, kCur = 6,
                   kCap = 16, kVol = 17, kPad = 26;

uint32_t grid_for(size_t n) { return (uint32_t)((n + 255) / 256); }

}  // namespace

__global__ __launch_bounds__(256) void unpack_nodes_kernel(const float4* __restrict__ host,
                                                           uint32_t first, uint32_t n,
                                                           DevCircuit c) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float4 v = host[i];  // charge, voltage, capacitance, leakage
  c.charge[first + i] = v.x;
  c.voltage[first + i] = v.y;
  c.ncap[first + i] = v.z;
  c.leak[first + i] = v.w;
}

__global__ __launch_bounds__(256) void unpack_rest_kernel(const uint8_t* __restrict__ host,
                                                          LoadRest r, DevCircuit c,
                                                          uint32_t* __restrict__ blocks,
                                                          LoadFaults* faults) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i == 0) *faults = LoadFaults{~0ull, ~0ull, ~0ull};
  if (i < r.nodes) {
    const float4 v = ((const float4*)host)[i];  // charge, voltage, capacitance, leakage
    c.charge[i] = v.x;
    c.voltage[i] = v.y;
    c.ncap[i] = v.z;
    c.leak[i] = v.w;
    if (r.locator) c.locator[i] = ((const int32_t*)(host + r.locator_at))[i] ? 1 : 0;
  }
  if (i < r.pieces) ((uint4*)c.pieces)[i] = ((const uint4*)(host + r.pieces_at))[i];
  if (i < r.blocks) blocks[i] = ((const uint32_t*)(host + r.blocks_at))[i];
}

__global__ void clear_faults_kernel(LoadFaults* faults) {
  *faults = LoadFaults{~0ull, ~0ull, ~0ull};
}

__global__ __launch_bounds__(256) void pack_nodes_kernel(float4* __restrict__ host, uint32_t first,
                                                         uint32_t n, DevCircuit c) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  host[i] = make_float4(c.charge[first + i], c.voltage[first + i], c.ncap[first + i],
                        c.leak[first + i]);
}

__global__ __launch_bounds__(256) void unpack_wires_kernel(const uint4* __restrict__ host,
                                                           uint32_t first, uint32_t n,
                                                           DevCircuit c, IndexScratch sc,
                                                           LoadFaults* faults) {
  __shared__ uint32_t rec[kWords * kRow];
  const uint32_t base = blockIdx.x * kTile;
  const uint32_t here = base < n ? (n - base < kTile ? n - base : kTile) : 0u;
#pragma unroll
  for (uint32_t k = 0; k < 8; k++) {  // eight 16-byte parts per record
    const uint32_t q = k * kTile + threadIdx.x, w = q >> 3, part = 4u * (q & 7u);
    uint4 v = make_uint4(0, 0, 0, 0);
    if (w < here) v = host[(size_t)base * 8 + q];
    rec[(part + 0) * kRow + w] = v.x;
    rec[(part + 1) * kRow + w] = v.y;
    rec[(part + 2) * kRow + w] = v.z;
    rec[(part + 3) * kRow + w] = v.w;
  }
  __syncthreads();
  const uint32_t t = threadIdx.x, w = first + base + t;
  if (w >= c.ws) return;
  // past the last wire of the circuit: the zeroed padding of the stride
  if (t >= here && w < c.num_wires) return;
  auto word = [&](uint32_t k) { return rec[k * kRow + t]; };
  auto real = [&](uint32_t k) { return __uint_as_float(rec[k * kRow + t]); };
#pragma unroll
  for (uint32_t s = 0; s < kSeg; s++) c.cur[(size_t)s * c.ws + w] = real(kCur + s);
#pragma unroll
  for (uint32_t s = 0; s < kSeg - 1; s++) c.vol[(size_t)s * c.ws + w] = real(kVol + s);
  c.ind[w] = real(kInd);
  c.res[w] = real(kRes);
  c.wcap[w] = real(kCap);
  const uint32_t a = word(kInPtr), b = word(kOutPtr), la = word(kInLoc), lb = word(kOutLoc);
  c.in_ptr[w] = a;
  c.out_ptr[w] = b;
  c.in_loc[w] = (uint8_t)la;
  c.out_loc[w] = (uint8_t)lb;
  if (t < here) {
    // an invalid pointer is refused after the build; its entry only has to
    // stay in range
    const uint32_t last = c.num_nodes - 1;
    *(uint2*)(sc.keys + 2 * (size_t)w) = make_uint2(a < last ? a : last, b < last ? b : last);
    *(uint2*)(sc.vals + 2 * (size_t)w) = make_uint2(w << 1, (w << 1) | 1u);
    if (la > 2u || lb > 2u) atomicMin(&faults->location, (unsigned long long)w);
    if (a >= c.num_nodes || b >= c.num_nodes) atomicMin(&faults->pointer, (unsigned long long)w);
  }
}

__device__ __forceinline__ void pack_tile(uint4* __restrict__ host, uint32_t tile, uint32_t first,
                                          uint32_t n, const DevCircuit& c) {
  __shared__ uint32_t rec[kWords * kRow];
  const uint32_t base = tile * kTile;
  const uint32_t here = n - base < kTile ? n - base : kTile;
  const uint32_t t = threadIdx.x;
  if (t < here) {
    const uint32_t w = first + base + t;
    auto put = [&](uint32_t k, uint32_t v) { rec[k * kRow + t] = v; };
#pragma unroll
    for (uint32_t s = 0; s < kSeg; s++) put(kCur + s, __float_as_uint(c.cur[(size_t)s * c.ws + w]));
#pragma unroll
    for (uint32_t s = 0; s < kSeg - 1; s++)
      put(kVol + s, __float_as_uint(c.vol[(size_t)s * c.ws + w]));
    put(kInd, __float_as_uint(c.ind[w]));
    put(kRes, __float_as_uint(c.res[w]));
    put(kCap, __float_as_uint(c.wcap[w]));
    put(kInPtr, c.in_ptr[w]);
    put(kOutPtr, c.out_ptr[w]);
    put(kInLoc, c.in_loc[w]);
    put(kOutLoc, c.out_loc[w]);
#pragma unroll
    for (uint32_t k = kPad; k < kWords; k++) put(k, 0u);
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < 8; k++) {
    const uint32_t q = k * kTile + t, w = q >> 3, part = 4u * (q & 7u);
    if (w < here)
      host[(size_t)base * 8 + q] =
          make_uint4(rec[(part + 0) * kRow + w], rec[(part + 1) * kRow + w],
                     rec[(part + 2) * kRow + w], rec[(part + 3) * kRow + w]);
  }
}

__global__ __launch_bounds__(256) void pack_wires_kernel(uint4* __restrict__ host, uint32_t first,
                                                         uint32_t n, DevCircuit c) {
  pack_tile(host, blockIdx.x, first, n, c);
}

// Workgroups [0, wire_tiles) pack wires, the others nodes.
__global__ __launch_bounds__(256) void pack_all_kernel(uint4* __restrict__ wires,
                                                       float4* __restrict__ nodes,
                                                       uint32_t wire_tiles, DevCircuit c) {
  if (blockIdx.x < wire_tiles) {
    pack_tile(wires, blockIdx.x, 0, c.num_wires, c);
    return;
  }
  const uint32_t i = (blockIdx.x - wire_tiles) * 256u + threadIdx.x;
  if (i < c.num_nodes) nodes[i] = make_float4(c.charge[i], c.voltage[i], c.ncap[i], c.leak[i]);
}

__global__ __launch_bounds__(256) void unpack_locator_kernel(const int32_t* __restrict__ host,
                                                             uint32_t first, uint32_t n,
                                                             uint8_t* __restrict__ locator) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) locator[first + i] = host[i] ? 1 : 0;
}

__global__ __launch_bounds__(256) void pack_locator_kernel(int32_t* __restrict__ host,
                                                           uint32_t first, uint32_t n,
                                                           const uint8_t* __restrict__ locator) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) host[i] = locator[first + i];
}

__global__ __launch_bounds__(256) void private_nodes_kernel(uint8_t* __restrict__ locator,
                                                            uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) locator[i] = 1;
}

__global__ __launch_bounds__(256) void shared_ends_kernel(DevCircuit c) {
  const uint32_t w = blockIdx.x * 256u + threadIdx.x;
  if (w >= c.num_wires) return;
  const uint32_t a = c.in_ptr[w], b = c.out_ptr[w];
  // every writer stores the same value
  if (c.in_loc[w] != CKT_PRIVATE_PTR && a < c.num_nodes) c.locator[a] = 0;
  if (c.out_loc[w] != CKT_PRIVATE_PTR && b < c.num_nodes) c.locator[b] = 0;
}

__global__ __launch_bounds__(256) void check_pieces_kernel(PieceIndex ix, DevCircuit c,
                                                           LoadFaults* faults) {
  uint32_t k;
  const uint32_t pi = piece_of_block(ix.first_block, ix.num_pieces, blockIdx.x, threadIdx.x, &k);
  const ckt_piece_t p = ix.pieces[pi];
  if (k >= p.num_wires) return;
  const uint32_t w = p.first_wire + k;
  bool bad = false;
  const uint32_t ends[2] = {c.in_ptr[w], c.out_ptr[w]};
#pragma unroll
  for (int e = 0; e < 2; e++)
    bad |= ends[e] < c.num_nodes && ends[e] - p.first_node >= p.num_nodes && c.locator[ends[e]];
  if (bad) atomicMin(&faults->foreign, (unsigned long long)pi << 32 | w);
}

__global__ __launch_bounds__(256) void copy_words_kernel(uint32_t* __restrict__ host,
                                                         const uint32_t* __restrict__ dev,
                                                         uint32_t n) {
  const uint32_t i = (blockIdx.x * 256u + threadIdx.x) * 4u;
  if (i + 4 <= n) {
    *(uint4*)(host + i) = *(const uint4*)(dev + i);
  } else {
    for (uint32_t k = i; k < n; k++) host[k] = dev[k];
  }
}

hipError_t launch_unpack_rest(const void* host, const LoadRest& r, const DevCircuit& c,
                              uint32_t* blocks, LoadFaults* faults, hipStream_t s) {
  uint32_t n = r.nodes > r.pieces ? r.nodes : r.pieces;
  n = n > r.blocks ? n : r.blocks;
  hipLaunchKernelGGL(unpack_rest_kernel, dim3(grid_for(n)), dim3(256), 0, s, (const uint8_t*)host, r,
                     c, blocks, faults);
  return hipGetLastError();
}

hipError_t launch_clear_faults(LoadFaults* faults, hipStream_t s) {
  hipLaunchKernelGGL(clear_faults_kernel, dim3(1), dim3(1), 0, s, faults);
  return hipGetLastError();
}

hipError_t launch_unpack_nodes(const ckt_node_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, hipStream_t s) {
  hipLaunchKernelGGL(unpack_nodes_kernel, dim3(grid_for(n)), dim3(256), 0, s, (const float4*)host,
                     first, n, c);
  return hipGetLastError();
}

hipError_t launch_unpack_wires(const ckt_wire_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, const IndexScratch& sc, LoadFaults* faults,
                               hipStream_t s) {
  const uint32_t lanes = first + n == c.num_wires ? c.ws - first : n;
  hipLaunchKernelGGL(unpack_wires_kernel, dim3(grid_for(lanes)), dim3(256), 0, s,
                     (const uint4*)host, first, n, c, sc, faults);
  return hipGetLastError();
}

hipError_t launch_unpack_locator(const int32_t* host, uint32_t first, uint32_t n,
                                 const DevCircuit& c, hipStream_t s) {
  hipLaunchKernelGGL(unpack_locator_kernel, dim3(grid_for(n)), dim3(256), 0, s, host, first, n,
                     c.locator);
  return hipGetLastError();
}

hipError_t launch_derive_locator(const DevCircuit& c, hipStream_t s) {
  hipLaunchKernelGGL(private_nodes_kernel, dim3(grid_for(c.num_nodes)), dim3(256), 0, s, c.locator,
                     c.num_nodes);
  if (c.num_wires)
    hipLaunchKernelGGL(shared_ends_kernel, dim3(grid_for(c.num_wires)), dim3(256), 0, s, c);
  return hipGetLastError();
}

hipError_t launch_check_pieces(const PieceIndex& ix, uint32_t blocks, const DevCircuit& c,
                               LoadFaults* faults, hipStream_t s) {
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(check_pieces_kernel, dim3(blocks), dim3(256), 0, s, ix, c, faults);
  return hipGetLastError();
}

hipError_t launch_pack_nodes(ckt_node_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                             hipStream_t s) {
  hipLaunchKernelGGL(pack_nodes_kernel, dim3(grid_for(n)), dim3(256), 0, s, (float4*)host, first, n,
                     c);
  return hipGetLastError();
}

hipError_t launch_pack_wires(ckt_wire_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                             hipStream_t s) {
  hipLaunchKernelGGL(pack_wires_kernel, dim3(grid_for(n)), dim3(256), 0, s, (uint4*)host, first, n,
                     c);
  return hipGetLastError();
}

hipError_t launch_pack_all(ckt_wire_t* wires, ckt_node_t* nodes, const DevCircuit& c,
                           hipStream_t s) {
  const uint32_t tiles = grid_for(c.num_wires);
  hipLaunchKernelGGL(pack_all_kernel, dim3(tiles + grid_for(c.num_nodes)), dim3(256), 0, s,
                     (uint4*)wires, (float4*)nodes, tiles, c);
  return hipGetLastError();
}

hipError_t launch_pack_locator(int32_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                               hipStream_t s) {
  hipLaunchKernelGGL(pack_locator_kernel, dim3(grid_for(n)), dim3(256), 0, s, host, first, n,
                     c.locator);
  return hipGetLastError();
}

hipError_t launch_copy_words(uint32_t* host, const uint32_t* dev, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(copy_words_kernel, dim3(grid_for(((size_t)n + 3) / 4)), dim3(256), 0, s, host,
                     dev, n);
  return hipGetLastError();
}

}  // namespace ckt
