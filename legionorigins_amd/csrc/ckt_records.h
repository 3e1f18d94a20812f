// ckt_records.h -- circuits moved between the caller's reference-layout
// records (host memory) and the structure-of-arrays slab in HBM.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include "ckt_internal.h"

namespace ckt {

// Kernels between pinned host memory (read and written over PCIe) and a
// slab.  `first` and `n` count records; `host` holds records first..first+n-1.

// What load found wrong, in device memory: the lowest wire index (or piece
// << 32 | wire) of each kind, all ones if none.
struct LoadFaults {
  unsigned long long location;  // a PointerLocation that is none
  unsigned long long pointer;   // a pointer past the last node
  unsigned long long foreign;   // a private node of another piece reached
};

hipError_t launch_unpack_nodes(const ckt_node_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, hipStream_t s);
// Records first.. into the wire arrays; the launch that holds the last wire
// also zeroes the padding up to the wire stride.
hipError_t launch_unpack_wires(const ckt_wire_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, LoadFaults* faults, hipStream_t s);
hipError_t launch_unpack_locator(const int32_t* host, uint32_t first, uint32_t n,
                                 const DevCircuit& c, hipStream_t s);
// The locator of a circuit loaded without one: 0 for every node that a wire
// names as a shared or ghost end, else 1.
hipError_t launch_derive_locator(const DevCircuit& c, hipStream_t s);
// Wires of pieces [0, num_pieces) of `ix` (over wires) that reach a private
// node of another piece.
hipError_t launch_check_pieces(const PieceIndex& ix, uint32_t blocks, const DevCircuit& c,
                               LoadFaults* faults, hipStream_t s);

hipError_t launch_pack_nodes(ckt_node_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                             hipStream_t s);
hipError_t launch_pack_wires(ckt_wire_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                             hipStream_t s);
hipError_t launch_pack_locator(int32_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                               hipStream_t s);
hipError_t launch_copy_words(uint32_t* host, const uint32_t* dev, uint32_t n, hipStream_t s);

// The node -> (wire, end) index of a slab whose pointers are written
// (ckt_devgen.hip): scratch bytes, and the build enqueued on `s`.
size_t index_scratch_bytes(uint32_t N, uint32_t W);
int index_enqueue(const DevCircuit& c, void* scratch, hipStream_t s);

}  // namespace ckt
