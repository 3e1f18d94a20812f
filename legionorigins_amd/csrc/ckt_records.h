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

// The node -> (wire, end) index under construction, in scratch memory: entry
// 2 w + e is keyed by the node at end e of wire w (ckt_devgen.hip).
struct IndexScratch {
  uint32_t *keys, *vals, *keys_sorted;
  void* work;
  size_t sort_bytes;
};
// Bytes of scratch for N nodes and W wires; with `base`, carves *sc from it.
int index_scratch(uint32_t N, uint32_t W, void* base, IndexScratch* sc, size_t* bytes);
// Sorts the entries (stable, so each node's stay in (wire, in-before-out)
// order), then finds the rows.  The second also copies *faults, if not NULL, to
// *host_faults (pinned).
int index_sort(const DevCircuit& c, const IndexScratch& sc, hipStream_t s);
hipError_t launch_index_rows(const DevCircuit& c, const IndexScratch& sc, const LoadFaults* faults,
                             LoadFaults* host_faults, hipStream_t s);


// What a load reads besides the wires, in one piece of pinned memory: nodes,
// locator (if `locator`), pieces, and the pieces' first workgroups, each on a
// 16-byte boundary.
struct LoadRest {
  uint32_t nodes, pieces, blocks;  // counts
  bool locator;
  size_t locator_at, pieces_at, blocks_at, bytes;
  LoadRest(uint32_t N, bool has_locator, uint32_t P, uint32_t num_blocks)
      : nodes(N), pieces(P), blocks(num_blocks), locator(has_locator),
        locator_at(sizeof(ckt_node_t) * (size_t)N),
        pieces_at(locator_at + (has_locator ? ((size_t)N * 4 + 15) / 16 * 16 : 0)),
        blocks_at(pieces_at + sizeof(ckt_piece_t) * (size_t)P),
        bytes(blocks_at + 4 * (size_t)num_blocks) {}
};
// Unpacks it (`blocks` into device memory) and clears *faults.
hipError_t launch_unpack_rest(const void* host, const LoadRest& r, const DevCircuit& c,
                              uint32_t* blocks, LoadFaults* faults, hipStream_t s);

hipError_t launch_clear_faults(LoadFaults* faults, hipStream_t s);
hipError_t launch_unpack_nodes(const ckt_node_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, hipStream_t s);
// Records first.. into the wire arrays, and their index entries; the launch
// that holds the last wire also zeroes the padding up to the wire stride.
hipError_t launch_unpack_wires(const ckt_wire_t* host, uint32_t first, uint32_t n,
                               const DevCircuit& c, const IndexScratch& sc, LoadFaults* faults,
                               hipStream_t s);
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
// All of a small circuit's wires and nodes in one launch.
hipError_t launch_pack_all(ckt_wire_t* wires, ckt_node_t* nodes, const DevCircuit& c,
                           hipStream_t s);
hipError_t launch_pack_locator(int32_t* host, uint32_t first, uint32_t n, const DevCircuit& c,
                               hipStream_t s);
hipError_t launch_copy_words(uint32_t* host, const uint32_t* dev, uint32_t n, hipStream_t s);

}  // namespace ckt
