// Host checks of piece_check_blocks (ckt_index.h): a load's piece table either
// fits a launch or is refused.  Built and run by tests/test_load_limits.py;
// exits non-zero on a failure, after printing it.
#include <cstdio>
#include <vector>

#include "ckt_index.h"

struct Piece {
  uint32_t first_wire, num_wires, first_node, num_nodes;
};

static int fails = 0;

static void check(const char* what, const std::vector<Piece>& p, uint32_t N, uint32_t W, bool fits,
                  uint32_t good) {
  std::vector<uint32_t> first(1, 0u);
  uint32_t got = ~0u;
  const bool f = ckt::piece_check_blocks(p.data(), (uint32_t)p.size(), N, W, &first, &got);
  bool ok = f == fits;
  if (ok && f) {
    ok = got == good && first.size() == good + 1u;
    for (uint32_t k = 0; ok && k < good; k++)
      ok = first[k + 1] - first[k] == (p[k].num_wires + 255u) / 256u;
    // the launch: HIP refuses 2^32 lanes or more in a dimension
    ok = ok && (uint64_t)first.back() * 256u < 1ull << 32;
  }
  if (!ok) {
    std::printf("FAIL %s: fits %d, good %u\n", what, (int)f, got);
    fails++;
  }
}

int main() {
  const uint32_t W = 1u << 22, N = 1u << 20, all = W / 256;  // 16384 workgroups a piece
  const Piece whole{0, W, 0, N};
  check("no pieces", {}, N, W, true, 0);
  check("one", {whole}, N, W, true, 1);
  check("ragged", {{0, 1, 0, 1}, {1, 0, 0, 0}, {1, 257, 0, 1}}, N, W, true, 3);
  check("past the wires", {whole, {1, W, 0, N}, whole}, N, W, true, 1);
  check("past the nodes", {whole, whole, {0, W, 1, N}}, N, W, true, 2);
  // overlapping pieces, each over every wire: 2^24 - 1 workgroups are the most
  const uint32_t most = (1u << 24) / all;
  check("under the limit", std::vector<Piece>(most - 1, whole), N, W, true, most - 1);
  std::vector<Piece> p(most - 1, whole);
  p.push_back({0, W - 256, 0, N});
  check("at the limit", p, N, W, true, most);
  check("past the limit", std::vector<Piece>(most, whole), N, W, false, 0);
  check("1025 pieces", std::vector<Piece>(1025, whole), N, W, false, 0);
  if (fails) return 1;
  std::printf("piece check: ok\n");
}
