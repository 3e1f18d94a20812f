"""Records streamed to and from the device (ckt_ctx_load, ckt_ctx_store,
ckt_ctx_store_topology, ckt_batch_add): contents at the edges of the tiles,
slots and workers, and what a load refuses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _circuit(C, N, W, seed):
    """N nodes in two pieces (one if N is 1), W wires split between them, every
    node shared, so that wires may name any node."""
    rng = np.random.default_rng(seed)
    n, w = np.zeros(N, C.NODE), np.zeros(W, C.WIRE)
    for f in ("charge", "voltage", "capacitance", "leakage"):
        n[f] = rng.standard_normal(N)
    w["in_ptr"], w["out_ptr"] = rng.integers(0, N, W), rng.integers(0, N, W)
    w["in_loc"], w["out_loc"] = rng.integers(1, 3, W), rng.integers(1, 3, W)
    for f in ("inductance", "resistance", "capacitance"):
        w[f] = rng.standard_normal(W)
    w["current"], w["voltage"] = rng.standard_normal((W, 10)), rng.standard_normal((W, 9))
    P = 1 if N == 1 else 2
    p = np.zeros(P, C.PIECE)
    cut_w, cut_n = (W, N) if P == 1 else (W // 3, N // 2)
    p[0] = (0, cut_w, 0, cut_n)
    if P == 2:
        p[1] = (cut_w, W - cut_w, cut_n, N - cut_n)
    return C.HostCircuit(n, w, np.zeros(N, np.int32), p)


# tiles of 256 records, slots of 16384 wires, 131072 nodes and 524288 words;
# the host path below 512 wires, the one-workgroup index up to 4096 wires of
# 32768 nodes
@pytest.mark.parametrize("N,W", [(1, 0), (1, 1), (3, 63), (255, 511), (1, 512), (300, 769),
                                 (32768, 4096), (32769, 4096), (5, 4095), (2000, 4097),
                                 (700, 16384), (64, 16385),
                                 (131073, 49153), (131072, 262145), (300000, 300001)])
def test_round_trip_and_index(C, N, W):
    c = _circuit(C, N, W, N + W)
    with C.Context(0) as ctx:
        for _ in range(2):  # the second load replaces the first circuit
            ctx.load(c)
            nodes, wires = ctx.store()
            assert nodes.tobytes() == c.nodes.tobytes()
            assert wires.tobytes() == c.wires.tobytes()
            assert ctx.store_nodes().tobytes() == c.nodes.tobytes()
            assert ctx.pieces().tobytes() == c.pieces.tobytes()
            loc, row, ent = ctx.store_topology()
            assert not loc.any()
            ends = np.stack([c.wires["in_ptr"], c.wires["out_ptr"]], 1).reshape(-1)
            assert np.array_equal(ent, np.argsort(ends, kind="stable"))
            assert np.array_equal(row, np.concatenate([[0], np.cumsum(np.bincount(ends, minlength=N))]))


def test_batch_add_and_derived_locator(C):
    c = _circuit(C, 500, 3000, 1)
    own = np.repeat(np.arange(2), [1000, 2000])
    c.wires["in_ptr"] = own * 250 + c.wires["in_ptr"] % 250
    c.wires["in_loc"] = np.where(c.wires["in_ptr"] % 2, C.PRIVATE_PTR, C.SHARED_PTR)
    c.wires["out_ptr"] &= ~np.uint32(1)
    want = np.ones(500, np.int32)
    want[c.wires["out_ptr"]] = 0
    want[c.wires["in_ptr"][c.wires["in_loc"] == C.SHARED_PTR]] = 0
    lib = C.lib()
    with C.Context(0) as ctx:
        C._check(lib.ckt_ctx_load(ctx.h, C._p(c.nodes), 500, C._p(c.wires), 3000, None,
                                  C._p(c.pieces), 2))
        assert np.array_equal(ctx.store_topology()[0], want)
    b = C.Batch(0)
    cid = b.add(c, 1)
    nodes, wires = b.store(cid, 500, 3000)
    assert nodes.tobytes() == c.nodes.tobytes() and wires.tobytes() == c.wires.tobytes()
    b.close()


def test_refused_records(C):
    # The first fault in the order of a pass over locations, pointers, then
    # pieces and their wires; the circuit loaded before stays.
    good = _circuit(C, 600, 40000, 2)

    def fault(change):
        c = good.copy()
        change(c)
        with pytest.raises(C.CircuitError) as e:
            ctx.load(c)
        return e.value.status, str(e.value)

    def location(c):
        c.wires["in_ptr"][5] = 600
        c.wires["out_loc"][[39999, 20000]] = -1, 256

    def pointer(c):
        c.wires["out_ptr"][[30001, 30000]] = 600, 2**32 - 1
        c.pieces["num_wires"][0] = 50000

    def private(c):
        c.locator[10] = 1  # owned by piece 0, named by wires of both
        c.wires["out_ptr"][[13333, 13400]] = 10
        keep = (c.wires["out_ptr"] == 10) | (c.wires["in_ptr"] == 10)
        keep[[13333, 13400]] = False
        c.wires["out_ptr"][keep] = c.wires["in_ptr"][keep] = 11

    def piece(c):
        c.pieces["num_nodes"][1] = 301

    with C.Context(0) as ctx:
        ctx.load(good)
        assert fault(location) == (1, "invalid argument: wire 20000 has an invalid PointerLocation (status 1)")
        assert fault(pointer) == (2, "out of range: wire 30000 points past the last node (status 2)")
        assert fault(private) == (1, "invalid argument: wire 13333 of piece 1 reaches a private node "
                                     "of another piece (status 1)")
        assert fault(piece) == (2, "out of range: piece 1 exceeds the circuit (status 2)")
        assert ctx.store()[1].tobytes() == good.wires.tobytes()
