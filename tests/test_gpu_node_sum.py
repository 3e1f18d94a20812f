"""distribute_charge over the node->wire index, alone and in one launch with
update_voltages: at the edges of its 256-node tiles and 2048-entry chunks,
against the sums in the reference's order (circuit.cc:415-460), bit for bit;
and where the joined launch does not apply."""
import numpy as np
import pytest

from helpers import TOL, assert_bit_identical, max_rel_err

pytestmark = pytest.mark.gpu
DT = np.float32(1e-6)


def _circuit(C, N, W, hub, seed):
    """One piece; `hub` of the contributions go to one node."""
    rng = np.random.default_rng(seed)
    n, w = np.zeros(N, C.NODE), np.zeros(W, C.WIRE)
    n["charge"], n["voltage"] = rng.standard_normal(N) * 1e-6, rng.standard_normal(N)
    n["capacitance"], n["leakage"] = rng.uniform(1, 2, N), rng.uniform(0, 0.1, N)
    for f in ("in_ptr", "out_ptr"):
        w[f] = np.where(rng.random(W) < hub, N // 2, rng.integers(0, N, W))
    w["in_loc"] = w["out_loc"] = C.SHARED_PTR
    w["current"] = rng.standard_normal((W, 10))
    w["inductance"], w["resistance"], w["capacitance"] = 1e-7, 5, 0.005
    p = np.zeros(1, C.PIECE)
    p[0] = (0, W, 0, N)
    return C.HostCircuit(n, w, np.zeros(N, np.int32), p)


def _expected(c, currents):
    """(charge after distribute_charge, voltage after update_voltages)."""
    q = c.nodes["charge"].copy()
    for w in range(len(c.wires)):
        q[c.wires["in_ptr"][w]] += -DT * currents[w, 0]
        q[c.wires["out_ptr"][w]] += DT * currents[w, 9]
    v = c.nodes["voltage"] + q / c.nodes["capacitance"]
    return q, v * (np.float32(1) - c.nodes["leakage"])


@pytest.mark.parametrize("N,W,hub", [(1, 1, 0), (1, 3000, 1), (255, 1024, 0), (256, 1024, 0.5),
                                     (257, 1025, 0), (700, 6000, 0.7), (3000, 20, 0),
                                     (513, 2048, 0)])
def test_sums_and_update(C, N, W, hub):
    c = _circuit(C, N, W, hub, N + W)
    with C.Context(0) as ctx:  # the task on its own
        ctx.load(c)
        ctx.distribute_charge(mode=C.REDUCE_CSR)
        q, _ = _expected(c, c.wires["current"])
        assert_bit_identical(ctx.store_nodes()["charge"], q)
    for mode in (C.REDUCE_CSR, C.REDUCE_CSR_KAHAN64):
        with C.Context(0) as ctx:  # the loop, both tasks in one launch
            ctx.load(c)
            ctx.run_loops(1, policy=C.POLICY_EXACT, mode=mode)
            nodes, wires = ctx.store()
            _, v = _expected(c, wires["current"])
            assert not nodes["charge"].any()
            if mode == C.REDUCE_CSR:
                assert_bit_identical(nodes["voltage"], v)
            else:
                assert max_rel_err(nodes["voltage"], v, floor=1e-3) <= TOL


def test_atomic_takes_the_index_in_large_launches(C):
    # 40000 wires: the index form, so the bits are those of the CSR mode; with
    # a node that belongs to no piece the joined launch does not apply, and its
    # voltage must not be updated.
    c = _circuit(C, 9000, 40000, 0.01, 3)
    for nodes_in_piece in (9000, 8999):
        c.pieces["num_nodes"][0] = nodes_in_piece
        out = {}
        for mode in (C.REDUCE_ATOMIC, C.REDUCE_CSR):
            with C.Context(0) as ctx:
                ctx.load(c)
                ctx.run_loops(2, policy=C.POLICY_SCALED, mode=mode)
                out[mode] = ctx.store_nodes()
        if nodes_in_piece == 9000:
            assert out[0].tobytes() == out[1].tobytes()
        else:
            for m in out:
                assert out[m]["voltage"][8999] == c.nodes["voltage"][8999]
                assert out[m]["charge"][8999] != 0
            assert max_rel_err(out[0]["voltage"], out[1]["voltage"]) <= TOL
