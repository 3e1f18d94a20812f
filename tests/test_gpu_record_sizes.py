"""Loads and stores either side of the slab sizes at which they change their way:
104 KiB (stored by a pass on the host or on the device) and 1408 KiB (unpacked on
the host or on the device), with few and with many nodes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _footprint(C, N, W):
    n = C.ctypes.c_uint64()
    C._check(C.lib().ckt_footprint_bytes(N, W, 1, C.ctypes.byref(n)))
    return n.value


def _largest(C, fits, hi):
    lo = 1
    while hi - lo > 1:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if fits(mid) else (lo, mid)
    return lo


@pytest.mark.parametrize("limit", [104 << 10, 1408 << 10])
@pytest.mark.parametrize("many_nodes", [False, True])
def test_either_side(C, limit, many_nodes):
    if many_nodes:
        n = _largest(C, lambda x: _footprint(C, x, 40) <= limit, 100000)
        below, above = (n, 40), (n + 1, 40)
    else:
        w = _largest(C, lambda x: _footprint(C, 9, x) <= limit, 20000)
        below, above = (9, w), (9, w + 1)
    assert _footprint(C, *below) <= limit < _footprint(C, *above)
    for N, W in (below, above):
        rng = np.random.default_rng(N + W)
        n, w = np.zeros(N, C.NODE), np.zeros(W, C.WIRE)
        for f in ("charge", "voltage", "capacitance", "leakage"):
            n[f] = rng.standard_normal(N)
        w["in_ptr"], w["out_ptr"] = rng.integers(0, N, W), rng.integers(0, N, W)
        w["in_loc"], w["out_loc"] = rng.integers(0, 3, W), rng.integers(0, 3, W)
        for f in ("inductance", "resistance", "capacitance"):
            w[f] = rng.standard_normal(W)
        w["current"], w["voltage"] = rng.standard_normal((W, 10)), rng.standard_normal((W, 9))
        c = C.HostCircuit(n, w, rng.integers(0, 2, N).astype(np.int32),
                          np.array([(0, W, 0, N)], C.PIECE))
        ends = np.stack([w["in_ptr"], w["out_ptr"]], 1).reshape(-1)
        with C.Context(0) as ctx:
            for _ in range(2):
                ctx.load(c)
                nodes, wires = ctx.store()
                assert nodes.tobytes() == n.tobytes() and wires.tobytes() == w.tobytes()
                assert ctx.store_nodes().tobytes() == n.tobytes()
                loc, row, ent = ctx.store_topology()
                assert np.array_equal(loc, c.locator)
                assert np.array_equal(ent, np.argsort(ends, kind="stable"))
                assert np.array_equal(row, np.concatenate([[0], np.cumsum(np.bincount(ends, minlength=N))]))
