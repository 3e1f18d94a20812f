"""The accessor-form calls with short piece tables (launch arguments) and
long ones (device memory): the same results either side of the limit of 64
pieces, and the same report of invalid records."""
import threading

import numpy as np
import pytest

from helpers import TOL, assert_bit_identical, max_rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 100])
def test_tables_on_both_sides_of_the_limit(C, O, n):
    c = O.generate(100, 7, 30, 80, n, O.PROFILE_STABLE)
    N = len(c.nodes)
    sel = c.pieces[:n]
    dw, pvt = C.DeviceArray(c.wires), C.DeviceArray(c.nodes)
    ofold, gfold = (C.DeviceArray(np.zeros(N, np.float32)) for _ in range(2))
    ref = c.copy()
    C.calc_new_currents_index_gpu(sel, dw, pvt, pvt, pvt)
    for p in sel:
        O.calc_new_currents(ref, p)
    got = dw.download()
    for f in ("current", "voltage"):
        assert_bit_identical(got[f], ref.wires[f], f)
    C.distribute_charge_index_gpu(sel, dw, pvt, ofold, gfold)
    want, wo, wg = ref.nodes.copy(), np.zeros(N, np.float32), np.zeros(N, np.float32)
    O.distribute_charge_fold(ref.wires, want, wo, wg, 0, int(sel["num_wires"].sum()))
    for a, b in ((pvt.download()["charge"], want["charge"]), (ofold.download(), wo),
                 (gfold.download(), wg)):
        assert max_rel_err(a, b, floor=1e-12) <= TOL
    pre = pvt.download()
    C.update_voltages_index_gpu(sel, pvt, pvt, C.DeviceArray(c.locator))
    v = pre["voltage"] + pre["charge"] / pre["capacitance"]
    k = int(sel["num_nodes"].sum())
    post = pvt.download()
    assert_bit_identical(post["voltage"][:k], (v * (np.float32(1) - pre["leakage"]))[:k])
    assert post[k:].tobytes() == pre[k:].tobytes() and not post["charge"][:k].any()


@pytest.mark.parametrize("n", [1, 64, 65])
def test_invalid_records_are_counted(C, O, n):
    c = O.generate(70, 7, 30, 80, 5, O.PROFILE_STABLE)
    k = int(c.pieces["num_wires"][:n].sum())
    c.wires["in_loc"][[0, k - 1]] = 3, -1
    c.wires["out_loc"][[0, k // 2]] = 7, 99
    dw, pvt = C.DeviceArray(c.wires), C.DeviceArray(c.nodes)
    fold = C.DeviceArray(np.zeros(len(c.nodes), np.float32))
    for call in (lambda: C.calc_new_currents_index_gpu(c.pieces[:n], dw, pvt, pvt, pvt),
                 lambda: C.distribute_charge_index_gpu(c.pieces[:n], dw, pvt, fold, fold)):
        for _ in range(2):  # nothing is left over from the call before
            with pytest.raises(C.CircuitError, match="3 wires with an invalid PointerLocation"):
                call()
    dw.upload(O.generate(70, 7, 30, 80, 5, O.PROFILE_STABLE).wires)
    C.calc_new_currents_index_gpu(c.pieces[:n], dw, pvt, pvt, pvt)


def test_concurrent_calls(C, O):
    # Eight threads, half of them with an invalid record: each gets its own report.
    c = O.generate(8, 16, 64, 100, 5, O.PROFILE_STABLE)
    pvt = C.DeviceArray(c.nodes)
    bad = c.wires.copy()
    bad["in_loc"][70] = 5
    seen = [0] * 8

    def work(t):
        dw = C.DeviceArray(bad if t % 2 else c.wires)
        for _ in range(20):
            try:
                C.calc_new_currents_index_gpu(c.pieces, dw, pvt, pvt, pvt, flag=C.POLICY_FAST)
            except C.CircuitError:
                seen[t] += 1

    th = [threading.Thread(target=work, args=(t,)) for t in range(8)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert seen == [0, 20] * 4


@pytest.mark.parametrize("P,npp,wpp,off", [
    (4, 20480, 65537, 0),     # the largest node range whose sums fit in LDS; partial wire blocks
    (4, 20481, 65537, 0),     # one more: atomics
    (70, 5, 3745, 0),         # a table in device memory; far fewer nodes than lanes
    (3, 1000, 87382, 4),      # records that start off a 16-byte boundary
    (64, 4095, 4095, 0),      # just below the size from which LDS is used
    (64, 4097, 4097, 0),      # above it, with as many nodes as wires
])
def test_large_tables_sum_charges(C, P, npp, wpp, off):
    rng = np.random.default_rng(P + npp)
    N, W = P * npp, P * wpp
    w = np.zeros(W, C.WIRE)
    piece = np.arange(W) // wpp
    w["in_ptr"] = piece * npp + rng.integers(0, npp, W)
    w["out_ptr"] = np.where(rng.random(W) < 0.8, piece * npp, rng.integers(0, P, W) * npp) + \
        rng.integers(0, npp, W)
    w["in_loc"], w["out_loc"] = rng.integers(0, 3, W), rng.integers(0, 3, W)
    w["current"] = rng.standard_normal((W, 10))
    pieces = np.zeros(P, C.PIECE)
    k = np.arange(P)
    pieces["first_wire"], pieces["num_wires"] = k * wpp, wpp
    pieces["first_node"], pieces["num_nodes"] = k * npp, npp
    n = np.zeros(N, C.NODE)
    n["charge"] = rng.standard_normal(N) * 1e-6
    raw = np.concatenate([np.zeros(off, np.uint8), w.view(np.uint8).reshape(-1),
                          np.zeros(16 - off, np.uint8)])
    dev = C.DeviceArray(raw)

    class At:
        ptr = type(dev.ptr)(dev.ptr.value + off)

    dn = C.DeviceArray(n)
    folds = [C.DeviceArray(np.zeros(N, np.float32)) for _ in range(2)]
    want = [n["charge"].astype(np.float64), np.zeros(N), np.zeros(N)]
    terms = [np.abs(want[0]), np.zeros(N), np.zeros(N)]
    dt = np.float32(1e-6)
    for ptr, loc, q in (("in_ptr", "in_loc", -dt * w["current"][:, 0]),
                        ("out_ptr", "out_loc", dt * w["current"][:, 9])):
        for kind in range(3):
            m = w[loc] == kind
            np.add.at(want[kind], w[ptr][m], q[m].astype(np.float64))
            np.add.at(terms[kind], w[ptr][m], np.abs(q[m]).astype(np.float64))
    C.distribute_charge_index_gpu(pieces, At, dn, *folds)
    got = [dn.download()["charge"], folds[0].download(), folds[1].download()]
    most = max(np.bincount(w["in_ptr"], minlength=N).max(), np.bincount(w["out_ptr"], minlength=N).max())
    for g, x, t in zip(got, want, terms):
        # each of at most 2 most + 1 additions rounds by 2^-24 of a partial sum
        assert (np.abs(g - x) <= (2 * most + 1) * 2.0 ** -24 * t).all()
    # the relaxation reads the same records (off the boundary word by word)
    if off:
        one = C.DeviceArray(w)
        C.calc_new_currents_index_gpu(pieces, At, dn, dn, dn, flag=C.POLICY_FAST)
        C.calc_new_currents_index_gpu(pieces, one, dn, dn, dn, flag=C.POLICY_FAST)
        back = dev.download()[off:off + W * 128].view(C.WIRE)
        assert back.tobytes() == one.download().tobytes()
    bad = w.copy()
    bad["in_loc"][[0, W - 1]] = 4
    dev.upload(np.concatenate([raw[:off], bad.view(np.uint8).reshape(-1), raw[:16 - off]]))
    with pytest.raises(C.CircuitError, match="2 wires"):
        C.distribute_charge_index_gpu(pieces, At, dn, *folds)
