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
