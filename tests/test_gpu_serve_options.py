"""Options of a server: EXACT requests with the early end (CKT_OPT_ALL_STEPS 0)
against the server's default, every step executed."""
import pytest

pytestmark = pytest.mark.gpu


def test_exact_requests_with_the_early_end(C, O):
    shapes = [(1, 64, 256, 95, 70, 2), (4, 1024, 16384, 95, 71, 8), (4, 1024, 16384, 50, 72, 8)]
    reqs = [C.Request(C.GenParams(*x[:5], C.PROFILE_STABLE), x[5], 0.0) for x in shapes]
    s = C.Server(0, policy=C.POLICY_EXACT, mode=C.REDUCE_CSR)
    s.set_keep_state(True)
    got, took = {}, {}
    for every in (1, 0):
        s.set_option(C.OPT_ALL_STEPS, every)
        results, report = s.run_trace(reqs)
        assert all(r["status"] == 0 for r in results)
        took[every] = report["elapsed_s"]
        got[every] = [b"".join(a.tobytes() for a in s.fetch(k, x[0] * x[1], x[0] * x[2]))
                      for k, x in enumerate(shapes)]
    assert got[0] == got[1]
    # 10000 steps a loop against about 20
    assert took[0] < took[1], took
    ref = O.generate(*shapes[0][:5], O.PROFILE_STABLE)
    O.run(ref, 2)
    assert got[0][0] == ref.nodes.tobytes() + ref.wires.tobytes()
    # refused: while running, an unknown option
    s.start()
    with pytest.raises(C.CircuitError) as e:
        s.set_option(C.OPT_ALL_STEPS, 1)
    assert e.value.status == 7  # CKT_ERR_STATE
    s.stop()
    with pytest.raises(C.CircuitError):
        s.set_option(99, 1)
    s.close()
