"""Graph-captured loops around the number a graph holds (16): below it, at it,
with a remainder and replayed, each against the same loops launched directly,
with eager work and synchronisation between the runs."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy,mode", [(0, 1), (3, 1), (0, 2)],
                         ids=["exact-csr", "scaled-csr", "exact-kahan"])
def test_graph_loops_match_launched_loops(C, policy, mode):
    params = C.GenParams(4, 500, 2001, 80, 78, C.PROFILE_STABLE)
    with C.Context(0) as g, C.Context(0) as e:
        for ctx in (g, e):
            ctx.generate(params)
        for loops in (1, 15, 16, 35, 16, 48):
            g.run_loops(loops, policy=policy, mode=mode, use_graph=True)
            e.run_loops(loops, policy=policy, mode=mode)
            gn, gw = g.store()
            en, ew = e.store()
            assert gn.tobytes() == en.tobytes() and gw.tobytes() == ew.tobytes(), loops
            assert g.sanity_check_wires() == 0


def test_batch_replays_while_its_circuits_stay(C):
    # 40 and 20 loops: 20 together, then 20 of the first alone.
    shapes = [C.GenParams(2, 100, 400, 80, 5, C.PROFILE_STABLE),
              C.GenParams(1, 64, 300, 80, 6, C.PROFILE_STABLE)]
    out = []
    for graph in (True, False):
        b = C.Batch(0)
        ids = [b.add_generated(s, n) for s, n in zip(shapes, (40, 20))]
        rep = b.run(b.config(policy=C.POLICY_EXACT, mode=C.REDUCE_CSR, use_graph=graph))
        assert rep["loops_run"] == 40
        out.append([b.store(i, s.num_pieces * s.nodes_per_piece, s.num_pieces * s.wires_per_piece)
                    for i, s in zip(ids, shapes)])
        b.close()
    for (gn, gw), (en, ew) in zip(*out):
        assert gn.tobytes() == en.tobytes() and gw.tobytes() == ew.tobytes()
