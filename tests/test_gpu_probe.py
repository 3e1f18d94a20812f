"""What a schedule probe times: every launch of it starts from the batch's own
state, not from what the launch before left.

The wires grow slowly (L = 1.01 R dt) and leave the finite range after some
thousand steps.  With the early end a launch then takes most of a loop's steps
from the batch's state and about ten from its result, whose wires are all NaN.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_probe_starts_from_the_batch_state(C):
    steps = 10000
    circ = C.generate(C.GenParams(16, 1024, 4096, 95, 3, C.PROFILE_STABLE))
    w = circ.wires
    w["inductance"] = w["resistance"] * np.float32(1e-6) * np.float32(1.01)
    w["current"] = np.random.default_rng(0).uniform(-1, 1, w["current"].shape)
    b = C.Batch(0)
    cid = b.add(circ, 1)
    cfg = C.Batch.config(policy=C.POLICY_EXACT, mode=C.REDUCE_CSR, persistent=0)
    b.set_option(C.OPT_ALL_STEPS, 1)
    every = b.probe(cfg, probe_steps=steps)
    b.set_option(C.OPT_ALL_STEPS, 0)
    early = [b.probe(cfg, probe_steps=steps) for _ in range(2)]
    print(f"probe of {steps} steps: {every:.3f} ms with every step, {early} ms with the early end")
    # over a quarter of the steps at the same rate, against a thousandth
    assert min(early) > 0.05 * every
    nodes, wires = b.store(cid, len(circ.nodes), len(w))
    assert wires.tobytes() == w.tobytes() and nodes.tobytes() == circ.nodes.tobytes()
    b.close()
