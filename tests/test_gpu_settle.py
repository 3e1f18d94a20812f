"""The early end of a loop (a wave stops stepping once every wire's state
repeats itself) against the same kernel executing every step: the same bits.

Wires of every kind share waves: settling ones, slowly decaying and undamped
ones (which never repeat within the loop, or late), growing ones that overflow
early or near the end, wires at rest and wires whose fixed point has zeros.
"""
import numpy as np
import pytest

from helpers import assert_bit_identical

pytestmark = pytest.mark.gpu


def _mixed(C, seed, profile):
    """A circuit of 4 x 1000 wires, a seventh of them each of one kind."""
    c = C.generate(C.GenParams(4, 250, 1000, 80, seed, profile))
    w, n = c.wires, c.nodes
    rng = np.random.default_rng(seed)
    k = rng.integers(0, 7, len(w))
    dt = np.float32(1e-6)
    w["inductance"][k == 1] = w["resistance"][k == 1] * dt           # undamped mode
    w["inductance"][k == 2] = w["resistance"][k == 2] * dt * np.float32(0.97)   # slow decay
    w["inductance"][k == 3] = w["resistance"][k == 3] * dt * np.float32(1.3)    # slow growth
    w["inductance"][k == 4] = np.float32(0.1)                        # overflows at once
    rest = k == 5
    w["capacitance"][k == 6] = (10.0 ** rng.uniform(-9, 3, (k == 6).sum())).astype(np.float32)
    w["current"] = rng.uniform(-1, 1, (len(w), 10)).astype(np.float32)
    w["voltage"] = rng.uniform(-1, 1, (len(w), 9)).astype(np.float32)
    w["current"][rest], w["voltage"][rest] = 0, 0
    n["voltage"][: len(n) // 2] = np.where(rng.random(len(n) // 2) < 0.5, 0.0, -0.0)
    return c


def _relax(C, circ, policy, steps, all_steps, loops):
    with C.Context(0) as ctx:
        ctx.load(circ)
        ctx.set_option(C.OPT_STEPS, steps)
        ctx.set_option(C.OPT_ALL_STEPS, all_steps)
        ctx.run_loops(loops, policy=policy, mode=C.REDUCE_CSR)
        return ctx.store()


@pytest.mark.parametrize("policy", [0, 1, 2, 3], ids=["exact", "recip", "fast", "scaled"])
@pytest.mark.parametrize("kind", ["stable", "reference", "mixed", "homogeneous"])
def test_early_end_gives_every_steps_bits(C, policy, kind):
    if kind == "mixed":
        circ = _mixed(C, 5, C.PROFILE_STABLE)
    elif kind == "homogeneous":  # whole waves of one kind: undamped, slow, at rest
        circ = C.generate(C.GenParams(3, 64, 192, 100, 3, C.PROFILE_STABLE))
        w, dt = circ.wires, np.float32(1e-6)
        w["inductance"][:64] = w["resistance"][:64] * dt
        w["inductance"][64:256] = w["resistance"][64:256] * dt * np.float32(0.9)
        circ.nodes["voltage"][128:] = 0
    else:
        circ = C.generate(C.GenParams(4, 250, 1000, 80, 9,
                                      C.PROFILE_STABLE if kind == "stable" else C.PROFILE_REFERENCE))
    # around the first checks, the last step of the dense ones, the first wide one, a whole loop
    for steps in (1, 4, 8, 9, 17, 30, 64, 65, 77, 1100, 10000):
        early = _relax(C, circ, policy, steps, 0, 2)
        every = _relax(C, circ, policy, steps, 1, 2)
        for f in ("current", "voltage"):
            assert_bit_identical(early[1][f], every[1][f], f"{kind} {steps} {f}")
        assert_bit_identical(early[0]["voltage"], every[0]["voltage"], f"{kind} {steps} nodes")
