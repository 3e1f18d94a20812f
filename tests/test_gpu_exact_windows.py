"""EXACT's first steps against the oracle, bit for bit: step counts around its
two-step windows (first one of six steps, two steps each up to 24, then four),
and inductive quotients from subnormal to infinite, on both sides of what the
split division by dt covers.
"""
import numpy as np
import pytest

from helpers import assert_bit_identical

pytestmark = pytest.mark.gpu


def _both(C, O, circ, steps):
    with C.Context(0) as ctx:
        ctx.load(C.HostCircuit(circ.nodes, circ.wires, circ.locator, circ.pieces))
        ctx.set_option(C.OPT_STEPS, steps)
        ctx.calc_new_currents(ctx.pieces(), C.POLICY_EXACT)
        got = ctx.store()[1]
    ref = circ.copy()
    for p in circ.pieces:
        O.calc_new_currents(ref, p, steps=steps)
    return got, ref.wires


@pytest.mark.parametrize("profile", [0, 1], ids=["reference", "stable"])
@pytest.mark.parametrize("steps", [1, 5, 6, 7, 8, 9, 13, 22, 23, 24, 25, 26, 29, 64, 65])
def test_step_counts_around_the_windows(C, O, profile, steps):
    circ = O.generate(3, 100, 333, 80, 11, profile)
    circ.wires["inductance"][::50] = circ.wires["resistance"][::50] * np.float32(1e-6)  # never repeats
    got, want = _both(C, O, circ, steps)
    for f in ("current", "voltage"):
        assert_bit_identical(got[f], want[f], f"{steps} steps {f}")


@pytest.mark.parametrize("steps", [1, 2, 3, 8, 24])
@pytest.mark.parametrize("seed", [1, 2])
def test_inductive_quotients_of_every_size(C, O, steps, seed):
    circ = O.generate(4, 128, 512, 80, seed, O.PROFILE_STABLE)
    w = circ.wires
    rng = np.random.default_rng(seed)
    n = len(w)
    # L from subnormal to near the largest float; R keeps the first currents in range
    e = rng.uniform(-145, 126, n)
    w["inductance"] = (2.0 ** e * rng.choice([-1.0, 1.0], n)).astype(np.float32)
    big = (rng.random(n) < 0.5) & (e > -20)
    w["resistance"][big] = (2.0 ** np.minimum(e[big] + 18, 120)).astype(np.float32)
    w["current"] = rng.uniform(-1, 1, (n, 10)).astype(np.float32)
    w["voltage"] = rng.uniform(-1, 1, (n, 9)).astype(np.float32)
    w["current"][::7] = np.float32(2.0 ** -140)
    got, want = _both(C, O, circ, steps)
    for f in ("current", "voltage"):
        assert_bit_identical(got[f], want[f], f"{steps} steps {f}")
