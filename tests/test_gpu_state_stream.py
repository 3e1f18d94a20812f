"""calc_new_currents with the early end moves the wires' state past the caches,
except where the last-level cache holds it for three loops or more in a row:
either side of both lines (64 and 256 MiB at 104 bytes a wire), the same bits as
with every step executed."""
import pytest

from helpers import assert_bit_identical

pytestmark = pytest.mark.gpu

LOW, HIGH = (64 << 20) // 104, (256 << 20) // 104


@pytest.mark.parametrize("wires", [LOW, LOW + 1, HIGH, HIGH + 1])
@pytest.mark.parametrize("policy,loops", [(0, 3), (3, 2), (3, 3), (2, 3)],
                         ids=["exact", "scaled-2", "scaled-3", "fast"])
def test_state_accesses(C, wires, policy, loops):
    params = C.GenParams(1, wires // 5, wires, 100, wires, C.PROFILE_STABLE)
    got = []
    for every in (1, 0):
        with C.Context(0) as ctx:
            ctx.generate_device(params)
            ctx.set_option(C.OPT_ALL_STEPS, every)
            ctx.run_loops(loops, policy=policy, mode=C.REDUCE_CSR)
            got.append(ctx.store())
    for f in ("current", "voltage"):
        assert_bit_identical(got[1][1][f], got[0][1][f], f)
    assert_bit_identical(got[1][0]["voltage"], got[0][0]["voltage"], "nodes")
