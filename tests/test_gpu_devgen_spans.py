"""The device generator's parallel chain of wire draws, against the host
generator, bit for bit: at the edges of its spans (1024 draws, 146 to 171
wires), with one span, several, and more than the scan's 1024 lanes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pct", [0, 50, 95, 100])
@pytest.mark.parametrize("P,npp,wpp", [(1, 1, 1), (3, 7, 1), (1, 5, 146), (1, 5, 147), (2, 9, 85),
                                       (2, 9, 86), (7, 33, 147), (5, 40, 1171), (9, 100, 20011)])
def test_spans_match_the_host_generator(C, P, npp, wpp, pct):
    for seed, profile in ((1, C.PROFILE_REFERENCE), (-5, C.PROFILE_STABLE)):
        gp = C.GenParams(P, npp, wpp, pct, seed, profile)
        host = C.generate(gp)
        with C.Context(0) as ctx:
            ctx.generate_device(gp)
            nodes, wires = ctx.store()
            loc = ctx.store_topology()[0]
        assert wires.tobytes() == host.wires.tobytes()
        assert nodes.tobytes() == host.nodes.tobytes()
        assert np.array_equal(loc, host.locator)
