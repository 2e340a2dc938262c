"""Surface statistics that run on as a case moves to a context which has never
sampled (tp_adopt_cases: a case keeps its state and scalars, its sampling interval
and integrals among them), eagerly and through a replayed step that the context had
captured before: the forces and wall arrays must be those of the case left in
place.  The context a sampling case leaves goes on with the others."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api

pytestmark = pytest.mark.gpu

SAMPLED = aerofoil_case(lxibk=(14, 18, 14), letbk=(14, 14), lzebk=(12,))
OTHER = aerofoil_case(lxibk=(16, 20, 16), letbk=(13, 15), lzebk=(12,), amach1=0.3)


def solver(*cases):
    s = api.Solver([(lay, p) for lay, ss, p in cases])
    for c, (lay, ss, p) in enumerate(cases):
        for b in range(lay.nb):
            s.set_grid(c, b, ss[b])
    s.setup_geometry()
    for c in range(len(cases)):
        s.initialo(c)
    return s


def surface(s, case):
    return s.stats_forces(case), [s.stats_wall(case, b) for b in range(SAMPLED[0].nb)]


@pytest.mark.parametrize("graph", [False, True], ids=["eager", "replayed"])
@pytest.mark.parametrize("every", [1, 2])
def test_statistics_go_on_in_an_adopting_context(every, graph):
    print("statistics of an adopted case, every", every, "replayed" if graph else "eager", flush=True)
    stay, src, dst = solver(SAMPLED), solver(SAMPLED, OTHER), solver(OTHER)
    for s in (stay, src):
        s.step(2)
        s.stats_start(0, every)
        s.step(3, graph=graph)
    dst.step(3, graph=graph)
    new, = dst.adopt([(src, 0)])
    for s in (stay, dst, src):
        s.step(4, graph=graph)
        s.sync()
    want, got = surface(stay, 0), surface(dst, new)
    assert got[0] == want[0] and got[0]["samples"] >= 3
    walls = 0
    for a, b in zip(want[1], got[1]):
        assert (a is None) == (b is None)
        if a is not None:
            walls += 1
            for x, y in zip(a, b):
                np.testing.assert_array_equal(x, y)
    assert walls
    for b in range(SAMPLED[0].nb):
        np.testing.assert_array_equal(dst.download(new, b, "qa"), stay.download(0, b, "qa"))
    # what the sampling case left behind equals a case that never met it
    alone = solver(OTHER)
    alone.step(9)
    alone.sync()
    for b in range(OTHER[0].nb):
        np.testing.assert_array_equal(src.download(1, b, "qa"), alone.download(0, b, "qa"))
    for s in (stay, src, dst, alone):
        s.close()
