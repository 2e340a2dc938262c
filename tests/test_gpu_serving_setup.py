"""A request that arrives while a large case steps is set up beside it and joins
it: its set-up must not wait for the steps in flight at every small allocation it
gives back (hipFree waits for the whole device).  The running case has 25
iterations of 10 steps left when the request is submitted; the set-up is some 20 ms
of host work and four waits for its own kernels, a few iterations.  The result
equals the request's case run alone."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api
from tandemproject_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_request_is_set_up_beside_a_running_case():
    big, bss, bp, _ = W.naca0012_20m(scale=0.45)
    lay, ss, p = aerofoil_case(lxibk=(24, 30, 20), letbk=(16, 16), amach1=0.45, inflow=1, nmodes=32, seed=7,
                               ntz=16, slit=2.0, tu=0.04, lturb=0.3, gustw=1.5)
    print("set-up beside", big.npoints(), "points", flush=True)
    srv = api.Server(budget_bytes=0, max_active=4, graph=True)
    rb = srv.submit(big, bp, bss, 260)
    while srv.result(rb, with_state=False)[0]["steps"] < 10:
        srv.iterate(10)
    r = srv.submit(lay, p, ss, 6)
    srv.run(10)
    ib, i = srv.result(rb, with_state=False)[0], srv.result(r, with_state=False)[0]
    print(f"  arrival {i['arrival']:.3f} admitted {i['admitted']:.3f}, the running case done {ib['done']:.3f}", flush=True)
    assert ib["state"] == i["state"] == "done"
    assert i["admitted"] < ib["done"] and srv.stats()["joined_running"] == 1
    qa = srv.result(r)[1]
    srv.close()
    s = api.Solver([(lay, p)])
    for b in range(lay.nb):
        s.set_grid(0, b, ss[b])
    s.setup_geometry()
    s.initialo(0)
    s.step(6)
    s.sync()
    for b in range(lay.nb):
        np.testing.assert_array_equal(qa[b], s.download(0, b, "qa"))
    s.close()
