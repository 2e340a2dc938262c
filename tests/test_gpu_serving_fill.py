"""Admission under a fill target: on a device at least half full a request that
would take it past the target waits until there is room, smaller later ones that
fit go first, and what goes first is bounded by an eighth of the waiting request's
work (points times steps).  Below half of the target any request joins."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api
from test_serving import wait_staged

pytestmark = pytest.mark.gpu

SMALL = aerofoil_case(lxibk=(13, 15, 13), letbk=(8, 8), lzebk=(12,))
MID = aerofoil_case(lxibk=(16, 20, 16), letbk=(14, 14), lzebk=(12,))
LARGE = aerofoil_case(lxibk=(24, 30, 24), letbk=(20, 20), lzebk=(12,))


def serve(fill, jobs):
    """Infos of the jobs (case, steps), all set up before the loop starts."""
    srv = api.Server(budget_bytes=0, max_active=len(jobs), graph=True, fill_points=fill)
    reqs = [srv.submit(lay, p, ss, n, 1e-6 * i) for i, ((lay, ss, p), n) in enumerate(jobs)]
    wait_staged(srv, len(jobs))
    srv.run(max_steps=2)
    infos = [srv.result(r, with_state=False)[0] for r in reqs]
    assert all(i["state"] == "done" for i in infos)
    srv.close()
    return infos


def test_large_request_waits_and_small_ones_pass_within_the_bound():
    s, m, l = (c[0].npoints() for c in (SMALL, MID, LARGE))
    fill = m + s + s // 2                       # room for two small beside nothing large
    assert 2 * m >= fill and m + l > fill and m + s <= fill < m + 2 * s
    steps = -(-8 * 2 * 4 * s // l)              # the large one's steps: two small of 4 steps may pass, not three
    assert 8 * 2 * 4 * s <= l * steps < 8 * 3 * 4 * s
    print("fill", fill, "small, mid, large", s, m, l, "steps", steps, flush=True)
    mid, large, *small = serve(fill, [(MID, 40), (LARGE, steps)] + 3 * [(SMALL, 4)])
    assert large["admitted"] >= mid["done"]
    assert small[0]["admitted"] < mid["done"] and small[1]["admitted"] < mid["done"]
    assert small[1]["admitted"] >= small[0]["done"]          # no room for both at once
    assert small[2]["admitted"] >= large["admitted"]


def test_request_joins_a_device_less_than_half_full():
    s, l = SMALL[0].npoints(), LARGE[0].npoints()
    fill = max(l + s // 2, 2 * s + 1)
    assert 2 * s < fill < s + l
    print("fill", fill, "small, large", s, l, flush=True)
    small, large = serve(fill, [(SMALL, 8), (LARGE, 4)])
    assert large["admitted"] < small["done"]
