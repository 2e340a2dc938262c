"""The filter on lines of 513 to 1024 points at cut-offs from the usual 0.85 pi
to ones whose carries hardly decay along the line (the slow root of the filter's
left-hand side is 0.72 at 0.85 pi, 0.90 at 0.95, 0.96 at 0.98), against the
oracle's sequential filte: alone in each direction, and across a split chord.

The bar is 1e-14 of the field's largest value at every cut-off: both sweeps
solve for the increment, whose rounding against a solve in extended precision
was emulated at 1.1e-16 (0.85 pi) to 1e-15 (0.98 pi) for either.
"""
import numpy as np
import pytest

import pyoracle as po
from caseutil import BASE_PARAMS, aerofoil_case, seeded_field
from tandemproject_amd import api
from tandemproject_amd import layout as L

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("cut", [0.85, 0.92, 0.95, 0.97, 0.98])
@pytest.mark.parametrize("ends", [[10, 30], [45, 45]], ids=["one-sided", "periodic"])
@pytest.mark.parametrize("n,axis", [(513, 0), (701, 0), (701, 1), (701, 2), (1024, 0), (1024, 2)])
def test_long_filter_at_sharp_cutoffs(n, axis, ends, cut):
    print("long filter:", n, axis, ends, cut, flush=True)
    dims, codes = [12, 8, 14], [[10, 25], [20, 10], [10, 30]]
    dims[axis], codes[axis] = n - 1, ends
    lay = L.single_block(*dims, codes)
    p = dict(BASE_PARAMS, fltk=cut, fltkbc=cut)
    o, s = po.Oracle(lay, p), api.Solver([(lay, p)])
    f = np.concatenate([seeded_field(tuple((lay.dims[0] + 1)[::-1]), 71 + c) for c in range(3)])
    o.array(0, "rr")[:] = f
    s.upload(0, 0, "rr", f)
    o.mpigo(1, 1, 0); s.mpigo(1, 1, 0)
    o.filte(axis + 1, 1); s.filte(axis + 1, 1)
    g, r = s.download(0, 0, "rr"), o.array(0, "rr")
    assert rel(g, r) <= 1e-14
    s.close()


@pytest.mark.parametrize("cut", [0.85, 0.95])
def test_long_filter_across_a_split_chord(cut):
    """A chord column of 1101 points in two halves of 551 and 550: closures
    between long lines, other blocks of the launch shorter."""
    print("long filter, split chord:", cut, flush=True)
    lay, ss, p = aerofoil_case(lxibk=(14, 40, 1100), letbk=(14, 14), lzebk=(16,), npcx=[1, 1, 2])
    p = dict(p, fltk=cut, fltkbc=cut)
    o, s = po.Oracle(lay, p), api.Solver([(lay, p)])
    for b in range(lay.nb):
        f = np.concatenate([seeded_field(tuple((lay.dims[b] + 1)[::-1]), 91 + 3 * b + c) for c in range(3)])
        o.array(b, "rr")[:] = f
        s.upload(0, b, "rr", f)
    o.mpigo(1, 1, 0); s.mpigo(1, 1, 0)
    o.filte(1, 1); s.filte(1, 1)
    long = [b for b in range(lay.nb) if lay.dims[b][0] >= 512]
    assert len(long) == 4
    for b in long:
        assert rel(s.download(0, b, "rr"), o.array(b, "rr")) <= 1e-14
    s.close()
