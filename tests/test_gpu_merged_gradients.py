"""The gradients of a small case run along all three directions in one launch;
those of a context with many blocks in a launch per direction.  Both must give
the same bits: the stresses a case leaves (tp_viscous, every point) and whole
steps, alone against among copies that take the context past the limit, at
line lengths on either side of each chunk capacity (12, 16, 24, 32 points)."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api

pytestmark = pytest.mark.gpu


def context(case, copies):
    lay, ss, p = case
    s = api.Solver([(lay, p)] * copies)
    for c in range(copies):
        for b in range(lay.nb):
            s.set_grid(c, b, ss[b])
    s.setup_geometry()
    for c in range(copies):
        s.initialo(c)
    return s


@pytest.mark.parametrize("lx,ly,nz,copies", [
    ((12, 16, 13), (12, 13), 13, 12), ((23, 24, 25), (16, 22), 16, 8), ((31, 33, 32), (14, 14), 24, 8),
    ((14, 47, 44), (46, 13), 13, 8), ((13, 119, 64), (13, 15), 13, 8)])
def test_gradients_together_and_apart(lx, ly, nz, copies):
    print("merged gradients:", lx, ly, nz, flush=True)
    case = aerofoil_case(lxibk=lx, letbk=ly, lzebk=(nz - 1,))
    one, many = context(case, 1), context(case, copies)
    for s in (one, many):
        s.step(2)
        s.stage_part(1, "primitives")
        s.stage_part(1, "viscous")
        s.sync()
    for b in range(case[0].nb):
        for name in ("tv", "qa"):
            np.testing.assert_array_equal(one.download(0, b, name), many.download(copies - 1, b, name), err_msg=name)
    one.close()
    many.close()
