"""Launches that hold different line solves: the gradients of a small case along
all three directions, and blocks of different chunk counts, capacities and end
types in one launch of a direction.  Either way a block must get the bits that
launches of its own give it."""
import numpy as np
import pytest

from caseutil import aerofoil_case
from tandemproject_amd import api

pytestmark = pytest.mark.gpu


def context(*cases):
    s = api.Solver([(lay, p) for lay, ss, p in cases])
    for c, (lay, ss, p) in enumerate(cases):
        for b in range(lay.nb):
            s.set_grid(c, b, ss[b])
    s.setup_geometry()
    for c in range(len(cases)):
        s.initialo(c)
    return s


def same(a, ca, b, cb, lay, names=("qa",)):
    for blk in range(lay.nb):
        for name in names:
            np.testing.assert_array_equal(a.download(ca, blk, name), b.download(cb, blk, name), err_msg=f"{blk} {name}")


def gradient_waves(lay, most):
    """Waves of the gradients' one launch: its work items (64 lines) times the
    most chunks of a line, four fields."""
    items = 0
    for b in range(lay.nb):
        n = [int(v) + 1 for v in lay.dims[b]]
        for d in range(3):
            items += -(-(n[0] * n[1] * n[2] // n[d]) // 64)
    return 4 * most * items


# capacities 12, 16, 24, 32 (the longest chunk of the three directions): zeta
# periodic or split in the span, whose closure sums the launch forms
@pytest.mark.parametrize("lx,ly,lz,npcz,chunks", [
    ((12, 16, 13), (12, 13), 12, None, 2), ((23, 28, 25), (12, 13), 12, None, 2), ((14, 44, 46), (12, 8), 12, None, 2),
    ((13, 124, 14), (7, 7), 12, None, 4), ((13, 101, 14), (7, 7), 12, None, 4), ((12, 20, 13), (12, 13), 27, [2], 2),
    ((12, 40, 13), (7, 8), 27, [2], 2)])
def test_gradients_in_one_launch_and_apart(lx, ly, lz, npcz, chunks):
    """The launch is the one for all directions while its waves are at most half
    the 4096 slots and no derivative is timed; timing them runs a launch each."""
    case = aerofoil_case(lxibk=lx, letbk=ly, lzebk=(lz,), npcz=npcz)
    waves = gradient_waves(case[0], chunks)
    print("gradients:", lx, ly, lz, npcz, waves, "waves", flush=True)
    assert waves <= 2048
    one, apart = context(case), context(case)
    assert max(one.col_config()[d, "deriv"] for d in range(3)) <= chunks
    apart.profile_classes(["deriv"])
    for s in (one, apart):
        s.step(2)
        s.stage_part(1, "primitives")
        s.stage_part(1, "viscous")
        s.sync()
    # 3 directions of gradients and 3 of fluxes in each of 8 stages, and the section's gradients
    assert apart.profile_read("deriv")[1] == 8 * 6 + 3
    same(one, 0, apart, 0, case[0], ("tv", "qa"))
    one.close()
    apart.close()


# in each direction: one-sided lines of a few chunks beside longer ones, beside
# lines split across a closure face, beside periodic ones, and long lines of 6, 8
# and 11 waves (521, 701 and 1001 points, and halves of a split 1101-point chord)
MIXES = {
    "chunk counts": [dict(lxibk=(8, 24, 60), letbk=(14, 40)), dict(lxibk=(13, 130, 100), letbk=(70, 8))],
    "split chord": [dict(lxibk=(14, 24, 60), letbk=(14, 20)), dict(lxibk=(13, 20, 81), letbk=(14, 14), npcx=[1, 1, 2])],
    "split span": [dict(lxibk=(14, 24, 20), letbk=(14, 20), lzebk=(12,)),
                   dict(lxibk=(13, 20, 17), letbk=(14, 14), lzebk=(71,), npcz=[2])],
    "long lines": [dict(lxibk=(14, 520, 16), letbk=(8, 8), lzebk=(12,)),
                   dict(lxibk=(13, 700, 1000), letbk=(8, 8), lzebk=(12,)),
                   dict(lxibk=(13, 16, 1100), letbk=(8, 9), lzebk=(12,), npcx=[1, 1, 2])],
}


@pytest.mark.parametrize("name", list(MIXES))
def test_blocks_of_one_launch_equal_each_alone(name):
    cases = [aerofoil_case(**kw) for kw in MIXES[name]]
    print("merged launches:", name, [c[0].npoints() for c in cases], flush=True)
    many = context(*cases)
    many.step(3)
    many.sync()
    for i, case in enumerate(cases):
        alone = context(case)
        alone.step(3)
        alone.sync()
        same(many, i, alone, 0, case[0])
        alone.close()
    many.close()
