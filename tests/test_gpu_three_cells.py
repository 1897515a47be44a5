"""Boxes of exactly three cells a side of rc + skin (to a rounding step): a pair
at the list radius, an atom of it on a cell bound, is in reach around the far
side of the box as well.  Along each axis, against the oracle's pair set."""
import numpy as np
import pytest

from conftest import KG_LJ, pos4_of

pytestmark = pytest.mark.gpu

f = np.float32
# (rc + skin, box side): the float cell coordinate of an atom on the upper bound
# of the middle cell comes out one cell low
BOXES = [(3.2307708, 9.692312), (3.4622886, 10.386866), (2.6861198, 8.058359), (2.6032546, 7.8097634), (2.8, 8.4)]


@pytest.mark.parametrize("rcs,L", BOXES)
def test_pairs_on_cell_bounds(fmd, engine, orc, rcs, L):
    rcs, L = f(rcs), f(L)
    rc = f(0.9) * rcs
    skin = rcs - rc
    assert rc + skin == rcs and int(L / rcs) == 3
    marks = []
    for b in (f(0), L / f(3), f(2) * (L / f(3)), f(2) * rcs, rcs, L - rcs, L - f(2) * rcs):
        v = b
        for _ in range(3):
            v = np.nextafter(v, f(-1))
        for _ in range(7):
            if 0 <= v < L:
                marks.append(v)
            v = np.nextafter(v, f(100))
    marks = np.unique(np.array(marks, f))
    for axis in range(3):
        x = np.full((len(marks), 3), 1.0, f)
        x[:, axis] = marks
        sid = engine.add(fmd.Desc(pos4_of(x), L, KG_LJ, rc=float(rc), skin=float(skin), force_cap=10.0))
        p4, _, _ = engine.state(sid)
        ref = orc.pair_set(p4, L, rcs, None)
        got = engine.pairs(sid)
        engine.remove(sid)
        same = np.array_equal(got, ref)
        assert same, (axis, len(got), len(ref))
