"""Levels of up to 256 boxes run both n <= 64 QRCP shapes in one launch: the
problem alone (levels below the line) against a batch of copies of it (levels
above), and the randomized ID's leftovers against the strided form."""
import numpy as np
import pytest

import geometry as G
import iesolver

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _factor(geoms, method=None, caps=None, leaf=64):
    s = iesolver.RSSolver(0)
    s.set_geometry_batch(geoms)
    s.build_tree(leaf)
    if method is not None:
        s.set_id_method(*method)
    if caps is not None:
        s.set_launch_caps(caps)
    s.factor(TOL, iesolver.FP64)
    return s


# leaves around 32 and 64 DOFs: both shapes on a level, and either alone
@pytest.mark.parametrize("n,leaf", [(300, 32), (1024, 32), (1500, 64), (4100, 64)])
def test_pair_matches_separate_launches(n, leaf):
    g = G.star(n, k=3)
    copies = 40
    f = np.random.default_rng(n).standard_normal(n)
    one, many = _factor([g], leaf=leaf), _factor([g] * copies, leaf=leaf)
    i1, im = one.box_info(), many.box_info()
    lev = np.bincount(im["level"])
    assert lev.max() > 256 >= np.bincount(i1["level"]).max()
    nb = len(i1["rank"])
    assert np.array_equal(im["rank"][:nb], i1["rank"])
    x, _ = one.solve(f)
    y, _ = many.solve(np.tile(f, copies))
    # the same steps on the same boxes; the batch's levels may take the other
    # elimination, whose factors agree to rounding
    assert np.linalg.norm(y[-n:] - x) <= 1e-11 * np.linalg.norm(x)


@pytest.mark.parametrize("n,leaf", [(1024, 32), (3000, 64)])
def test_pair_takes_sketch_leftovers(n, leaf):
    g = G.star(n, k=3)
    # a 16-row sketch fails for most boxes: the fallback list is long
    method = (iesolver.ID_RANDOMIZED, 16)
    f = np.random.default_rng(n).standard_normal(n)
    s, t = _factor([g], method, leaf=leaf), _factor([g], method, [1] * 7 + [4096], leaf=leaf)
    assert np.array_equal(s.box_info()["rank"], t.box_info()["rank"])
    x, _ = s.solve(f)
    y, _ = t.solve(f)
    assert np.linalg.norm(y - x) <= 1e-11 * np.linalg.norm(x)
