"""First factorizations whose scratch pools overflow: the decouple of a level
runs beside the scan that reports the overflow for a level above, and the
factorization is repeated with larger pools."""
import numpy as np
import pytest

import geometry as G
import iesolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pde,n,leaf,prec", [
    (iesolver.PDE_STOKES, 12000, 150, iesolver.FP64), (iesolver.PDE_STOKES, 12000, 150, iesolver.FP32),
    (iesolver.PDE_LAPLACE, 40001, 150, iesolver.FP64)])
def test_overflow_beside_the_decouple(pde, n, leaf, prec):
    g = G.star(n, k=5)
    for _ in range(4):  # fresh contexts: each overflows and starts again
        s = iesolver.RSSolver(0)
        s.set_geometry(g, pde)
        s.build_tree(leaf)
        b = np.random.default_rng(n).standard_normal(s.ndof)
        s.factor(1e-6, prec)
        x, _ = s.solve(b)
        # the decouple operands (2 n^2 for a box above 64 DOFs) of the deepest
        # level fit the pool a context starts with, those of the next do not
        info = s.box_info()
        need = np.bincount(info["level"], np.where(info["n_active"] > 64,
                                                   2.0 * info["n_active"] ** 2, 0.0))
        assert need[-1] <= max(8 * s.ndof, 1 << 20) < need[-2]
        s.factor(1e-6, prec)  # the pools fit now
        y, _ = s.solve(b)
        assert np.array_equal(x, y)


def test_failed_sketches_take_slots_past_the_scan():
    """Boxes of at most 128 columns and ranks past 58 on the top levels fail
    their 64-row sketch and take their 128-row slot then: more than the pool
    of a context holds, so its first factorization starts again."""
    g = G.star(700, k=5)
    f = np.random.default_rng(1).standard_normal(1400)

    def factored(copies):
        s = iesolver.RSSolver(0)
        s.set_geometry_batch([g] * copies, iesolver.PDE_STOKES)
        s.build_tree(56)
        s.set_id_method(iesolver.ID_RANDOMIZED, 32)
        s.factor(1e-10)
        return s

    one, many = factored(1), factored(40)
    i = many.box_info()
    n = i["n_active"].astype(np.int64)
    failed = (i["level"] > 0) & (i["level"] <= 4) & (n > 64) & (n <= 128) & (i["rank"] > 58)
    print("failed 64-row sketches per level", np.bincount(i["level"][failed]), flush=True)
    need = np.bincount(i["level"][failed], (5 * 128 * ((n + 15) // 16 * 16))[failed])
    assert need.max() > max(16 * many.ndof, 1 << 22)
    x, _ = many.solve(np.tile(f, 40))
    many.factor(1e-10)
    y, _ = many.solve(np.tile(f, 40))
    assert np.array_equal(x, y)
    z, _ = one.solve(f)
    for p in (0, 17, 39):  # the batch's levels may take another elimination
        assert np.linalg.norm(x[1400 * p:1400 * (p + 1)] - z) <= 1e-9 * np.linalg.norm(z)
