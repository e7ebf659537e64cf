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
