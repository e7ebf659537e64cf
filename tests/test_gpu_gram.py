"""FP32 factorizations' IDs from FP64 Gram matrices, at the edges of the
column tiles and on either side of the tolerance that selects them: backward
error, and ranks against the FP64 factorization's pivoted QR."""
import numpy as np
import pytest

import geometry as G
import iesolver

pytestmark = pytest.mark.gpu

PDES = [iesolver.PDE_LAPLACE, iesolver.PDE_LAPLACE_NEUMANN, iesolver.PDE_STOKES]


def _factored(g, pde, leaf, tol, prec):
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(leaf)
    s.factor(tol, prec)
    return s


# leaves of up to 32, 33, 64, 65, 128 and 300 DOFs
@pytest.mark.parametrize("pde", PDES)
@pytest.mark.parametrize("n,leaf", [(400, 32), (401, 34), (1000, 64), (1003, 66), (1501, 128),
                                    (3000, 300)])
def test_gram_ids(pde, n, leaf):
    tol = 1e-6
    g = G.star(n, k=5)
    s = _factored(g, pde, leaf, tol, iesolver.FP32)
    b = np.random.default_rng(n).standard_normal(s.ndof)
    x, _ = s.solve(b)
    y, _ = s.apply(x)
    # the backward error bar of every form (ie_solver_test.cpp:84-95)
    assert np.linalg.norm(y - b) <= 50 * tol * np.linalg.norm(b)
    i32 = s.box_info()
    # The cut lies near 0.8 tol of the exact diagonal, which the Gram matrix gives to
    # 1e-8 of its norm (1 % of it): on the deepest level, where a leaf's ID
    # matrix is the same in every factorization, the rank lies between the
    # pivoted QR's at tolerances a little either side.
    lo, hi = (_factored(g, pde, leaf, t, iesolver.FP64).box_info() for t in (0.85e-6, 0.75e-6))
    deep = (lo["level"] == lo["level"].max()) & (lo["rank"] > 0)
    assert np.all(i32["rank"][deep] >= lo["rank"][deep])
    assert np.all(i32["rank"][deep] <= hi["rank"][deep])


@pytest.mark.parametrize("tol", [4.9e-7, 5e-7])
def test_gram_tolerance_limit(tol):
    g = G.star(2000)
    s = _factored(g, iesolver.PDE_LAPLACE, 64, tol, iesolver.FP32)
    b = np.random.default_rng(1).standard_normal(s.ndof)
    x, _, it, res = s.solve_refined(b, 1e-12, 10)
    assert res <= 1e-12 and it <= 5


def test_unrefined_error_is_no_larger_than_the_qr_form():
    """72 Stokes stars at 1e-6: the FP32 solve's backward error against the
    FP64 one's at the same tolerance, in the mean.  23.7 is what the FP32
    pivoted QR in the Gram form's place gave on these problems."""
    ratio = []
    for n in (900, 1300, 2000):
        for k in range(3, 9):
            for amp in (0.1, 0.14, 0.18, 0.22):
                s = iesolver.RSSolver(0)
                s.set_geometry(G.star(n, k=k, amp=amp), iesolver.PDE_STOKES)
                s.build_tree(64)
                b = np.random.default_rng(n + k).standard_normal(s.ndof)
                err = []
                for prec in (iesolver.FP32, iesolver.FP64):
                    s.factor(1e-6, prec)
                    err.append(np.linalg.norm(s.apply(s.solve(b)[0])[0] - b))
                ratio.append(err[0] / err[1])
    gm = float(np.exp(np.mean(np.log(ratio))))
    print(f"FP32 / FP64 backward error: mean {gm:.1f}", flush=True)
    assert gm <= 23.7


def test_gram_takes_over_at_its_limit():
    """Below 5e-7 the FP32 QR's ranks, from there on the Gram form's: the two
    tolerances lie 2 % apart, the forms' ranks on the deepest level about 3 %
    of all of them."""
    g = G.star(30000, k=5)
    i = [_factored(g, iesolver.PDE_LAPLACE, 64, t, iesolver.FP32).box_info()
         for t in (4.9e-7, 5e-7)]
    deep = (i[0]["level"] >= i[0]["level"].max() - 1) & (i[0]["is_leaf"] == 1) & (i[0]["rank"] > 0)
    assert deep.sum() > 100
    a, b = (x["rank"][deep].sum() for x in i)
    print(f"leaf ranks below the limit {a}, at it {b}", flush=True)
    # a larger tolerance cannot add ranks within one form
    assert b > a
