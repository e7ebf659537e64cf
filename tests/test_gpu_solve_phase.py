"""The solve phase at the edges of its kernels' tiles: interior evaluation
(128 targets and 512 sources per tile), the dense inverse of root blocks
(panels of 16 columns), and multi-column solves (16 columns at a time)."""
import threading

import numpy as np
import pytest
import torch

import geometry as G
import iesolver
import oracle

pytestmark = pytest.mark.gpu

PDES = [iesolver.PDE_LAPLACE, iesolver.PDE_LAPLACE_NEUMANN, iesolver.PDE_STOKES]


@pytest.mark.parametrize("pde", PDES)
@pytest.mark.parametrize("n,nt", [(63, 1), (511, 127), (513, 129), (8193, 1000)])
def test_evaluate_tile_edges(pde, n, nt):
    g = G.star(n)
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    mu = np.random.default_rng(n + nt).standard_normal(s.ndof)
    tg = G.interior_points(nt, nt, radius=0.2)
    u, uo = s.evaluate(tg, mu), oracle.evaluate(g, tg, mu, pde)
    # both sums round each term by a few ulp: 8 eps per term against the sum
    # of the terms' magnitudes, which the field of |mu| with every sign equal
    # bounds by at most n max|term|; at these distances terms stay below
    # w |mu| / (2 pi 0.04)
    bound = 8 * 2.3e-16 * np.abs(mu).sum() * g["weights"].max() * 25 + 1e-300
    assert np.abs(u - uo).max() <= bound


def test_evaluate_far_and_nan_targets():
    g = G.star(600)
    s = iesolver.RSSolver(0)
    s.set_geometry(g)
    mu = np.ones(600)
    tg = G.interior_points(3, 130, radius=0.2)
    u0 = s.evaluate(tg, mu)
    tg[5] = [1e200, 0.5]   # |r|^2 overflows: the quotient is 0
    tg[129] = [np.nan, 0.5]
    u = s.evaluate(tg, mu)
    assert u[5] == 0.0 and np.isnan(u[129])
    keep = np.ones(130, bool)
    keep[[5, 129]] = False
    # the other targets: the division instead of the refined reciprocal
    assert np.abs(u - u0)[keep].max() <= 600 * 8 * 2.3e-16 * g["weights"].max() * 25


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 192, 193, 500, 512])
def test_root_inverse_panel_edges(n):
    """A tree of one leaf: the root block is the whole operator."""
    g = G.star(n, amp=0.1, k=3)
    s = iesolver.RSSolver(0)
    s.set_geometry(g)
    s.build_tree(512)
    s.factor(1e-10)
    f = np.random.default_rng(n).standard_normal(n)
    mu, _ = s.solve(f)
    K = oracle.dense_matrix(g)
    # Gauss-Jordan with partial pivoting: n eps cond, with growth below 64
    tol = 64 * n * 2.3e-16 * np.linalg.cond(K)
    assert np.linalg.norm(mu - np.linalg.solve(K, f)) <= tol * np.linalg.norm(f)


@pytest.mark.parametrize("problems", [15, 16])
def test_batch_roots_either_inverse(problems):
    """Batches below and from the size that inverts roots one per workgroup:
    each problem as it is solved alone."""
    geoms = [G.star(600 + 37 * p, k=3 + p % 5, amp=0.15) for p in range(problems)]
    f = G.batch_data(geoms)
    s = iesolver.RSSolver(0)
    s.set_geometry_batch(geoms)
    s.build_tree(64)
    s.factor(1e-10)
    mu, _ = s.solve(f)
    for p in range(0, problems, 7):
        sl = slice(s.dof_offsets[p], s.dof_offsets[p + 1])
        a = iesolver.RSSolver(0)
        a.set_geometry(geoms[p])
        a.build_tree(64)
        a.factor(1e-10)
        mp, _ = a.solve(f[sl])
        assert np.linalg.norm(mu[sl] - mp) <= 1e-12 * np.linalg.norm(mp)


@pytest.mark.parametrize("pde,leaf", [(iesolver.PDE_LAPLACE, 64), (iesolver.PDE_STOKES, 300)])
@pytest.mark.parametrize("prec", [iesolver.FP64, iesolver.FP32])
def test_multi_column_tiles_equal_columns(pde, leaf, prec):
    """2, 16, 17 and 33 columns (leaves of up to 300 DOFs: boxes too large for
    16 columns in LDS): every column bit for bit as solved alone."""
    g = G.star(3001)
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(leaf)
    s.factor(1e-6, prec)
    B = np.random.default_rng(2).standard_normal((s.ndof, 33))
    for nrhs in (2, 16, 17, 33):
        MU, _ = s.solve_many(B[:, :nrhs])
        for j in {0, 1, nrhs // 2, nrhs - 1}:
            assert np.array_equal(MU[:, j], s.solve(B[:, j])[0]), (nrhs, j)


@pytest.mark.parametrize("prec", [iesolver.FP64, iesolver.FP32])
def test_two_contexts_invert_roots_at_once(prec):
    """Batches whose roots take 25 workgroups each, more than fit the card,
    factored by two threads: each as it is factored alone, bit for bit."""
    runs = []
    for q in range(2):
        s = iesolver.RSSolver(0)
        s.set_geometry_batch([G.star(390 + p % 11, k=3 + p % 5, amp=0.1 + 0.05 * q)
                              for p in range(64)])
        s.build_tree(512)  # a tree of one leaf: the root block is the operator
        f = np.random.default_rng(q).standard_normal(s.ndof)
        s.factor(1e-10, prec)
        runs.append((s, f, s.solve(f)[0]))
    bad = []

    def work(s, f, want):
        for _ in range(10):
            s.factor(1e-10, prec)
            if not np.array_equal(s.solve(f)[0], want):
                bad.append(1)

    th = [threading.Thread(target=work, args=r) for r in runs]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


@pytest.mark.parametrize("pde", [iesolver.PDE_LAPLACE, iesolver.PDE_STOKES])
def test_evaluate_term_rounds_as_a_division(pde):
    """One source: every target's single term to the roundings of its
    operations, none of which may be a reciprocal short of full accuracy."""
    g = G.star(600)
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    sd = 2 if pde == iesolver.PDE_STOKES else 1
    j = 77
    mu = np.zeros(s.ndof)
    mu[sd * j:sd * j + sd] = (0.7, 0.3)[:sd]
    tg = G.interior_points(5, 20000, radius=0.2)
    u = s.evaluate(tg, mu).reshape(-1, sd)
    L = np.longdouble
    r = tg.astype(L) - g["points"][j].astype(L)
    n, w, m = g["normals"][j].astype(L), L(g["weights"][j]), mu[sd * j:sd * j + sd].astype(L)
    d2, rn = (r * r).sum(1), (r * n).sum(1)
    an = (abs(r) * abs(n)).sum(1)  # what rn's rounding is relative to
    pi = L("3.14159265358979323846")
    # In units of half an eps, to first order: the scaled weight 3, times n 1,
    # r 1, the two products of a dot 2, d2 4, its reciprocal 1, the sum 1; for
    # Stokes the reciprocal (and d2) twice, the dot with mu and the product
    # with r besides.
    if pde == iesolver.PDE_STOKES:
        am = (abs(r) * abs(m)).sum(1)
        want = (w / pi * rn * (r * m).sum(1) / d2 ** 2)[:, None] * r
        size, c = (w / pi * an * am / d2 ** 2)[:, None] * abs(r), 3 + 1 + 1 + 2 + 10 + 1 + 2 + 1 + 4
    else:
        want = (-w / (2 * pi) * rn / d2 * m[0])[:, None]
        size, c = (w / (2 * pi) * an / d2 * abs(m[0]))[:, None], 3 + 1 + 1 + 2 + 4 + 1 + 1
    err = float((abs(u - want) / size).max()) / 2.2e-16
    print(f"largest error {err:.1f} eps, bound {c / 2} eps", flush=True)
    assert err <= c / 2


def test_evaluate_far_sources():
    """A source whose |r|^2 overflows contributes the quotient, 0."""
    g = G.star(600)
    tg = G.interior_points(3, 130, radius=0.2)
    far = {k: np.array(v) for k, v in g.items() if isinstance(v, np.ndarray)}
    far["points"][100] = [1e200, 0.5]
    mu = np.ones(600)
    s, t = iesolver.RSSolver(0), iesolver.RSSolver(0)
    s.set_geometry(g)
    t.set_geometry(far)
    mu0 = mu.copy()
    mu0[100] = 0
    u, u0 = t.evaluate(tg, mu), s.evaluate(tg, mu0)
    assert np.all(np.isfinite(u))
    assert np.abs(u - u0).max() <= 600 * 8 * 2.3e-16 * g["weights"].max() * 25


@pytest.mark.parametrize("nrhs", [1, 256, 257, 512, 530])
def test_many_columns_in_pieces(nrhs):
    """Columns are swept up to 256 at once: every one as solved alone."""
    s = iesolver.RSSolver(0)
    s.set_geometry(G.star(700))
    s.build_tree(64)
    s.factor(1e-10)
    B = np.random.default_rng(4).standard_normal((s.ndof, nrhs))
    MU, _ = s.solve_many(B)
    for j in sorted({0, nrhs // 2, min(255, nrhs - 1), min(256, nrhs - 1), nrhs - 1}):
        assert np.array_equal(MU[:, j], s.solve(B[:, j])[0]), j


def test_multi_column_workspace():
    """One copy of the right-hand sides on the device and a bounded piece of
    them: a solve that fits the card with its columns does so still."""
    s = iesolver.RSSolver(0)
    s.set_geometry(G.star(2048))
    s.build_tree(64)
    s.factor(1e-10)
    B = np.zeros((2048, 16384), order="F")
    B[:, ::1000] = 1.0
    free0 = torch.cuda.mem_get_info()[0]
    s.solve_many(B)
    assert free0 - torch.cuda.mem_get_info()[0] <= 1.25 * B.nbytes
