"""The drop-in boundary's multi-column solve, caller-supplied border blocks
and per-box factor read-back, on the GPU.

* A multi-column b is solved column by column as the reference's sweeps do
  (apply_sweep_matrix takes every column, skel_factorization.cpp:388-406):
  each column equals that column solved alone, bit for bit.
* skeletonize reads the caller's U and Psi (linear_solve.cpp:256-257): the
  solution satisfies the caller's bordered system (dense check).
* A box's T is the interpolative decomposition of its ID matrix: the
  oracle's ID matrix of the same box (the trees are identical) satisfies
  A(:, redundant) = A(:, skeleton) T to the ID tolerance.
"""
import numpy as np
import pytest
import torch

import geometry as G
import iesolver
import oracle

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _solver(g, pde=iesolver.PDE_LAPLACE, holes=True, tol=TOL, precision=iesolver.FP64):
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(64)
    if holes and "holes" in g:
        s.set_holes(g["holes"]["centers"], g["holes"]["radii"])
    s.factor(tol, precision)
    return s


@pytest.mark.parametrize("case", ["star", "star_fp32", "annulus", "stokes_holes"])
def test_multi_column_solve_equals_columns(case):
    if case == "stokes_holes":
        g, pde = G.circle_with_holes(4096, 4, 1), iesolver.PDE_STOKES
    elif case == "annulus":
        g, pde = G.annulus(4000), iesolver.PDE_LAPLACE
    else:
        g, pde = G.star(8192), iesolver.PDE_LAPLACE
    prec = iesolver.FP32 if case.endswith("fp32") else iesolver.FP64
    s = _solver(g, pde, tol=1e-6 if prec == iesolver.FP32 else TOL, precision=prec)
    B = np.random.default_rng(5).standard_normal((s.ndof, 3))
    MU, AL = s.solve_many(B)
    for j in range(3):
        mu, al = s.solve(B[:, j])
        assert np.array_equal(MU[:, j], mu), j
        if AL is not None:
            assert np.array_equal(AL[:, j], al), j


def test_callers_border_blocks_are_used():
    g = G.annulus(2000)
    s = iesolver.RSSolver(0)
    s.set_geometry(g)
    s.build_tree(64)
    s.set_holes(g["holes"]["centers"], g["holes"]["radii"])
    o = oracle.OracleProblem(g)
    U, Psi = o.U_Psi()
    U2 = 2 * U + 0.25  # not the formula's blocks
    s.set_border(U2, Psi)
    s.factor(TOL)
    f = G.harmonic_data(g["points"], *G.exterior_sources(3))
    mu, alpha = s.solve(f)
    K = oracle.dense_matrix(g)
    r1 = K @ mu + U2 @ alpha - f
    r2 = Psi @ mu - alpha
    err = max(np.abs(r1).max(), np.abs(r2).max())
    print(f"caller's border: residual {err:.2e}", flush=True)
    assert err <= 50 * TOL
    with pytest.raises(iesolver.IeGpuError):  # the border's width must match
        s.set_border(U2[:, :1], Psi[:1])


def test_box_factors_t_is_the_interpolative_decomposition():
    g = G.star(8192)
    s = _solver(g)
    o = oracle.OracleProblem(g, record_id_mats=True)
    o.factor(TOL, 4)
    info = s.box_info()
    nl = info["level"].max()
    boxes = [b for b in np.flatnonzero((info["level"] == nl) & (info["rank"] > 0))][:12]
    assert boxes
    for b in boxes:
        fac = s.box_factors(int(b))
        k, r = fac["k"], fac["r"]
        assert k == info["rank"][b] and k + r == info["n_active"][b]
        sk, rd = s.box_list(int(b), 3), s.box_list(int(b), 4)
        A = o.id_mat(int(b))
        pos = {d: i for i, d in enumerate(o.box_list(int(b), 2))}
        As, Ar = A[:, [pos[d] for d in sk]], A[:, [pos[d] for d in rd]]
        err = np.linalg.norm(Ar - As @ fac["T"]) / np.linalg.norm(A)
        assert err <= 20 * TOL, (b, err)
        # X_rr^{-1} U = X_rr^{-1} K_rs and L = K_sr X_rr^{-1}: both factor
        # through the same X_rr^{-1}, so L X_rr^{-1}^{-1} U = K_sr X^{-1} K_rs,
        # the Schur part of the carried block; shapes are the reference's
        assert fac["L"].shape == (k, r) and fac["U"].shape == (r, k)
        assert fac["Xinv"].shape == (r, r) and fac["S"].shape == (k, k)
        assert np.all(np.isfinite(fac["Xinv"]))


@pytest.mark.parametrize("pde", [iesolver.PDE_LAPLACE, iesolver.PDE_STOKES])
def test_border_after_a_non_finite_one(pde):
    """A context whose border products overflowed, then an ordinary border at
    a larger tolerance, where other DOFs reach the root: as a fresh context."""
    g = G.annulus(2000) if pde == iesolver.PDE_LAPLACE else G.circle_with_holes(2000, 4, 1)
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(64)
    s.set_holes(g["holes"]["centers"], g["holes"]["radii"])
    U, Psi = oracle.OracleProblem(g, pde).U_Psi()
    big = 1e307 * np.sign(np.random.default_rng(1).standard_normal(U.shape))
    s.set_border(big, Psi)
    try:
        s.factor(TOL)
        assert not np.all(np.isfinite(s.solve(np.ones(s.ndof))[0]))
    except iesolver.IeGpuError:
        pass  # an elimination that meets only zeros and infinities may stop
    s.set_border(U, Psi)
    f = np.random.default_rng(2).standard_normal(s.ndof)
    for tol in (1e-4, 1e-6, TOL):
        s.factor(tol)
        mu, alpha = s.solve(f)
        t = iesolver.RSSolver(0)
        t.set_geometry(g, pde)
        t.build_tree(64)
        t.set_holes(g["holes"]["centers"], g["holes"]["radii"])
        t.set_border(U, Psi)
        t.factor(tol)
        mf, af = t.solve(f)
        assert np.all(np.isfinite(mf)) and np.all(np.isfinite(af))
        assert np.array_equal(mu, mf) and np.array_equal(alpha, af)


def test_apply_beside_a_solve_on_another_stream():
    """A solve with holes on the caller's stream and the operator on the
    context's, unordered: they share no scratch."""
    g = G.circle_with_holes(30000, 8, 1)
    s = _solver(g, iesolver.PDE_STOKES)
    rng = np.random.default_rng(6)
    b, x, a = (rng.standard_normal(k) for k in (s.ndof, s.ndof, 24))
    mu, alpha = s.solve(b)
    y, z = s.apply(x, a)
    st = torch.cuda.Stream()
    db = torch.from_numpy(b).cuda()
    torch.cuda.synchronize()
    for _ in range(20):
        dm, da = torch.empty_like(db), torch.empty(24, dtype=torch.float64, device="cuda")
        st.wait_stream(torch.cuda.current_stream())
        s.solve_device(db.data_ptr(), dm.data_ptr(), da.data_ptr(), st.cuda_stream)
        y2, z2 = s.apply(x, a)
        st.synchronize()
        assert np.array_equal(y2, y) and np.array_equal(z2, z)
        assert np.array_equal(dm.cpu().numpy(), mu) and np.array_equal(da.cpu().numpy(), alpha)


# Border widths of 5, 33, 64, 66 and 192 (the products' row lanes are 256 / h,
# the Gram matrix takes 1,024 of its h^2 sums per pass, 4,096 rows of a block
# at a time and past h = 48 4,096 per workgroup), DOF counts one and two past
# a multiple of the chunks, bordered systems past the inverse's 512 rows.
@pytest.mark.parametrize("pde,n,h,real", [
    (iesolver.PDE_LAPLACE, 2049, 5, True), (iesolver.PDE_LAPLACE, 3000, 33, True),
    (iesolver.PDE_LAPLACE, 4097, 64, False), (iesolver.PDE_STOKES, 3000, 11, True),
    (iesolver.PDE_STOKES, 1537, 22, False), (iesolver.PDE_STOKES, 2049, 64, False)])
def test_border_widths_against_the_dense_system(pde, n, h, real):
    rng = np.random.default_rng(h)
    if real:
        g = G.circle_with_holes(n, h, 1)
        c, r = g["holes"]["centers"], g["holes"]["radii"]
    else:  # a simple boundary with a border of the caller's
        g = G.star(n)
        c, r = 0.5 + 0.01 * rng.standard_normal((h, 2)), np.full(h, 0.001)
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(64)
    s.set_holes(c, r)
    hd = h * (3 if pde == iesolver.PDE_STOKES else 1)
    if real:
        U, Psi = oracle.OracleProblem(g, pde).U_Psi()
    else:
        U = rng.standard_normal((s.ndof, hd)) / np.sqrt(s.ndof)
        Psi = rng.standard_normal((hd, s.ndof)) / np.sqrt(s.ndof)
        s.set_border(U, Psi)
    s.factor(TOL)
    print("root", s.box_info()["n_active"][0], "border", hd, flush=True)
    f = rng.standard_normal(s.ndof)
    mu, alpha = s.solve(f)
    K = oracle.dense_matrix(g, pde)
    r1, r2 = K @ mu + U @ alpha - f, Psi @ mu - alpha
    # the backward error bar of every form (ie_solver_test.cpp:84-95)
    assert np.sqrt(np.sum(r1 ** 2) + np.sum(r2 ** 2)) <= 50 * TOL * np.linalg.norm(f)
    y, z = s.apply(mu, alpha)  # the operator's own border products
    bound = 1e-12 * (np.abs(K) @ np.abs(mu) + np.abs(U) @ np.abs(alpha)).max()
    assert np.abs(y - (r1 + f)).max() <= bound
    assert np.abs(z - r2).max() <= 1e-12 * (np.abs(Psi) @ np.abs(mu) + np.abs(alpha)).max()
