"""The 128-row sketch of the top levels' large boxes, and the 64-row sketch
walked over a list on levels of many boxes: backward error and ranks at the
edges of their column tiles."""
import os

import numpy as np
import pytest

import geometry as G
import iesolver
import oracle

pytestmark = pytest.mark.gpu

MODEL = os.path.join(os.path.dirname(iesolver.__file__), "rank_model_default.npy")


def _solver(g, pde, leaf, learned, prec=iesolver.FP64, tol=1e-10):
    s = iesolver.RSSolver(0)
    s.set_geometry(g, pde)
    s.build_tree(leaf)
    if learned:
        s.set_rank_model(np.load(MODEL), margin=3)
        s.set_id_method(iesolver.ID_RANDOMIZED, 0)
    s.factor(tol, prec)
    return s


# leaves of up to `leaf` DOFs on levels 1 to 4 make boxes of 65 to 256 columns
@pytest.mark.parametrize("n,leaf,pde", [
    (700, 128, iesolver.PDE_STOKES), (1100, 150, iesolver.PDE_STOKES),
    (1500, 256, iesolver.PDE_STOKES), (3000, 300, iesolver.PDE_LAPLACE_NEUMANN),
    (2049, 64, iesolver.PDE_STOKES), (16385, 64, iesolver.PDE_STOKES)])
def test_large_box_sketches(n, leaf, pde):
    tol = 1e-10
    g = G.star(n, k=5)
    s = _solver(g, pde, leaf, True)
    b = np.random.default_rng(n).standard_normal(s.ndof)
    x, _ = s.solve(b)
    y, _ = s.apply(x)
    # the backward error bar of every form (ie_solver_test.cpp:84-95)
    assert np.linalg.norm(y - b) <= 50 * tol * np.linalg.norm(b)
    info = s.box_info()
    big = (info["n_active"] > 64) & (info["level"] > 0)
    plain = _solver(g, pde, leaf, False).box_info()
    assert big.any()
    # first-level differences compound upward: the sketch's rank of a leaf
    # stays within three of the full pivoted QR's
    leafbig = big & (info["is_leaf"] == 1) & (info["rank"] > 0) & (plain["rank"] > 0)
    assert np.abs(info["rank"] - plain["rank"])[leafbig].max(initial=0) <= 3


def test_large_box_sketch_fp32():
    g = G.star(1100, k=5)
    s = _solver(g, iesolver.PDE_STOKES, 150, True, iesolver.FP32, 1e-5)
    b = np.random.default_rng(3).standard_normal(s.ndof)
    x, _, it, res = s.solve_refined(b, 1e-12, 10)
    assert res <= 1e-12


def test_learned_form_is_as_close_as_the_full_qr():
    """Ranks near a sketch's width: against the exact discrete solution the
    learned form is on average no further off than the pivoted QR."""
    ratio = []
    for k in (3, 4, 5, 6, 7, 8):
        for amp in (0.1, 0.15, 0.2):
            g = G.star(1000, k=k, amp=amp)
            K = oracle.dense_matrix(g, iesolver.PDE_STOKES)
            p = g["points"] - 0.5  # a rotation plus a linear flow: no net flux
            f = np.stack([0.3 - p[:, 1] + 0.7 * p[:, 0], p[:, 0] - 0.7 * p[:, 1]], 1).reshape(-1)
            x = np.linalg.solve(K, f)
            err = [np.linalg.norm(_solver(g, iesolver.PDE_STOKES, 64, form).solve(f)[0] - x)
                   for form in (False, True)]
            ratio.append(err[1] / err[0])
    gm = float(np.exp(np.mean(np.log(ratio))))
    print(f"learned / plain error: mean {gm:.2f}, largest {max(ratio):.2f}", flush=True)
    assert gm <= 1


def _eligible(i, pde):
    proxy = np.where(i["level"] >= 3, 512 if pde == iesolver.PDE_STOKES else 256, 0)
    return ((i["level"] > 0) & (i["m_rows"] > 0) & (i["n_active"] <= 256) &
            ((i["m_rows"] - proxy) // 2 <= 1280))


@pytest.mark.parametrize("n,leaf,pde", [
    (700, 128, iesolver.PDE_STOKES), (1100, 150, iesolver.PDE_STOKES),
    (1500, 256, iesolver.PDE_STOKES), (3000, 300, iesolver.PDE_LAPLACE_NEUMANN)])
def test_large_boxes_are_sketched(n, leaf, pde):
    """Trees whose compressed boxes all lie on levels 1 to 4: every one up to
    256 columns and 1,280 near DOFs ends with a sketch's ID, those of more
    than 128 columns or ranks past 58, which only the 128-row sketch gives,
    among them."""
    s = _solver(G.star(n, k=5), pde, leaf, True)
    i = s.box_info()
    el = _eligible(i, pde)
    assert i["level"][el].max() <= 4
    sketched, fallback = s.id_stats()
    assert fallback == 0 and sketched == el.sum()
    assert (el & ((i["n_active"] > 128) | (i["rank"] > 58))).sum() >= 4
    assert (el & (i["n_active"] > 64) & (i["is_leaf"] == 1)).any()


@pytest.mark.parametrize("n,leaf,pde", [
    (1500, 256, iesolver.PDE_STOKES), (3000, 300, iesolver.PDE_LAPLACE_NEUMANN)])
def test_large_boxes_are_sketched_fp32(n, leaf, pde):
    """At 1e-6 a few narrow sketches fail; fewer than there are boxes of more
    than 128 columns, so the 128-row sketch gave some of those their IDs."""
    s = _solver(G.star(n, k=5), pde, leaf, True, iesolver.FP32, 1e-6)
    i = s.box_info()
    el = _eligible(i, pde)
    sketched, fallback = s.id_stats()
    assert sketched + fallback == el.sum()
    assert fallback < (el & (i["n_active"] > 128)).sum()
