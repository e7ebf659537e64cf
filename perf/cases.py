"""The work that the framework's users have it do, as cases that can be timed.

A case is a dict of plain values.  `listed()` names the fixed ones, `draw(rng)`
gives more of the same ranges, `prepare(case, seed)` makes what a user's program
holds before the call (geometry, quadtree, right-hand sides, rank model),
`run(state)` is one pass through the public binding (ie-solver_amd/iesolver.py),
`work(case)` the bytes and operations a pass cannot do without, and
`exact(case, seed)` the same outputs in plain torch and numpy, 64 bits.

Operations ("op"):

  step     factor + solve of one right-hand side on device vectors
           (factor_solve_device), the framework's headline call
  host     factor, then solve, on host vectors: skeletonize + linear_solve as
           the reference's bie_time_trial calls them
           (ie_solver/linear_solve.cpp:156-185)
  refined  FP32 factorization at tolerance 1e-6 + FP64 iterative refinement
  batch    `problems` independent boundaries factored and solved together
  solves   solves of `nrhs` right-hand sides with a stored factorization
  field    holes: FP32 factorization + refinement, then the interior field; returns
           the density, the hole strengths and the field
           (boundary_integral_solve, ie_solver/linear_solve.cpp:188-266)
  evaluate the interior field of a given density
  update   a local deformation of the boundary and back: update_geometry,
           re-factorization of the marked boxes, solve, twice

Forms of the interpolative decomposition ("form"): plain (pivoted QR, the
reference's algorithm) and learned (Gaussian sketches sized by the committed
rank model, the benchmark's default).
"""
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "ie-solver_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import geometry as G  # noqa: E402
import iesolver  # noqa: E402

LEAF = 64          # the reference's leaf capacity (quadtree.h:10)
TOL = 1e-10        # ID tolerance of the FP64 forms
TOL32 = 1e-6       # ID tolerance of the FP32 preconditioner
RTOL = 1e-12       # relative residual the refinement goes to

_PDES = {"laplace": iesolver.PDE_LAPLACE, "neumann": iesolver.PDE_LAPLACE_NEUMANN,
         "stokes": iesolver.PDE_STOKES}


def listed():
    return [
        # The smallest calls: a boundary of the size the reference's own
        # end-to-end tests use, host vectors in and out.  Launches and
        # latency are all of it.
        dict(name="circle1k_host_plain", op="host", pde="laplace", shape="circle", n=1000,
             form="plain"),
        # The reference's CPU-runnable benchmark: a circle of 4,096 nodes.
        dict(name="circle4k_step_plain", op="step", pde="laplace", shape="circle", n=4096,
             form="plain"),
        # An ordinary problem, the pivoted-QR form on the star boundary.
        dict(name="star65k_step_plain", op="step", pde="laplace", shape="star", n=65536,
             form="plain"),
        # The headline: N = 262,144 on the wavy boundary, learned sketches.
        dict(name="wavy262k_step_learned", op="step", pde="laplace", shape="wavy", n=262144,
             form="learned"),
        # The adjoint kernel (Laplace Neumann), host vectors, an odd size.
        dict(name="star20k_host_neumann", op="host", pde="neumann", shape="star", n=20001,
             form="learned"),
        # Stokes flow, two unknowns per node, an odd size.
        dict(name="star16k_step_stokes", op="step", pde="stokes", shape="star", n=16385,
             form="learned"),
        # The mixed-precision form: FP32 factorization, FP64 refinement.
        dict(name="wavy262k_refined", op="refined", pde="laplace", shape="wavy", n=262144,
             form="learned"),
        # The serving form of many problems: 256 star boundaries of 2,048 to
        # 32,768 nodes, one call.
        dict(name="batch256_learned", op="batch", pde="laplace", shape="star", n=32768,
             nmin=2048, problems=256, form="learned"),
        # Stored factorization, new data: 16 right-hand sides at once.
        dict(name="wavy262k_solves16", op="solves", pde="laplace", shape="wavy", n=262144,
             nrhs=16, form="learned"),
        # Stokes flow around 8 holes with its interior field, 262,144 + 24
        # unknowns.
        dict(name="holes131k_field_stokes", op="field", pde="stokes", shape="holes", n=131072,
             targets=10000, form="plain"),
        # The field on a 100 x 100 grid of interior points.
        dict(name="star65k_evaluate", op="evaluate", pde="laplace", shape="star", n=65536,
             targets=10000),
        # A moving boundary: two frames of a local deformation.
        dict(name="wavy65k_update", op="update", pde="laplace", shape="wavy", n=65536,
             form="learned"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["step", "step", "step", "host", "refined", "batch", "solves", "field",
                     "evaluate", "update"])
    c = dict(op=op, pde="laplace", shape=rng.choice(["star", "wavy"]),
             form=rng.choice(["plain", "learned"]))
    if op == "step":
        c["pde"] = rng.choice(["laplace", "laplace", "neumann", "stokes"])
        c["n"] = _log_int(rng, 1000, 65536 if c["pde"] == "stokes" else 262144)
    elif op == "host":
        c["pde"] = rng.choice(["laplace", "neumann", "stokes"])
        c["n"] = _log_int(rng, 1000, 65536)
    elif op == "refined":
        c["n"] = _log_int(rng, 4096, 262144)
    elif op == "batch":
        c.update(shape="star", problems=_log_int(rng, 4, 128), nmin=2048,
                 n=_log_int(rng, 4096, 32768))
    elif op == "solves":
        c.update(n=_log_int(rng, 1000, 262144), nrhs=rng.randint(1, 16))
    elif op == "field":
        c.update(shape="holes", pde="stokes", form="plain", n=_log_int(rng, 4096, 65536),
                 targets=_log_int(rng, 100, 10000))
    elif op == "evaluate":
        c.update(n=_log_int(rng, 1000, 65536), targets=_log_int(rng, 100, 10000),
                 pde=rng.choice(["laplace", "stokes"]))
        del c["form"]
    else:
        c.update(shape="wavy", n=_log_int(rng, 16384, 131072))
    return c


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _curve(case, seed, n=None):
    """The boundary of a case: the family's shape with parameters from seed."""
    n = case["n"] if n is None else n
    rng = np.random.default_rng([seed, 11])
    if case["shape"] == "circle":
        return G.circle(n)
    if case["shape"] == "star":
        return G.star(n, amp=float(rng.uniform(0.15, 0.25)), k=int(rng.integers(5, 10)))
    if case["shape"] == "holes":
        return G.circle_with_holes(n, 8, seed)
    return G.wavy(n, seed=seed)


def _data(case, seed, g, k=0):
    """Boundary data k of a case on the nodes of g."""
    if case["pde"] == "stokes":
        rng = np.random.default_rng([seed, 13, k])
        a = rng.normal(size=6)
        # a rigid rotation plus a linear incompressible flow: no net flux
        p, f = g["points"] - 0.5, np.zeros(2 * g["points"].shape[0])
        f[0::2] = a[0] - a[2] * p[:, 1] + a[3] * p[:, 0] + a[4] * p[:, 1]
        f[1::2] = a[1] + a[2] * p[:, 0] - a[3] * p[:, 1] + a[4] * p[:, 0]
        if "holes" in g:  # no slip on the holes
            f[2 * int(g["counts"][0]):] = 0
        return f
    return G.harmonic_data(g["points"], *G.exterior_sources(1000 * seed + k))


def _targets(case, seed, g):
    """Interior points: a disc every boundary of the family encloses, clear of
    the holes."""
    m = case["targets"]
    if case["shape"] != "holes":
        return G.interior_points(seed, m, radius=0.1)
    c, r = g["holes"]["centers"], g["holes"]["radii"]
    out, k = np.zeros((0, 2)), 0
    while out.shape[0] < m:
        p = G.interior_points(seed + 7919 * k, m, radius=0.45)
        d = np.hypot(p[:, None, 0] - c[None, :, 0], p[:, None, 1] - c[None, :, 1])
        out = np.concatenate([out, p[(d > r[None, :] + 0.01).all(1)]])
        k += 1
    return out[:m]


def _batch_shapes(case, seed):
    """(nodes, lobes, amplitude) per problem: sizes log-uniform as
    geometry.star_batch draws them, the same for every seed; shapes from seed."""
    _, meta = G.star_batch(case["problems"], seed=0, nmin=case["nmin"], nmax=case["n"])
    rng = np.random.default_rng([seed, 23])
    return [(int(n), int(rng.integers(3, 10)), float(rng.uniform(0.05, 0.25)))
            for n in meta["sizes"]]


def _batch_geometries(case, seed):
    return [G.star(n, amp=a, k=k) for n, k, a in _batch_shapes(case, seed)]


def _update_frames(case, seed):
    """The undeformed boundary and one with a bump of 3e-4 r0 over 0.2 rad."""
    t0 = float(np.random.default_rng([seed, 17]).uniform(0, 2 * math.pi))
    return (G.wavy(case["n"], seed=seed),
            G.bump_wavy(case["n"], 3e-4, t0, seed=seed))


def _density(case, seed, g):
    """A smooth density on g (evaluate takes what an earlier solve gave)."""
    rng = np.random.default_rng([seed, 19])
    sd = 2 if case["pde"] == "stokes" else 1
    th = np.arctan2(g["points"][:, 1] - 0.5, g["points"][:, 0] - 0.5)
    mu = np.zeros((th.size, sd))
    for k in range(6):
        mu += np.cos(k * th)[:, None] * rng.normal(size=sd) / (1 + k)
        mu += np.sin(k * th)[:, None] * rng.normal(size=sd) / (1 + k)
    return mu.reshape(-1)


def _set_form(s, case):
    if case.get("form") == "learned":
        s.set_rank_model(np.load(os.path.join(_PKG, "rank_model_default.npy")), margin=3)
        s.set_id_method(iesolver.ID_RANDOMIZED, 0)
    else:
        s.set_id_method(iesolver.ID_QRCP)


def _solver(case, g):
    s = iesolver.RSSolver(0)
    if isinstance(g, list):
        s.set_geometry_batch(g, _PDES[case["pde"]])
    else:
        s.set_geometry(g, _PDES[case["pde"]])
    s.build_tree(LEAF)
    if not isinstance(g, list) and "holes" in g:
        s.set_holes(g["holes"]["centers"], g["holes"]["radii"])
    _set_form(s, case)
    return s


def prepare(case, seed):
    op = case["op"]
    st = dict(op=op)
    if op == "batch":
        geoms = _batch_geometries(case, seed)
        st["s"] = _solver(case, geoms)
        st["b"] = torch.from_numpy(G.batch_data(geoms, seed)).cuda()
        st["x"] = torch.empty_like(st["b"])
    elif op == "update":
        st["frames"] = _update_frames(case, seed)
        st["s"] = _solver(case, st["frames"][0])
        st["f"] = [_data(case, seed, g) for g in st["frames"]]
        st["s"].factor(TOL, iesolver.FP64)
    else:
        g = _curve(case, seed)
        st["s"] = _solver(case, g)
        if op == "step":
            st["b"] = torch.from_numpy(_data(case, seed, g)).cuda()
            st["x"] = torch.empty_like(st["b"])
        elif op == "solves":
            st["B"] = np.asfortranarray(np.stack(
                [_data(case, seed, g, k) for k in range(case["nrhs"])], axis=1))
            st["s"].factor(TOL, iesolver.FP64)
        elif op == "evaluate":
            st["mu"] = _density(case, seed, g)
        else:
            st["f"] = _data(case, seed, g)
        if op in ("field", "evaluate"):
            st["targets"] = _targets(case, seed, g)
    torch.cuda.synchronize()
    return st


def run(st):
    s, op = st["s"], st["op"]
    if op in ("step", "batch"):
        s.factor_solve_device(TOL, iesolver.FP64, st["b"].data_ptr(), st["x"].data_ptr())
        return st["x"]
    if op == "host":
        s.factor(TOL, iesolver.FP64)
        return s.solve(st["f"])[0]
    if op == "refined":
        s.factor(TOL32, iesolver.FP32)
        return s.solve_refined(st["f"], RTOL, 10)[0]
    if op == "solves":
        return s.solve_many(st["B"])[0]
    if op == "field":
        s.factor(TOL32, iesolver.FP32)
        mu, alpha, _, _ = s.solve_refined(st["f"], RTOL, 10)
        return [mu, alpha, s.evaluate(st["targets"], mu, alpha)]
    if op == "evaluate":
        return s.evaluate(st["targets"], st["mu"])
    out = []
    for k in (1, 0):  # the deformed boundary, then back
        s.update_geometry(st["frames"][k])
        s.factor(TOL, iesolver.FP64)
        out.append(s.solve(st["f"][k])[0])
    return out


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
# Per unknown of a factorization at these tolerances with 64-DOF leaves,
# counted from the boxes of the wavy boundary of 262,144 nodes (22,941 boxes):
# the products of a sketched interpolative decomposition of each box's ID
# matrix (2 l m n, 13.6 GFLOP in all) and of its Schur complement (6 s^2 r +
# 8 r^2 s + 2/3 r^3, 1.33 GFLOP), and the stored factors T, L, U, X_rr^{-1}
# (3 s r + r^2 elements, 3.3 kB in 64 bits) that every solve reads.
_FLOPS_FACTOR = {"laplace": 5.7e4, "neumann": 5.7e4, "stokes": 1.1e5}
_FACTOR_ELEMS = 100.0
_PAIR = {"laplace": 12.0, "stokes": 20.0, "neumann": 12.0}


def _unknowns(case):
    n = case["n"]
    if case["op"] == "batch":  # mean of a log-uniform size
        lo, hi = case["nmin"], case["n"]
        n = (hi - lo) / math.log(hi / lo) * case["problems"]
    return n * (2 if case["pde"] == "stokes" else 1)


def work(case):
    op, u = case["op"], _unknowns(case)
    geo = 48.0 * u / (2 if case["pde"] == "stokes" else 1)
    io = 16.0 * u
    factor = _FLOPS_FACTOR[case["pde"]] * u
    solve = 2 * 2 * _FACTOR_ELEMS * u
    if op in ("step", "host", "batch"):
        return {"bytes": geo + io, "flops": factor + solve}
    if op == "refined":
        return {"bytes": geo + io, "flops": factor + 3 * solve}
    if op == "solves":
        return {"bytes": 8 * _FACTOR_ELEMS * u + io * case["nrhs"], "flops": solve * case["nrhs"]}
    if op == "update":  # two frames of about a tenth of the boxes, two solves
        return {"bytes": 2 * (geo + io), "flops": 2 * (0.1 * factor + solve)}
    sd = 2 if case["pde"] == "stokes" else 1
    pairs = float(case["targets"]) * case["n"] * _PAIR[case["pde"]]
    out = 8.0 * (2 + sd) * case["targets"]
    if op == "evaluate":
        return {"bytes": geo + 8 * u + out, "flops": pairs}
    return {"bytes": geo + io + out, "flops": factor + 3 * solve + pairs}


# --------------------------------------------------------------------------
# The same outputs in plain torch and numpy
# --------------------------------------------------------------------------
_COARSE = 3072  # nodes that resolve every smooth boundary above to rounding


def _dense(case, g):
    """The boundary operator's matrix on the nodes of g (GPU, 64 bits)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p, nv, k, w = (torch.from_numpy(np.ascontiguousarray(g[q])).to(dev)
                   for q in ("points", "normals", "curvatures", "weights"))
    N = w.numel()
    r = [p[:, None, a] - p[None, :, a] for a in (0, 1)]
    d2 = r[0] * r[0] + r[1] * r[1]
    d2.fill_diagonal_(1.0)
    eye = torch.arange(N, device=dev)
    if case["pde"] == "neumann":
        K = w[None] + w[None] / (2 * math.pi) * (r[0] * nv[:, None, 0] + r[1] * nv[:, None, 1]) / d2
        K[eye, eye] = w - 0.5 + 0.5 * k * w / (2 * math.pi)
        return K
    rn = r[0] * nv[None, :, 0] + r[1] * nv[None, :, 1]
    if case["pde"] == "laplace":
        K = -w[None] / (2 * math.pi) * rn / d2
        K[eye, eye] = 0.5 + 0.5 * k * w / (2 * math.pi)
        return K
    c = w[None] / math.pi * rn / (d2 * d2)
    K = torch.empty((N, 2, N, 2), dtype=torch.float64, device=dev)
    pot = -0.5 * k * w / math.pi
    t = (-nv[:, 1], nv[:, 0])
    for a in (0, 1):
        for b in (0, 1):
            M = c * r[a] * r[b]
            M[eye, eye] = pot * t[a] * t[b] - (0.5 if a == b else 0.0)
            K[:, a, :, b] = M + w[None] * nv[:, None, a] * nv[None, :, b]
    return K.reshape(2 * N, 2 * N)


def _fourier(v, n):
    """Values at n equispaced parameters of the trigonometric interpolant of
    the rows of v."""
    m = v.shape[0]
    if m == n:
        return v
    c = np.fft.rfft(v, axis=0)
    out = np.zeros((n // 2 + 1,) + v.shape[1:], dtype=complex)
    q = min((m - 1) // 2 + 1, out.shape[0])
    out[:q] = c[:q]
    return np.fft.irfft(out, n, axis=0) * (n / m)


def _solution(case, make, data, n):
    """Solutions (columns) on n nodes of a smooth boundary.  The trapezoid
    rule converges faster than any power of 1/n there, so the discrete
    solution on many nodes is the interpolant of the one on _COARSE."""
    m = min(n, _COARSE)
    g = make(m)
    B = np.stack(data(g), axis=1)
    K = _dense(case, g)
    X = torch.linalg.solve(K, torch.from_numpy(B).to(K.device)).cpu().numpy()
    sd = 2 if case["pde"] == "stokes" else 1
    X = X.reshape(m, sd * B.shape[1]) if sd == 1 else X.reshape(m, 2, B.shape[1])
    X = _fourier(X, n)
    return X.reshape(n * sd, B.shape[1])


def _borders(g, N):
    """U (2N x 3h) and Psi (3h x 2N) of Stokes holes."""
    p, w, c, rad = g["points"], g["weights"], g["holes"]["centers"], g["holes"]["radii"]
    h = rad.size
    U, P, s = np.zeros((2 * N, 3 * h)), np.zeros((3 * h, 2 * N)), 1 / (4 * math.pi)
    free = np.ones(N, bool)
    for k in range(h):
        r = p - c[k]
        rn = np.hypot(r[:, 0], r[:, 1])
        U[:, 3 * k:3 * k + 3] = _hole_flow(r, s)
        on = free & (rn < rad[k] + 1e-8)
        free &= ~on
        i = np.nonzero(on)[0]
        P[3 * k, 2 * i] = w[i]
        P[3 * k + 1, 2 * i + 1] = w[i]
        P[3 * k + 2, 2 * i] = w[i] * p[i, 1]
        P[3 * k + 2, 2 * i + 1] = -w[i] * p[i, 0]
    return U, P


def _hole_flow(r, s):
    """Stokeslet (two columns) and rotlet of a hole at offsets r."""
    rn2 = r[:, 0] ** 2 + r[:, 1] ** 2
    lg = -0.5 * np.log(rn2)
    out = np.zeros((2 * r.shape[0], 3))
    out[0::2, 0] = s * (lg + r[:, 0] ** 2 / rn2)
    out[1::2, 0] = out[0::2, 1] = s * r[:, 0] * r[:, 1] / rn2
    out[1::2, 1] = s * (lg + r[:, 1] ** 2 / rn2)
    out[0::2, 2] = s * r[:, 1] / rn2
    out[1::2, 2] = -s * r[:, 0] / rn2
    return out


def _field(case, g, targets, mu):
    """The double layer potential of mu at interior targets."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p, nv, w, m = (torch.from_numpy(np.ascontiguousarray(q)).to(dev)
                   for q in (g["points"], g["normals"], g["weights"], mu))
    sd = 2 if case["pde"] == "stokes" else 1
    m = m.reshape(-1, sd)
    out = []
    for part in np.array_split(targets, max(1, targets.shape[0] * w.numel() // 50_000_000)):
        t = torch.from_numpy(np.ascontiguousarray(part)).to(dev)
        r0, r1 = (t[:, None, a] - p[None, :, a] for a in (0, 1))
        d2 = r0 * r0 + r1 * r1
        rn = w[None] * (r0 * nv[None, :, 0] + r1 * nv[None, :, 1])
        if sd == 1:
            out.append((-(rn / d2) @ m / (2 * math.pi)).reshape(-1))
        else:
            c = rn / (d2 * d2) * (r0 * m[None, :, 0] + r1 * m[None, :, 1]) / math.pi
            out.append(torch.stack([(c * r0).sum(1), (c * r1).sum(1)], 1).reshape(-1))
    return torch.cat(out).cpu().numpy()


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        out = []
        for i, (n, k, a) in enumerate(_batch_shapes(case, seed)):
            src = G.exterior_sources(seed + 1000 * i)
            out.append(_solution(case, lambda m: G.star(m, amp=a, k=k),
                                 lambda q: [G.harmonic_data(q["points"], *src)], n)[:, 0])
        return np.concatenate(out)
    if op == "evaluate":
        g = _curve(case, seed)
        return _field(case, g, _targets(case, seed, g), _density(case, seed, g))
    if op == "update":  # the bump is twice differentiable: no coarse grid resolves it
        return None
    if op == "field":
        if case["n"] > 8192:  # dense, and the curves' node counts fix the quadrature
            return None
        g = _curve(case, seed)
        N = case["n"]
        K = _dense(case, g)
        U, P = _borders(g, N)
        h = U.shape[1]
        A = torch.zeros((2 * N + h, 2 * N + h), dtype=torch.float64, device=K.device)
        A[:2 * N, :2 * N] = K
        A[:2 * N, 2 * N:] = torch.from_numpy(U).to(K.device)
        A[2 * N:, :2 * N] = torch.from_numpy(P).to(K.device)
        A[2 * N:, 2 * N:] = -torch.eye(h, dtype=torch.float64, device=K.device)
        b = np.concatenate([_data(case, seed, g), np.zeros(h)])
        x = torch.linalg.solve(A, torch.from_numpy(b).to(K.device)).cpu().numpy()
        tg = _targets(case, seed, g)
        u = _field(case, g, tg, x[:2 * N])
        for k in range(h // 3):
            u += _hole_flow(tg - g["holes"]["centers"][k], 1 / (4 * math.pi)) @ \
                x[2 * N + 3 * k:2 * N + 3 * k + 3]
        return [x[:2 * N], x[2 * N:], u]
    nr = case.get("nrhs", 1)
    X = _solution(case, lambda m: _curve(case, seed, m),
                  lambda g: [_data(case, seed, g, k) for k in range(nr)], case["n"])
    return X if op == "solves" else X[:, 0]
