"""Device solves stopped at a given iteration against the same iteration in numpy.

The host queues several iterations before it reads the state of an earlier one, so a limit below,
at and beyond a queued group must stop at exactly that iteration; rows longer than 128 columns leave
the part of the K product that is loaded ahead. Conjugate gradients and BiCGSTAB with the diagonal
preconditioner are restated densely on C^T K C. Tolerance: at most 9 iterations on systems with
condition numbers below 1e4, each step's rounding (1e-16) amplified by at most the condition number,
with 3 digits to spare: 1e-9 of the largest entry.
"""
import numpy as np
import pytest

import nuto_amd as N
from pairs import Pair, make_mesh, to_dev
from test_gpu_parity import gdm_params, le_params

pytestmark = pytest.mark.gpu


class Masked:
    """rows and columns `ind` of a sparse matrix, with its diagonal"""

    def __init__(self, K, ind, diag):
        self.K, self.ind, self.diag = K, ind, diag[ind]

    def __matmul__(self, v):
        full = np.zeros(self.K.shape[0])
        full[self.ind] = v
        return (self.K @ full)[self.ind]


def cg(A, b, k):
    d = 1.0 / (A.diag if isinstance(A, Masked) else np.diag(A))
    x, r = np.zeros_like(b), b.copy()
    z = d * r
    p, rz = z.copy(), r @ z
    for _ in range(k):
        q = A @ p
        a = rz / (p @ q)
        x, r = x + a * p, r - a * q
        z = d * r
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return x, np.linalg.norm(r) / np.linalg.norm(b)


def bicgstab(A, b, k):
    d = 1.0 / (A.diag if isinstance(A, Masked) else np.diag(A))
    x, r, r0 = np.zeros_like(b), b.copy(), b.copy()
    p = v = np.zeros_like(b)
    rho = alpha = w = 1.0
    for _ in range(k):
        rho, old = r0 @ r, rho
        p = r + (rho / old) * (alpha / w) * (p - w * v)
        y = d * p
        v = A @ y
        alpha = rho / (r0 @ v)
        s = r - alpha * v
        z = d * s
        t = A @ z
        w = (t @ s) / (t @ t)
        x = x + alpha * y + w * z
        r = s - w * t
    return x, np.linalg.norm(r) / np.linalg.norm(b)


@pytest.mark.parametrize("element,n,terms", [("quad4", (1, 1), False), ("quad4", (7, 3), True), ("hex8", (2, 3, 2), False),
                                             ("hex20", (2, 1, 2), True), ("hex20", (1, 2, 1), False)])
@pytest.mark.parametrize("method", [N.SOLVER_CG, N.SOLVER_BICGSTAB])
def test_stops_at_the_limit(element, n, terms, method):
    ct = N.QUAD4 if element == "quad4" else N.HEX8
    dt = {"quad4": N.QUAD4, "hex8": N.HEX8, "hex20": N.HEX20}[element]
    X, C = make_mesh(ct, n, (1.0, 1.2, 0.9))
    dim = N.DIM[ct]
    p = Pair(ct, dt, X, C, *le_params(dim), two_fields=False)
    ctx = p.context()
    K = ctx.build_matrix(to_dev(np.zeros(p.n_u)))
    rp, ci = ctx.pattern()
    dense = np.zeros((p.n_u, p.n_u))
    dense[np.repeat(np.arange(p.n_u), np.diff(rp)), ci] = K.cpu().numpy()
    xs = np.zeros((p.nn, dim))
    xs[p.ranks[:, :C.shape[1]].ravel()] = X[C.ravel(), :dim]
    xs[np.setdiff1d(np.arange(p.nn), p.ranks[:, :C.shape[1]])] = 1.0  # edge nodes: not clamped here
    left = np.nonzero(xs[:, 0] < 1e-12)[0]
    eqs = [(int(dim * r + c), []) for r in left for c in range(dim)]
    if terms:
        free = np.setdiff1d(np.arange(p.n_u), [q[0] for q in eqs])
        eqs.append((int(free[3]), [(int(free[0]), -0.5), (int(free[-1]), 0.25), (int(free[0]), 0.1)]))
        eqs.append((int(free[5]), [(int(free[0]), -0.3)]))
    ctx.set_constraints(0, eqs)
    ind = np.setdiff1d(np.arange(p.n_u), [q[0] for q in eqs])
    Cm = np.zeros((p.n_u, len(ind)))
    Cm[ind, np.arange(len(ind))] = 1.0
    for dep, ts in eqs:
        for g, coef in ts:
            Cm[dep, np.searchsorted(ind, g)] -= coef
    f = np.random.default_rng(3).uniform(-1.0, 1.0, p.n_u)
    A, b = Cm.T @ dense @ Cm, Cm.T @ f
    for k in [k for k in (1, 3, 4, 5, 8, 9) if k < len(ind) // 2]:
        x, info = ctx.solve(K, to_dev(f), method=method, tol=1e-300, max_iter=k)
        want, rel = (cg if method == N.SOLVER_CG else bicgstab)(A, b, k)
        want = Cm @ want
        assert info["iterations"] == k
        assert np.abs(x.cpu().numpy() - want).max() <= 1e-9 * np.abs(want).max()
        assert abs(info["relative_residual"] - rel) <= 1e-9 * max(rel, 1.0)
    # to convergence, and a right-hand side of zero
    x, info = ctx.solve(K, to_dev(f), method=method, tol=1e-13)
    want = Cm @ np.linalg.solve(A, b)
    assert np.abs(x.cpu().numpy() - want).max() <= 1e-9 * np.abs(want).max()
    x, info = ctx.solve(K, to_dev(np.zeros(p.n_u)), method=method)
    assert info["iterations"] == 0 and info["relative_residual"] == 0.0 and not x.cpu().numpy().any()


@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("form", ["0", "1", "terms"])
def test_bicgstab_restart(seed, form, monkeypatch):
    """A lower triangular matrix on one quad4 cell (all its dofs are coupled) with f = e_0: after the
    first iteration the residual has no entry at dof 0, so rho = 0 and the solver must restart: with stored
    vectors, with the products forming theirs, and with a constraint term (dof 7 = half of dof 6)."""
    if form != "terms":
        monkeypatch.setenv("NUTO_AMD_SOLVE_FORM", form)
    X, C = make_mesh(N.QUAD4, (1, 1), (1.0, 1.0, 1.0))
    p = Pair(N.QUAD4, N.QUAD4, X, C, *le_params(2), two_fields=False)
    ctx = p.context()
    rp, ci = ctx.pattern()
    assert len(ci) == 64
    rng = np.random.default_rng(seed)
    A = np.tril(rng.uniform(-0.5, 0.5, (8, 8)), -1) + np.diag(rng.uniform(1.0, 2.0, 8))
    K = to_dev(A[np.repeat(np.arange(8), np.diff(rp)), ci])
    ctx.set_constraints(0, [(7, [(6, -0.5)])] if form == "terms" else [])
    Cm = np.eye(8)[:, :7] if form == "terms" else np.eye(8)
    if form == "terms":
        Cm[7, 6] = 0.5
    f = np.zeros(8)
    f[0] = 1.0
    x, info = ctx.solve(K, to_dev(f), method=N.SOLVER_BICGSTAB, tol=1e-13, max_iter=200)
    want = Cm @ np.linalg.solve(Cm.T @ A @ Cm, Cm.T @ f)
    assert info["iterations"] < 200 and info["relative_residual"] <= 1e-13
    assert np.abs(x.cpu().numpy() - want).max() <= 1e-9 * np.abs(want).max()


@pytest.mark.parametrize("case,n", [("quad4", (1, 1)), ("quad4", (5, 4)), ("quad4", (100, 90)), ("hex8", (1, 1, 1)),
                                    ("hex8", (21, 21, 20)), ("hex20", (2, 1, 2)), ("gdm", (1, 2, 1)),
                                    ("gdm", (21, 21, 20))])
@pytest.mark.parametrize("method", [N.SOLVER_CG, N.SOLVER_BICGSTAB])
def test_formed_vectors_give_the_same_bits(case, n, method, monkeypatch):
    """The K product that forms its input where it gathers it, against the same iteration with a kernel of
    its own for every vector: one node per wave and several (more than 8192 nodes), every row structure,
    limits inside and beyond a queued group. The operations and the order of the sums are the same."""
    ct = N.QUAD4 if case == "quad4" else N.HEX8
    dt = {"quad4": N.QUAD4, "hex20": N.HEX20}.get(case, N.HEX8)
    X, C = make_mesh(ct, n, (1.0, 1.2, 0.9), jitter=0.1 if max(n) > 2 else 0.0)
    dim = N.DIM[ct]
    params = gdm_params() if case == "gdm" else le_params(dim)
    p = Pair(ct, dt, X, C, *params, two_fields=case == "gdm")
    ctx = p.context()
    K = ctx.build_vector_matrix(*[to_dev(v) for v in p.inputs()])[1] if case == "gdm" else \
        ctx.build_matrix(to_dev(np.zeros(p.n_u)))
    xs = np.ones((p.nn, dim))
    xs[p.ranks[:, :C.shape[1]].ravel()] = X[C.ravel(), :dim]
    ctx.set_constraints(0, [(int(dim * r + c), []) for r in np.nonzero(xs[:, 0] < 1e-12)[0] for c in range(dim)])
    f = to_dev(np.random.default_rng(4).uniform(-1.0, 1.0, len(ctx.pattern()[0]) - 1))
    for k in (1, 2, 4, 7):
        out = []
        for form in ("0", "1"):
            monkeypatch.setenv("NUTO_AMD_SOLVE_FORM", form)
            x, info = ctx.solve(K, f, method=method, tol=1e-12, max_iter=k)
            out.append((x.cpu().numpy(), info["iterations"], info["relative_residual"]))
        assert out[0][1:] == out[1][1:] and np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("case,n", [("quad4", (382, 255)), ("quad4", (383, 255)), ("quad4", (400, 300)), ("hex8", (41, 40, 40)),
                                    ("gdm", (37, 37, 36))])
@pytest.mark.parametrize("method", [N.SOLVER_CG, N.SOLVER_BICGSTAB])
def test_large_systems(case, n, method):
    """On either side of 196,608 rows, from where on a wave of the K product has one node and its partial sums
    are added by a kernel of their own; the same iterations in numpy on the sparse matrix."""
    from scipy.sparse import csr_matrix

    ct = N.QUAD4 if case == "quad4" else N.HEX8
    dim = N.DIM[ct]
    X, C = make_mesh(ct, n, tuple(float(v) for v in n) + (0.0,) * (3 - dim))
    ranks, nn = N.dof_layer(ct, C, ct)
    ctx = N.Context()
    ctx.set_cells(ct, X, C)
    ctx.set_dof_type(0, ct, dim, dim * nn, N.cell_dofs(ranks, dim))
    u = to_dev(np.random.default_rng(5).uniform(-1e-4, 1e-4, dim * nn))
    if case == "gdm":
        ctx.set_dof_type(1, ct, 1, nn, N.cell_dofs(ranks, 1))
        ctx.set_integrand(N.gradient_damage_params())
        ctx.set_rule(0, 2)
        ctx.build_pattern()
        K = ctx.build_matrix(u, to_dev(np.full(nn, 5e-5)), to_dev(np.zeros(8 * len(C))))
    else:
        ctx.set_integrand(N.linear_elastic_params(dim, 30000.0, 0.2))
        ctx.set_rule(0, 2)
        ctx.build_pattern()
        K = ctx.build_matrix(u)
    left = np.unique(ranks.ravel()[X[C.ravel(), 0] < 1e-12])
    dep = (dim * left[:, None] + np.arange(dim)).ravel()
    ctx.set_constraints(0, [(int(d), []) for d in dep])
    rp, ci = ctx.pattern()
    keep = np.ones(len(rp) - 1)
    keep[dep] = 0.0
    ind = np.nonzero(keep)[0]
    val = K.cpu().numpy()
    diag = csr_matrix((val, ci, rp)).diagonal()
    A = Masked(csr_matrix((val, ci, rp)), ind, diag)
    f = np.random.default_rng(4).uniform(-1.0, 1.0, len(keep))
    for k in (1, 5):
        x, info = ctx.solve(K, to_dev(f), method=method, tol=1e-300, max_iter=k)
        want, rel = (cg if method == N.SOLVER_CG else bicgstab)(A, f[ind], k)
        assert info["iterations"] == k
        assert np.abs(x.cpu().numpy()[ind] - want).max() <= 1e-9 * np.abs(want).max()
        assert not x.cpu().numpy()[dep].any()
        assert abs(info["relative_residual"] - rel) <= 1e-9 * max(rel, 1.0)
