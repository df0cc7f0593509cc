"""Residuals and adjoints that are assembled from cell vectors, at the edges of the kernels' groups of
cells: fewer cells than one group, a full one, one cell more, several with a remainder.

Residual against the oracle's R within 1e-12 of the sum of contribution magnitudes, the adjoint's state
part against K^T lambda of the oracle's K within 1e-12 of |K|^T |lambda|, its field part against central
differences of the oracle's R (relative step 1e-6, error 1e-6 of the largest entry).
"""
import numpy as np
import pytest

import nuto_amd as N
import oracle as O
from nuto_amd import synthetic as S
from pairs import Pair, check_values, make_mesh, to_dev
from test_gpu_adjoint import gdm_pair, kt_lambda

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (7, 1, 1), (2, 2, 2), (3, 3, 1), (5, 3, 2)])
@pytest.mark.parametrize("jitter", [0.0, 0.1])
@pytest.mark.parametrize("app", [N.FULL, N.UNILATERAL])
def test_gradient_damage(n, jitter, app):
    p, th = gdm_pair(n, app, jitter=jitter)
    u, e, kap = p.inputs()
    p.orc.set_theta(*th)
    ref = p.orc.assemble(u, e, kap)
    ctx = p.context()
    ctx.set_material_fields(*th)
    du, de, dk = to_dev(u), to_dev(e), to_dev(kap)
    check_values(ctx.build_vector(du, de, dk).cpu().numpy(), ref["R"], ref["R_bound"], "R")
    lam = S.uniform(0x51, len(ref["R"]), -1.0, 1.0)
    d_state, d_theta = ctx.vjp(du, de, dk, to_dev(lam))
    kt, kb = kt_lambda(ref, lam, len(lam))
    assert (np.abs(d_state.cpu().numpy() - kt) <= 1e-12 * kb + 1e-300).all()
    again, none = ctx.vjp(du, de, dk, to_dev(lam), want_theta=False)
    assert none is None and np.array_equal(again.cpu().numpy(), d_state.cpu().numpy())
    if n not in ((7, 1, 1), (3, 3, 1)):
        return
    got, fd = d_theta.cpu().numpy(), np.zeros((3, p.ncells))
    for k in range(3):
        for c in range(p.ncells):
            h, val = 1e-6 * th[k][c], []
            for sign in (1.0, -1.0):
                t = [np.array(v, dtype=np.float64) for v in th]
                t[k][c] += sign * h
                p.orc.set_theta(*t)
                val.append(lam @ p.orc.assemble(u, e, kap, want_k=False)["R"])
            fd[k, c] = (val[0] - val[1]) / (2 * h)
    assert (np.abs(got - fd) <= 1e-6 * np.abs(fd).max(axis=1, keepdims=True)).all()


@pytest.mark.parametrize("n,jitter", [((1, 1, 1), 0.0), ((3, 3, 1), 0.1), ((5, 3, 3), 0.0), ((4, 3, 3), 0.1)])
@pytest.mark.parametrize("app", [N.FULL, N.UNILATERAL])
@pytest.mark.parametrize("r", [0.005, 0.0])
def test_decreasing_interaction(n, jitter, app, r):
    """R and K of the decreasing nonlocal interaction (node kernel and cell vectors) against the oracle,
    also with a factor that reaches zero at omega = 1, and the residual alone."""
    X, C = make_mesh(N.HEX8, n, lengths=tuple(float(v) for v in n), jitter=jitter)
    dev = N.gradient_damage_params(damage_application=app, interaction=N.DECREASING, interaction_r=r)
    orc = O.Params(kind=1, dim=3, E=30000.0, nu=0.2, k=10.0, kappa0=1e-4, beta=100.0, alpha=0.99, c=4.0,
                   damage_application=app, interaction=1, interaction_r=r, interaction_eta=5.0)
    p = Pair(N.HEX8, N.HEX8, X, C, dev, orc, True)
    th = S.material_fields(p.ncells)
    p.orc.set_theta(*th)
    u, e, kap = p.inputs()
    ref = p.orc.assemble(u, e, kap)
    ctx = p.context()
    ctx.set_material_fields(*th)
    state = [to_dev(v) for v in (u, e, kap)]
    R, K = ctx.build_vector_matrix(*state)
    check_values(R.cpu().numpy(), ref["R"], ref["R_bound"], "R")
    check_values(K.cpu().numpy(), ref["val"], ref["bound"], "K")
    check_values(ctx.build_vector(*state).cpu().numpy(), ref["R"], ref["R_bound"], "R alone")
    assert np.array_equal(ctx.build_matrix(*state).cpu().numpy(), K.cpu().numpy())
    with pytest.raises(N.NutoError):
        ctx.vjp(*state, R)
