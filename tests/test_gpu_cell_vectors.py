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
from test_gpu_parity import gdm_params, ld_params, le_params

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
@pytest.mark.parametrize("prepass", ["0", "1"])
def test_decreasing_interaction(n, jitter, app, r, prepass, monkeypatch):
    """R and K of the decreasing nonlocal interaction (node kernel and cell vectors) against the oracle,
    also with a factor that reaches zero at omega = 1, and the residual alone."""
    monkeypatch.setenv("NUTO_AMD_GDM_PREPASS", prepass)
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


def test_adjoint_at_the_updated_history():
    """kappa' jumps where eeq meets the history, which is every loading point after an update: the adjoint
    and the tangent must take the same side there (K^T lambda of the device's K, within 1e-12 of |K|^T |lambda|)."""
    p, th = gdm_pair((5, 4, 3), N.FULL, jitter=0.1)
    u, e, kap = p.inputs()
    ctx = p.context()
    ctx.set_material_fields(*th)
    state = [to_dev(v) for v in (u, e, kap)]
    ctx.update_history(*state)
    lam = S.uniform(0x52, p.n_u + p.n_e, -1.0, 1.0)
    rp, ci = ctx.pattern()
    val = ctx.build_matrix(*state).cpu().numpy()
    kt, kb = kt_lambda(dict(row_ptr=rp, col=ci, val=val, bound=np.abs(val)), lam, len(lam))
    got = ctx.vjp(*state, to_dev(lam))[0].cpu().numpy()
    assert (np.abs(got - kt) <= 1e-12 * kb + 1e-300).all()


# (coordinate element, dof element, cells, rule); a workgroup takes 256 (one point), 16, 10 (25 points), 8, 4, 2 or 1 cells
GENERIC = [(N.QUAD4, N.QUAD4, (1, 1), (0, 1)), (N.QUAD4, N.QUAD4, (5, 4), (0, 2)), (N.QUAD4, N.QUAD4, (3, 3), (0, 5)),
           (N.QUAD4, N.QUAD4, (4, 3), (0, 5)), (N.QUAD4, N.QUAD4, (17, 16), (0, 1)), (N.TET4, N.TET4, (4, 4, 3), (1, 1)),
           (N.HEX8, N.HEX8, (3, 3, 1), (0, 2)), (N.HEX8, N.HEX8, (1, 1, 1), (0, 3)), (N.HEX8, N.HEX8, (2, 1, 1), (0, 4)),
           (N.HEX8, N.HEX20, (3, 1, 1), (0, 3)), (N.TET4, N.TET4, (1, 1, 1), (1, 1)), (N.TET4, N.TET4, (3, 2, 2), (1, 1)),
           (N.TET4, N.TET10, (3, 1, 1), (1, 2))]


@pytest.mark.parametrize("ct,dt,n,rule", GENERIC)
@pytest.mark.parametrize("kind", ["elastic", "local", "gradient"])
def test_generic_vectors_history_and_fields(ct, dt, n, rule, kind, monkeypatch):
    """The residual alone (cell vectors, and the single-pass kernel) against the oracle; kappa of the field
    output equals the updated history bit for bit."""
    dim = N.DIM[ct]
    if (kind != "elastic" and dim == 2) or (kind == "gradient" and (ct, dt) != (N.HEX8, N.HEX8)):
        pytest.skip("not provided")
    X, C = make_mesh(ct, n, lengths=tuple(float(v) for v in n) + (0.0,) * (3 - len(n)), jitter=0.0 if dim == 2 else 0.1)
    par = {"elastic": lambda: le_params(dim), "local": ld_params, "gradient": gdm_params}[kind]()
    p = Pair(ct, dt, X, C, *par, two_fields=kind == "gradient", rule=rule)
    u, e, kap = p.inputs()
    ctx = p.context()
    state = [to_dev(u), to_dev(e), to_dev(kap) if kind != "elastic" else None]
    ref = p.orc.assemble(u, e, kap)
    R = ctx.build_vector(*state)
    check_values(R.cpu().numpy(), ref["R"], ref["R_bound"], "R")
    monkeypatch.setenv("NUTO_AMD_GENERIC", "1")
    check_values(ctx.build_vector(*state).cpu().numpy(), ref["R"], ref["R_bound"], "R, single pass")
    monkeypatch.delenv("NUTO_AMD_GENERIC")
    stress = ctx.eval_ip(N.IP_STRESS, *state)
    assert stress.shape == (p.ncells, p.nip, 3 if dim == 2 else 6)
    if kind == "elastic":
        return
    kappa, before = ctx.eval_ip(N.IP_KAPPA, *state), state[2].clone()
    ctx.update_history(*state)
    assert np.array_equal(state[2].view(p.nip, p.ncells).T.cpu().numpy(), kappa[:, :, 0].cpu().numpy())
    assert (state[2] >= before).all() and (state[2] > before).any()
    # the residual depends on max(history, driving strain): unchanged by the update
    assert np.array_equal(ctx.build_vector(*state).cpu().numpy(), R.cpu().numpy())
    ctx.update_history(*state)
    assert np.array_equal(state[2].view(p.nip, p.ncells).T.cpu().numpy(), kappa[:, :, 0].cpu().numpy())


@pytest.mark.parametrize("n,order", [((511, 511), 1), ((600, 500), 2), ((180, 180), 3), ((255, 127), 5)])
def test_quad4_vectors_at_the_limits(n, order, monkeypatch):
    """quad4 residuals on either side of the sizes between cell vectors and the row-owner kernel: the same as the
    row-owner kernel's (forced), within 1e-13 of the largest entry"""
    for m in ((n[0] - 1, n[1]), n):
        X, C = make_mesh(N.QUAD4, m)
        ranks, nn = N.dof_layer(N.QUAD4, C, N.QUAD4)
        ctx = N.Context()
        ctx.set_cells(N.QUAD4, X, C)
        ctx.set_dof_type(0, N.QUAD4, 2, 2 * nn, N.cell_dofs(ranks, 2))
        ctx.set_integrand(N.linear_elastic_params(2, 30000.0, 0.2))
        ctx.set_rule(0, order)
        ctx.build_pattern()
        u = to_dev(S.uniform(S.SEED_U, 2 * nn, -1e-3, 1e-3))
        R = ctx.build_vector(u).cpu().numpy()
        monkeypatch.setenv("NUTO_AMD_GENERIC", "1")
        want = ctx.build_vector(u).cpu().numpy()
        monkeypatch.delenv("NUTO_AMD_GENERIC")
        assert np.abs(R - want).max() <= 1e-13 * np.abs(want).max()


# local damage: (coordinate element, dof element, cells, rule, forms of the matrix assembly)
LOCAL = [(N.HEX8, N.HEX8, (4, 3, 3), (0, 2), "0123"), (N.HEX8, N.HEX8, (2, 2, 2), (0, 3), "0123"),
         (N.HEX8, N.HEX8, (2, 2, 2), (0, 4), "0"), (N.HEX8, N.HEX20, (3, 2, 2), (0, 3), "0123"),
         (N.TET4, N.TET4, (3, 3, 3), (1, 1), "01234"), (N.TET4, N.TET10, (2, 2, 2), (1, 2), "0123"),
         (N.TET10, N.TET10, (2, 2, 2), (1, 2), "0123")]


def tet10_mesh(n):
    """quadratic tetrahedra with curved edges"""
    X, C = make_mesh(N.TET4, n, lengths=tuple(float(v) for v in n), jitter=0.1)
    C10, nn = N.dof_layer(N.TET4, C, N.TET10)
    mid = X[C[:, [0, 1, 0, 0, 2, 1]]] + X[C[:, [1, 2, 2, 3, 3, 3]]]
    X10 = np.zeros((nn, 3))
    X10[C10[:, :4]] = X[C]
    X10[C10[:, 4:]] = 0.5 * mid
    edge = np.unique(C10[:, 4:])
    X10[edge] += S.uniform(0x53, 3 * len(edge), -0.02, 0.02).reshape(-1, 3)
    return X10, C10


def at_updated_history(ct, dt, n, rule):
    """A context, displacements, the history right after an update with them, and a history lower by 1e-10 of
    itself, at which every point that the update raised is loading for certain."""
    X, C = tet10_mesh(n) if ct == N.TET10 else make_mesh(ct, n, lengths=tuple(float(v) for v in n), jitter=0.1)
    p = Pair(ct, dt, X, C, *ld_params(), two_fields=False, rule=rule)
    u, _, kap = p.inputs()
    ctx = p.context()
    du, dk = to_dev(u), to_dev(kap)
    ctx.update_history(du, None, dk)
    return p, ctx, du, dk, dk * (1.0 - 1e-10)


def check_loading(matrix, updated, low):
    """omega differs by at most 1e-8 of the entries' magnitude between the two histories; points that the update
    did not raise (history above the strain) load in neither"""
    K, want = matrix(updated), matrix(low)
    assert np.abs(K - want).max() <= 1e-7 * np.abs(want).max()


@pytest.mark.parametrize("ct,dt,n,rule,forms", LOCAL)
def test_local_damage_loads_at_the_updated_history(ct, dt, n, rule, forms, monkeypatch):
    """Right after a history update every point it raised is loading: the tangent there equals the tangent
    at a history lower by 1e-10 of itself, in every form of the cell matrices and in the row-owner kernel."""
    _, ctx, du, dk, low = at_updated_history(ct, dt, n, rule)
    for form in forms + "r":
        if form == "r":
            monkeypatch.setenv("NUTO_AMD_TWO_PHASE", "0")
        else:
            monkeypatch.setenv("NUTO_AMD_CELL_GRAM", form)
        check_loading(lambda k: ctx.build_matrix(du, None, k).cpu().numpy(), dk, low)


def test_local_damage_loads_at_the_updated_history_in_large_tet4_meshes():
    """beyond 2048 nodes, where the rows come from node tiles by default"""
    _, ctx, du, dk, low = at_updated_history(N.TET4, N.TET4, (15, 12, 9), (1, 1))
    check_loading(lambda k: ctx.build_matrix(du, None, k).cpu().numpy(), dk, low)


@pytest.mark.parametrize("ct,dt,n,rule,forms", [v for v in LOCAL if v[:2] != (N.TET10, N.TET10) and v[3] not in ((0, 4),) and
                                                (v[1] == N.HEX20 or v[3] != (0, 3))])
def test_local_damage_loads_at_the_updated_history_in_batches(ct, dt, n, rule, forms, monkeypatch):
    """the launch modes of a batch (its meshes take each element's default rule)"""
    p, _, du, dk, low = at_updated_history(ct, dt, n, rule)
    b = N.Batch()
    b.set_integrand(p.params_dev)
    b.add_mesh(ct, dt, p.X, p.C, p.ranks, p.nn)
    b.build()
    for mode in range(7):
        for form in forms if mode >= 5 else forms[:1]:
            monkeypatch.setenv("NUTO_AMD_CELL_GRAM", form)
            check_loading(lambda k: b.assemble(du, None, k, mode=mode)[1].cpu().numpy(), dk, low)


@pytest.mark.parametrize("rule", [(0, 2), (0, 3), (0, 4)])
@pytest.mark.parametrize("env", [{}, {"NUTO_AMD_GDM_PREPASS": "0"}, {"NUTO_AMD_GDM_PREPASS": "1"}, {"NUTO_AMD_GENERIC": "1"}])
def test_gradient_damage_loads_at_the_updated_history(rule, env, monkeypatch):
    """The same for gradient damage, whose nonlocal strain decides: the node kernel with and without the
    pre-pass, the row-owner kernel, and the rules that only the latter has."""
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    X, C = make_mesh(N.HEX8, (9, 6, 5), lengths=(9.0, 6.0, 5.0), jitter=0.1)  # more than one block of 256 cells
    p = Pair(N.HEX8, N.HEX8, X, C, *gdm_params(), two_fields=True, rule=rule)
    u, e, kap = p.inputs()
    ctx = p.context()
    du, de, dk = to_dev(u), to_dev(e), to_dev(kap)
    kappa = ctx.eval_ip(N.IP_KAPPA, du, de, dk)
    ctx.update_history(du, de, dk)
    assert np.array_equal(dk.view(p.nip, p.ncells).T.cpu().numpy(), kappa[:, :, 0].cpu().numpy())
    check_loading(lambda k: ctx.build_matrix(du, de, k).cpu().numpy(), dk, dk * (1.0 - 1e-10))


@pytest.mark.parametrize("n,jitter", [((15, 15, 15), 0.0), ((15, 15, 15), 0.1), ((16, 15, 15), 0.0)])
@pytest.mark.parametrize("app", [N.FULL, N.UNILATERAL])
def test_one_launch_gives_the_same_bits(n, jitter, app, monkeypatch):
    """Meshes on either side of the size from which on the pre-pass runs (4096 nodes): with and without it
    the same bits, so a mesh gives the same result alone and in a large batch."""
    X, C = make_mesh(N.HEX8, n, lengths=tuple(float(v) for v in n), jitter=jitter)
    p = Pair(N.HEX8, N.HEX8, X, C, N.gradient_damage_params(damage_application=app), gdm_params(app)[1], True)
    state = [to_dev(v) for v in p.inputs()]
    out = []
    for prepass in ("0", "1", None):
        monkeypatch.delenv("NUTO_AMD_GDM_PREPASS", raising=False)
        if prepass:
            monkeypatch.setenv("NUTO_AMD_GDM_PREPASS", prepass)
        out.append([v.cpu().numpy() for v in p.context().build_vector_matrix(*state)])
    for R, K in out[1:]:
        assert np.array_equal(R, out[0][0]) and np.array_equal(K, out[0][1])
