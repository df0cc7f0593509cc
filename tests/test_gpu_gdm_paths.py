"""The hex8 gradient-damage node kernel with and without its per-(cell, IP) state pre-pass
(NUTO_AMD_GDM_PREPASS=0 recomputes the IP state in the node kernel), against the oracle on
jittered and degenerate meshes, and with Cell::Id history columns (GradientDamage.h:137 indexes
mKappas by cell id)."""
import numpy as np
import pytest

import nuto_amd as N
import oracle as O
from pairs import Pair, check_values, make_mesh, to_dev

pytestmark = pytest.mark.gpu


def gdm(app=N.FULL):
    dev = N.gradient_damage_params(damage_application=app)
    orc = O.Params(kind=1, dim=3, E=30000.0, nu=0.2, k=10.0, kappa0=1e-4, beta=100.0, alpha=0.99, c=4.0,
                   damage_application=app)
    return dev, orc


@pytest.fixture(params=["1", "0"], ids=["prepass", "recompute"])
def path(request, monkeypatch):
    monkeypatch.setenv("NUTO_AMD_GDM_PREPASS", request.param)
    return request.param


@pytest.mark.parametrize("dims,jitter,app", [((3, 3, 2), 0.15, N.FULL), ((3, 2, 3), 0.15, N.UNILATERAL),
                                             ((1, 1, 1), 0.0, N.FULL), ((3, 1, 1), 0.05, N.FULL)])
def test_against_oracle(path, dims, jitter, app):
    X, C = make_mesh(N.HEX8, dims, tuple(float(d) for d in dims), jitter=jitter, seed=11)
    dev, orc = gdm(app)
    p = Pair(N.HEX8, N.HEX8, X, C, dev, orc, True)
    u, e, kap = p.inputs()
    ctx = p.context()
    R, K = ctx.build_vector_matrix(to_dev(u), to_dev(e), to_dev(kap))
    ref = p.orc.assemble(u, e, kap)
    rp, ci = ctx.pattern()
    assert np.array_equal(rp, ref["row_ptr"]) and np.array_equal(ci, ref["col"])
    check_values(R.cpu().numpy(), ref["R"], ref["R_bound"], "R")
    check_values(K.cpu().numpy(), ref["val"], ref["bound"], "K")


def test_cell_ids_select_history_columns(path):
    X, C = make_mesh(N.HEX8, (3, 2, 2), (3.0, 2.0, 2.0))
    dev, _ = gdm()
    ranks, nn = N.dof_layer(N.HEX8, C, N.HEX8)
    nc = C.shape[0]
    rng = np.random.default_rng(5)
    ids = rng.permutation(nc).astype(np.int32) + 3  # Cell::Id values, not positions
    ld = nc + 7
    from nuto_amd import synthetic as S
    u = S.uniform(S.SEED_U, 3 * nn, -5e-3, 5e-3)
    e = S.uniform(S.SEED_E, nn, 0.0, 5e-4)
    kap = S.uniform(S.SEED_KAPPA, nc * 8, 0.0, 3e-4)       # by position: c + ip * nc
    kap_id = np.full(ld * 8, np.nan)
    for c in range(nc):
        for ip in range(8):
            kap_id[ids[c] + ip * ld] = kap[c + ip * nc]     # by id: id(c) + ip * ld
    out = []
    for cell_ids, kk, hld in ((None, kap, None), (ids, kap_id, ld)):
        ctx = N.Context()
        ctx.set_cells(N.HEX8, X, C, cell_ids)
        ctx.set_dof_type(0, N.HEX8, 3, 3 * nn, N.cell_dofs(ranks, 3))
        ctx.set_dof_type(1, N.HEX8, 1, nn, N.cell_dofs(ranks, 1))
        ctx.set_integrand(dev)
        ctx.set_rule(0, 2)
        if hld:
            ctx.set_history_ld(hld)
        ctx.build_pattern()
        out.append([t.cpu().numpy() for t in ctx.build_vector_matrix(to_dev(u), to_dev(e), to_dev(kk))])
        dk = to_dev(kk)
        ctx.update_history(to_dev(u), to_dev(e), dk)
        out[-1].append(dk.cpu().numpy())
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    # the update writes the cells' own columns and nothing else
    updated, by_id = out[0][2].reshape(8, nc), out[1][2].reshape(8, ld)
    assert np.array_equal(by_id[:, ids], updated) and (updated > kap.reshape(8, nc)).any()
    assert np.isnan(np.delete(by_id, ids, axis=1)).all()
