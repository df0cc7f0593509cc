"""Node tiles (rows of 16 or 8 consecutive nodes built in LDS) at the edges of the tiles: fewer nodes than one
tile, exactly one, one node more; nodes with more cells than the lanes of a node take in one turn; and a node
whose rows do not fit in LDS, which leaves the tiles for the kernels behind them. R and K against the oracle.
"""
import numpy as np
import pytest

import nuto_amd as N
from pairs import Pair, check_values, make_mesh, to_dev
from test_gpu_parity import ld_params, le_params

pytestmark = pytest.mark.gpu


def quad_fan(k):
    """k quadrilaterals around one node"""
    a = np.linspace(0.0, 2.0 * np.pi, 2 * k, endpoint=False)
    radius = np.where(np.arange(2 * k) % 2 == 0, 1.0, 1.3)
    X = np.concatenate([[[0.0, 0.0]], np.stack([radius * np.cos(a), radius * np.sin(a)], 1)])
    ring = 1 + np.arange(2 * k)
    C = np.stack([np.zeros(k, int), ring[0::2], ring[1::2], np.roll(ring, -2)[0::2]], 1)
    return X, C.astype(np.int32)


def check(p, u, kap):
    ctx = p.context()
    R, K = ctx.build_vector_matrix(to_dev(u), None, to_dev(kap))
    ref = p.orc.assemble(u, None, kap)
    check_values(R.cpu().numpy(), ref["R"], ref["R_bound"], "R")
    check_values(K.cpu().numpy(), ref["val"], ref["bound"], "K")
    assert np.array_equal(ctx.build_matrix(to_dev(u), None, to_dev(kap)).cpu().numpy(), K.cpu().numpy())


@pytest.mark.parametrize("rule", [(0, 1), (0, 2), (0, 5)])
@pytest.mark.parametrize("mesh", [(1, 1), (7, 1), (3, 3), (16, 1), (9, 7), "fan3", "fan9", "fan1500"])
def test_quad4(mesh, rule):
    X, C = quad_fan(int(mesh[3:])) if isinstance(mesh, str) else make_mesh(N.QUAD4, mesh)
    p = Pair(N.QUAD4, N.QUAD4, X, C, *le_params(2), two_fields=False, rule=rule)
    u, _, _ = p.inputs(u_range=1e-3)
    check(p, u, None)


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (3, 3, 3), (15, 11, 9), (15, 12, 9)])
@pytest.mark.parametrize("kind", ["elastic", "local", "unilateral"])
@pytest.mark.parametrize("form", ["", "4"])
def test_tet4(n, kind, form, monkeypatch):
    """on either side of the size from which on the tiles are taken (2048 nodes), and the tiles at every size"""
    if form:
        monkeypatch.setenv("NUTO_AMD_CELL_GRAM", form)
    X, C = make_mesh(N.TET4, n, lengths=tuple(float(v) for v in n), jitter=0.1)
    par = {"elastic": lambda: le_params(3), "local": ld_params, "unilateral": lambda: ld_params(N.UNILATERAL)}[kind]()
    p = Pair(N.TET4, N.TET4, X, C, *par, two_fields=False)
    u, _, kap = p.inputs()
    check(p, u, None if kind == "elastic" else kap)
