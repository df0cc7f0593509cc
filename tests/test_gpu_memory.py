"""Device memory that contexts and batches hold: work memory that no call would use is not taken. Measured by the
device's free memory around a call, with 16 MiB to spare for the allocator's granularity."""
import numpy as np
import pytest
import torch

import nuto_amd as N
from nuto_amd import synthetic as S
from pairs import make_mesh, to_dev

pytestmark = pytest.mark.gpu
SPARE = 16 << 20


def taken(call):
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    out = call()
    torch.cuda.synchronize()
    return out, before - torch.cuda.mem_get_info()[0]


def prepared(ct, n, params, two_fields, jitter=0.1):
    """(context before its pattern, coordinates, connectivity, dof ranks, dof nodes)"""
    X, C = make_mesh(ct, n, lengths=tuple(float(v) for v in n), jitter=jitter)
    ranks, nn = N.dof_layer(ct, C, ct)
    ctx = N.Context()
    ctx.set_cells(ct, X, C)
    ctx.set_dof_type(0, ct, 3, 3 * nn, N.cell_dofs(ranks, 3))
    if two_fields:
        ctx.set_dof_type(1, ct, 1, nn, N.cell_dofs(ranks, 1))
    if params is not None:
        ctx.set_integrand(params)
    ctx.set_rule(*((0, 2) if ct == N.HEX8 else (1, 1)))
    return ctx, X, C, ranks, nn


@pytest.fixture(autouse=True)
def warm():
    """first launches load code and scratch"""
    for ct, params, two in ((N.HEX8, N.gradient_damage_params(), True), (N.HEX8, N.linear_elastic_params(3, 3e4, 0.2), False),
                            (N.TET4, N.local_damage_params(), False)):
        ctx, _, C, _, nn = prepared(ct, (16, 13, 13), params, two)
        ctx.build_pattern()
        state = [to_dev(np.zeros(k)) for k in (3 * nn, nn, len(C) * 8 if ct == N.HEX8 else len(C))]
        ctx.build_vector_matrix(state[0], state[1] if two else None, state[2] if ct == N.TET4 or two else None)


def test_gradient_damage_context():
    """The hex8 plan's own work memory serves the vectors too: nothing beside the pattern and the plan."""
    ctx, X, C, _, nn = prepared(N.HEX8, (64, 64, 64), N.gradient_damage_params(), True)
    _, got = taken(ctx.build_pattern)
    nc = len(C)
    pairs = ctx.nnz // 16
    graph = 4 * nn + 8 * nc * (4 + 1) + 64 * nc * 2 + 4 * nn + 4 * pairs  # incidence, slots, adjacency
    csr = 4 * 4 * nn + 4 * ctx.nnz
    plan = nn * (16 + 4) + nn * 8 * (4 + 1) + nn * 64 + nc * 8 * (80 + 144)  # heads, tables, geometry, records
    assert got <= graph + csr + plan + SPARE


def test_generic_vector_allocates_nothing():
    """reserved with the pattern, or with the integrand and the rule where they come later"""
    ctx, _, C, _, nn = prepared(N.HEX8, (64, 64, 64), None, False)
    ctx.build_pattern()
    _, got = taken(lambda: ctx.set_integrand(N.linear_elastic_params(3, 30000.0, 0.2)))
    assert got >= 192 * len(C) - SPARE  # 24 doubles per cell, now that they are needed
    u = to_dev(S.uniform(S.SEED_U, 3 * nn, -1e-3, 1e-3))
    R = torch.empty(3 * nn, dtype=torch.float64, device="cuda")
    ctx.build_vector(u, out=R)  # the tables of the rule
    _, got = taken(lambda: ctx.build_vector(u, out=R))
    assert got == 0


def test_tet4_tiles_stage_nothing():
    """the matrix of a tet4 mesh that takes node tiles, alone and in a batch"""
    ctx, X, C, ranks, nn = prepared(N.TET4, (30, 30, 30), N.local_damage_params(), False)
    ctx.build_pattern()
    u, kap = to_dev(S.uniform(S.SEED_U, 3 * nn, -5e-3, 5e-3)), to_dev(S.uniform(S.SEED_KAPPA, len(C), 0.0, 3e-4))
    R = torch.empty(ctx.n_rows, dtype=torch.float64, device="cuda")
    K = torch.empty(ctx.nnz, dtype=torch.float64, device="cuda")
    _, got = taken(lambda: ctx.build_vector_matrix(u, None, kap, R, K))
    assert got <= SPARE
    b = N.Batch()
    b.set_integrand(N.local_damage_params())
    b.add_mesh(N.TET4, N.TET4, X, C, ranks, nn)
    b.build()
    Rb, Kb = torch.empty_like(R), torch.empty_like(K)
    _, got = taken(lambda: b.assemble(u, None, kap, Rb, Kb, mode=5))
    assert got <= SPARE
    assert torch.equal(Rb, R) and torch.equal(Kb, K)


def test_batch_reserves_no_vectors():
    """a batch assembles no vector alone: its groups hold less than a context of the same mesh"""
    params = N.linear_elastic_params(3, 30000.0, 0.2)
    ctx, X, C, ranks, nn = prepared(N.HEX8, (64, 64, 64), params, False)
    _, alone = taken(ctx.build_pattern)
    b = N.Batch()
    b.set_integrand(params)
    b.add_mesh(N.HEX8, N.HEX8, X, C, ranks, nn)
    _, got = taken(b.build)
    mesh = 24 * nn + 32 * len(C) * 2  # coordinates and connectivities, which the context had before
    assert got <= alone + mesh - 192 * len(C) + SPARE
