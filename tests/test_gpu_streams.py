"""Calls of one context (or batch) on several streams that nothing else orders: they share the context's work
memory, so a call on a newly set stream runs after the calls on the last one. Shown by events: with a long
product in front of the first call, the second stream's call may not have ended before it. And the same
calls under capture, where no wait on work outside the graph may be recorded."""
import numpy as np
import pytest
import torch

import nuto_amd as N
from nuto_amd import binding as B
from nuto_amd import synthetic as S
from pairs import Pair, make_mesh, to_dev
from test_gpu_parity import gdm_params, ld_params

pytestmark = pytest.mark.gpu


def gdm_pair(n=(6, 5, 4)):
    X, C = make_mesh(N.HEX8, n, lengths=tuple(float(v) for v in n), jitter=0.1)
    return Pair(N.HEX8, N.HEX8, X, C, *gdm_params(), True)


def two_streams(set_stream, call):
    """call() on stream a behind a long product, then on stream b: the results, and whether a had ended with b"""
    A = torch.rand(4096, 4096, dtype=torch.float64, device="cuda")
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    ended = [torch.cuda.Event(), torch.cuda.Event()]
    torch.cuda.synchronize()
    out = []
    for s, e in zip((a, b), ended):
        with torch.cuda.stream(s):
            set_stream(s.cuda_stream)
            if s is a:
                for _ in range(10):
                    A @ A
            out.append(call())
            e.record()
    ended[1].synchronize()
    ordered = ended[0].query()
    torch.cuda.synchronize()
    set_stream(0)
    return out, ordered


@pytest.mark.parametrize("what", ["vjp", "vector", "generic vector", "matrix"])
def test_second_stream_waits(what):
    if what == "generic vector":
        X, C = make_mesh(N.TET4, (5, 4, 3), lengths=(5.0, 4.0, 3.0), jitter=0.1)
        p = Pair(N.TET4, N.TET10, X, C, *ld_params(), two_fields=False)
    else:
        p = gdm_pair()
    ctx = p.context()
    state = [to_dev(v) for v in p.inputs()]
    lam = to_dev(S.uniform(0x54, p.n_u + p.n_e, -1.0, 1.0))
    call = {"vjp": lambda: ctx.vjp(*state, lam), "matrix": lambda: (ctx.build_matrix(*state),)}.get(
        what, lambda: (ctx.build_vector(*state),))
    ref = [t.cpu().numpy() for t in call()]
    out, ordered = two_streams(ctx.set_stream, call)
    assert ordered
    for got in out:
        assert all(np.array_equal(g.cpu().numpy(), r) for g, r in zip(got, ref))


def test_second_stream_of_a_batch_waits():
    p = gdm_pair()
    b = N.Batch()
    b.set_integrand(p.params_dev)
    b.add_mesh(N.HEX8, N.HEX8, p.X, p.C, p.ranks, p.nn)
    b.build()
    state = [to_dev(v) for v in p.inputs()]
    R = torch.empty(b.sizes["R"], dtype=torch.float64, device="cuda")
    K = torch.empty(b.sizes["K"], dtype=torch.float64, device="cuda")
    ref = [t.cpu().numpy() for t in b.assemble(*state, mode=3)]

    def call():  # the C ABI call itself: the Python one orders its streams
        r, k = torch.empty_like(R), torch.empty_like(K)
        assert B.lib().nuto_batch_assemble(b.h, *B._ptrs(*state, r, k), 3) == 0
        return r, k

    def set_stream(s):
        assert B.lib().nuto_batch_set_stream(b.h, B.ctypes.c_void_p(s or b.stream.cuda_stream)) == 0

    out, ordered = two_streams(set_stream, call)
    assert ordered
    for got in out:
        assert all(np.array_equal(g.cpu().numpy(), r) for g, r in zip(got, ref))


def test_capture_on_another_stream():
    """set_stream to a stream that is being captured, and back: no wait on work outside the graph is recorded, and
    every replay gives the eager result"""
    p = gdm_pair()
    ctx = p.context()
    state = [to_dev(v) for v in p.inputs()]
    lam = to_dev(S.uniform(0x54, p.n_u + p.n_e, -1.0, 1.0))
    ref = [ctx.build_vector(*state).cpu().numpy(), ctx.vjp(*state, lam)[0].cpu().numpy()]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ctx.set_stream(torch.cuda.current_stream().cuda_stream)
        R = ctx.build_vector(*state)
        d = ctx.vjp(*state, lam)[0]
    ctx.set_stream(0)
    for _ in range(4):
        R.fill_(float("nan"))
        d.fill_(float("nan"))
        g.replay()
        assert np.array_equal(ctx.build_vector(*state).cpu().numpy(), ref[0])  # eager work in between
        torch.cuda.synchronize()
        assert np.array_equal(R.cpu().numpy(), ref[0]) and np.array_equal(d.cpu().numpy(), ref[1])
