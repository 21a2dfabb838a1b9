"""Solves queued a few launches ahead of the device (no host checks, the
default) equal solves checked after every CG iteration bit for bit: one after
the other on a context whose earlier solves left flags queued, behind other
work that outlasts the polling, and captured into a graph (where everything is
queued) and replayed."""
import numpy as np
import pytest

from arapgs_amd import arapgs, scenes as S
from helpers import small_scene

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def solver_of(ctx, sc, **kw):
    s = arapgs.Solver(ctx, sc["nbr"], sc["blocks"], sc["types"], sc["src_idx"], sc["src_w"], sc["nodes"], **kw)
    s.set_coarse_refresh(1000)
    return s


def same(a, b):
    import torch
    n = int(a[2].item())
    return n == int(b[2].item()) and torch.equal(a[0], b[0]) and torch.equal(a[1][: n + 1], b[1][: n + 1])


@pytest.fixture(scope="module")
def scene():
    return small_scene(n=20000, n_nodes=128, seed=1)


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("cap", [1, 2, 3, 100])
def test_queued_ahead_equals_checked(ctx, scene, mode, cap):
    nodes = T(scene["nodes"])
    s = solver_of(ctx, scene, cg_max_iters=cap)
    s.set_cg_mode(mode)
    for i, (fraction, iters) in enumerate(((0.7, 6), (0.1, 10), (0.0, 4), (0.4, 1), (0.4, 8))):
        aims = T(S.frame_aims(scene["scene"], scene["nodes"], scene["blocks"], scene["types"], fraction))
        got = {}
        for every in (1, 0) if i % 2 else (0, 1):
            s.set_host_checks(every)
            got[every] = s.solve(nodes, aims, iters, stop_rule=i != 3)
        assert same(got[0], got[1]), (mode, cap, fraction, iters)


@pytest.mark.parametrize("products,size", [(4, 8192), (1, 8192), (30, 4096), (8, 2048)])
@pytest.mark.parametrize("mode", [0, 2])
def test_behind_other_work(ctx, scene, products, size, mode):
    import torch
    nodes = T(scene["nodes"])
    aims = T(S.frame_aims(scene["scene"], scene["nodes"], scene["blocks"], scene["types"], 0.5))
    s = solver_of(ctx, scene)
    s.set_cg_mode(mode)
    s.set_host_checks(1)
    ref = s.solve(nodes, aims, 6)
    s.set_host_checks(0)
    a = torch.randn(size, size, device="cuda")
    torch.cuda.synchronize()
    b = a
    for _ in range(products):  # in front of the solve: from longer than it waits, to shorter (8192: about 8 ms each)
        b = a @ b * 1e-2
    got = s.solve(nodes, aims, 6)
    assert same(got, ref)
    assert same(s.solve(nodes, aims, 6), ref)


def test_captured(scene):
    import torch
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = arapgs.Context(0, stream=stream)
        nodes = T(scene["nodes"])
        aims = [T(S.frame_aims(scene["scene"], scene["nodes"], scene["blocks"], scene["types"], f))
                for f in (0.5, 0.2)]
        s = solver_of(c, scene)
        refs = [[t.clone() for t in s.solve(nodes, a, 6)] for a in aims]
        out = [torch.empty_like(refs[0][0]), torch.zeros_like(refs[0][1]), torch.zeros_like(refs[0][2])]
        target = aims[0].clone()
        s.solve(nodes, target, 6, x_out=out[0], energies=out[1], iters_done=out[2])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        s.solve(nodes, target, 6, x_out=out[0], energies=out[1], iters_done=out[2])
    for i in (0, 1, 0, 1):
        with torch.cuda.stream(stream):
            target.copy_(aims[i])
            g.replay()
        torch.cuda.synchronize()
        assert same(out, refs[i]), i
    del g
    s.close()
    c.close()
