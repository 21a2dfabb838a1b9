"""Farthest-point nodes and the K-nearest search at the sizes where their
kernels change (one wave, one and several workgroups, one launch a step; brute
force to cells, LDS above 64 KB), over spread, flat, clustered and far-off points, with
ties: bit-exact against the oracle."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def H(t):
    return t.detach().cpu().numpy()


def cloud(kind, n, rng):
    if kind == "box":
        p = rng.uniform(-1, 1, size=(n, 3))
    elif kind == "plane":
        p = rng.uniform(-1, 1, size=(n, 3)) * [1.0, 1.0, 0.0]
    elif kind == "line":
        p = rng.uniform(-1, 1, size=(n, 1)) * [1.0, 2.0, -0.5]
    elif kind == "clusters":
        p = rng.normal(size=(n, 3)) * 0.01 + rng.integers(0, 3, size=(n, 3)) * 4.0
    elif kind == "far":
        p = rng.uniform(-1, 1, size=(n, 3)) + [1000.0, -3000.0, 500.0]
    elif kind == "lattice":
        p = rng.integers(0, 12, size=(n, 3)) * 0.25
    else:  # one point
        p = np.tile([[0.5, -0.25, 3.0]], (n, 1))
    return p.astype(np.float32)


KINDS = ["box", "plane", "line", "clusters", "far", "lattice", "point"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n,m", [(1, 1), (63, 63), (64, 20), (65, 64), (4097, 300), (12288, 50), (12289, 400),
                                 (70000, 90)])
def test_fps_at_kernel_edges(ctx, kind, n, m):
    pos = cloud(kind, n, np.random.default_rng(n + m))
    assert np.array_equal(H(ctx.fps(T(pos), m)), O.fps(pos, m))


def test_fps_beyond_one_launch(ctx):
    """More points than the workgroups of the one-launch form hold."""
    pos = cloud("box", 3_200_001, np.random.default_rng(2))
    assert np.array_equal(H(ctx.fps(T(pos), 9)), O.fps(pos, 9))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,k", [(67, 1), (68, 1), (103, 4), (104, 4), (179, 8), (180, 8), (287, 12), (288, 12), (95, 8), (96, 8), (97, 1), (257, 12), (1500, 6), (2048, 8), (4096, 8), (5461, 4)])
def test_knn_at_kernel_edges(ctx, kind, m, k):
    rng = np.random.default_rng(m + k)
    nodes = cloud(kind, m, rng)
    span = nodes.max(0) - nodes.min(0) + 0.1
    q = np.concatenate([nodes[:200], nodes.mean(0) + span * rng.uniform(-0.9, 0.9, size=(1500, 3)),
                        nodes.mean(0) + 40 * span * rng.normal(size=(47, 3))]).astype(np.float32)
    ridx, rw = O.knn_weights(nodes, q, k)
    idx, w = ctx.knn(T(nodes), T(q), k)
    assert np.array_equal(ridx.astype(np.int64), H(idx).astype(np.int64))
    assert np.array_equal(rw.astype(np.float32), H(w), equal_nan=True)
    q[::7, 1] = np.inf
    q[::11, 0] = np.nan
    idx, _ = ctx.knn(T(nodes), T(q), k)   # no answer is defined for these: the others keep theirs
    fine = np.isfinite(q).all(1)
    assert np.array_equal(ridx.astype(np.int64)[fine], H(idx).astype(np.int64)[fine])


LAYOUTS = {"cube": (1, 1, 1), "plane": (1, 1, 0), "slab": (1, 1, 0.01), "line": (1, 0, 0), "thin": (1, 0.01, 0.01)}


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("m", [100, 2048])
@pytest.mark.parametrize("k", [1, 8])
def test_knn_away_from_the_nodes(ctx, layout, m, k):
    """Queries whose nearest nodes lie in a few cells, in many, and beyond what is
    searched by cells."""
    rng = np.random.default_rng(m + k)
    sides = np.array(LAYOUTS[layout])
    nodes = (rng.uniform(-1, 1, (m, 3)) * sides).astype(np.float32)
    q = np.concatenate([rng.uniform(-1, 1, (300, 3)) * sides + away * rng.normal(size=(300, 3))
                        for away in (0.01, 0.05, 0.3, 1.0, 10.0, 1e6)]).astype(np.float32)
    ridx, rw = O.knn_weights(nodes, q, k)
    idx, w = ctx.knn(T(nodes), T(q), k)
    assert np.array_equal(ridx.astype(np.int64), H(idx).astype(np.int64))
    assert np.array_equal(rw.astype(np.float32), H(w), equal_nan=True)


def knn_ms(ctx, nodes, q, k):
    import torch
    ctx.knn(nodes, q, k)
    times = []
    for _ in range(5):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        ctx.knn(nodes, q, k)
        e[1].record()
        torch.cuda.synchronize()
        times.append(e[0].elapsed_time(e[1]))
    return min(times)


@pytest.mark.parametrize("layout", ["cube", "plane", "line", "thin"])
def test_knn_away_costs_no_more_than_every_node(ctx, layout):
    """Searched by growing blocks of cells alone, queries away from a flat layout took
    40 to 500 times what queries among the nodes of a cube take; visiting every node
    takes about 3 times."""
    rng = np.random.default_rng(1)
    nodes = rng.uniform(-1, 1, (2048, 3))
    q = rng.uniform(-1, 1, (50000, 3))
    near = knn_ms(ctx, T(nodes.astype(np.float32)), T(q.astype(np.float32)), 8)
    sides = np.array(LAYOUTS[layout])
    far = (q * sides + 0.3 * rng.normal(size=q.shape)).astype(np.float32)
    away = knn_ms(ctx, T((nodes * sides).astype(np.float32)), T(far), 8)
    print(f"{layout}: among the nodes {near:.3f} ms, away {away:.3f} ms", flush=True)
    assert away <= 12 * near


AT = {"node": (0, 0, 0), "edge": (0.5, 0, 0), "face": (0.5, 0.5, 0), "centre": (0.5, 0.5, 0.5)}


def lattice(dims):
    side = 12 if dims == 3 else 45
    g = np.stack(np.meshgrid(*[np.arange(side)] * dims, indexing="ij"), -1).reshape(-1, dims)
    return np.concatenate([g, np.zeros((len(g), 3 - dims))], 1).astype(np.float32), side


def lattice_queries(dims, side, n, at, rng):
    q = rng.integers(1, side - 2, (n, 3)) + (np.array(AT[at]) if at else rng.random((n, 3)))
    return (q * ([1, 1, 1] if dims == 3 else [1, 1, 0])).astype(np.float32)


@pytest.mark.parametrize("dims", [2, 3])
@pytest.mark.parametrize("k", [1, 2, 4, 6, 8, 9, 12])
def test_knn_equal_distances(ctx, dims, k):
    """Up to 24 nodes at the K-th distance: within the short list of candidates, within
    the long one, and beyond both."""
    rng = np.random.default_rng(10 * dims + k)
    nodes, side = lattice(dims)
    nodes = nodes[rng.permutation(len(nodes))]
    q = np.concatenate([lattice_queries(dims, side, 400, at, rng) for at in AT])
    ridx, rw = O.knn_weights(nodes, q, k)
    idx, w = ctx.knn(T(nodes), T(q), k)
    assert np.array_equal(ridx.astype(np.int64), H(idx).astype(np.int64))
    assert np.array_equal(rw.astype(np.float32), H(w), equal_nan=True)


@pytest.mark.parametrize("dims,at,k", [(3, "node", 3), (3, "edge", 6), (3, "face", 8), (3, "centre", 4),
                                       (2, "edge", 8), (2, "face", 8)])
def test_knn_equal_distances_are_not_replayed(ctx, dims, at, k):
    """At most 16 nodes within the K-th distance: replayed one query at a time, these took
    70 to 350 times what queries without ties take; with the long list about twice."""
    rng = np.random.default_rng(3)
    nodes, side = lattice(dims)
    free = knn_ms(ctx, T(nodes), T(lattice_queries(dims, side, 100000, None, rng)), k)
    ties = knn_ms(ctx, T(nodes), T(lattice_queries(dims, side, 100000, at, rng)), k)
    print(f"{dims}D {at} k={k}: no ties {free:.3f} ms, ties {ties:.3f} ms", flush=True)
    assert ties <= 10 * free


def test_fps_workspace_does_not_grow_with_the_nodes():
    """Every point a node: the one-launch form's words once took 32 bytes a workgroup and
    step (29 MB here, 8 GB at 3M points and 1M nodes)."""
    import torch
    from arapgs_amd import arapgs
    n = 100_000
    pos = T(cloud("box", n, np.random.default_rng(4)))
    c = arapgs.Context(0)
    c.fps(pos, 2)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    idx = H(c.fps(pos, n))
    grown = before - torch.cuda.mem_get_info()[0]
    c.close()
    assert np.array_equal(np.sort(idx), np.arange(n))
    assert grown <= 8 << 20, grown


@pytest.mark.parametrize("kind", ["box", "lattice", "point"])
@pytest.mark.parametrize("n,m", [(20000, 60), (70000, 40)])
@pytest.mark.parametrize("polls", [0, 1, 3])
def test_fps_given_up(kind, n, m, polls):
    """Workgroups that look for each other's results a few times only give up, and the
    steps are taken one launch each (0: from the start)."""
    from arapgs_amd import arapgs
    pos = cloud(kind, n, np.random.default_rng(n + m))
    c = arapgs.Context(0)
    c.set_fps_polls(polls)
    ref = O.fps(pos, m)
    for _ in range(2):
        assert np.array_equal(H(c.fps(T(pos), m)), ref)
    c.set_fps_polls(50000)
    assert np.array_equal(H(c.fps(T(pos), m)), ref)
    with pytest.raises(arapgs.ArapgsError):
        c.set_fps_polls(-1)
    c.close()


@pytest.mark.parametrize("cus", [8, 64])
def test_fps_on_a_stream_of_few_cus(cus):
    """Nine workgroups that must run at once, on a stream with fewer CUs and with more."""
    import torch
    from arapgs_amd import arapgs
    pos = cloud("box", 100_000, np.random.default_rng(8))
    ref = O.fps(pos, 50)
    s = arapgs.CuStream(0, 0, cus)
    with torch.cuda.stream(s.torch):
        c = arapgs.Context(0, stream=s.torch)
        got = H(c.fps(T(pos), 50))
        c.close()
    torch.cuda.synchronize()
    s.close()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("m", [24, 25, 26])
def test_fps_around_the_one_launch_form(ctx, m):
    pos = cloud("box", 30000, np.random.default_rng(m))
    assert np.array_equal(H(ctx.fps(T(pos), m)), O.fps(pos, m))


def test_fps_of_few_nodes_needs_no_sort(ctx):
    """Two nodes of 100k points took 0.3 of the time of 128 while the points were sorted
    for them; one step takes a twentieth."""
    import time
    pos = T(cloud("box", 100_000, np.random.default_rng(6)))
    took = {}
    for m in (2, 128):
        ctx.fps(pos, m)
        times = []
        for _ in range(7):
            t0 = time.perf_counter()
            ctx.fps(pos, m)
            times.append(time.perf_counter() - t0)
        took[m] = min(times)
    print(f"2 nodes {took[2] * 1e6:.0f} us, 128 nodes {took[128] * 1e6:.0f} us", flush=True)
    assert took[2] <= 0.15 * took[128]


@pytest.mark.parametrize("m,k", [(41, 1), (42, 1), (151, 8), (152, 8), (291, 12), (292, 12)])
def test_knn_of_many_queries_at_kernel_edges(ctx, m, k):
    rng = np.random.default_rng(m)
    nodes = cloud("clusters", m, rng)
    q = (nodes[rng.integers(0, m, 300001)] + rng.normal(size=(300001, 3)) * 0.3).astype(np.float32)
    idx, w = ctx.knn(T(nodes), T(q), k)
    some = rng.integers(0, len(q), 4000)
    ridx, rw = O.knn_weights(nodes, q[some], k)
    assert np.array_equal(ridx.astype(np.int64), H(idx)[some].astype(np.int64))
    assert np.array_equal(rw.astype(np.float32), H(w)[some], equal_nan=True)
