"""The six-point update in workgroups of 64 Gaussians (few of them) and of 256
(many): every Gaussian's results are the same bit for bit."""
import numpy as np
import pytest

from helpers import random_node_xf, table_from

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("cache", [True, False])
@pytest.mark.parametrize("k", [8, 6, 1])
def test_workgroup_size_does_not_change_results(ctx, k, cache):
    import torch
    rng = np.random.default_rng(k)
    n, m = 65536 + 65, 40  # the first size of the large workgroups, with a ragged last one
    nodes = rng.uniform(-1, 1, (m, 3)).astype(np.float32)
    rot9, t3 = random_node_xf(m, rng)
    table = table_from(nodes, rot9, t3)
    pos = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    rot = rng.normal(size=(n, 4)).astype(np.float32)
    rot /= np.linalg.norm(rot, axis=1, keepdims=True)
    scale = rng.uniform(0.01, 0.05, (n, 3)).astype(np.float32)
    sh = rng.normal(size=(n, 48)).astype(np.float32)
    idx = rng.integers(0, m, (n, 6, k)).astype(np.int32)
    w = rng.uniform(0.1, 1.0, (n, 6, k)).astype(np.float32)
    w /= w.sum(-1, keepdims=True)
    static = (rng.random(n) < 0.1).astype(np.uint8)
    ends = ctx.end_points(T(pos), T(rot), T(scale)).cpu().numpy()

    def run(c):
        out = [T(ends[:c]), T(pos[:c]), T(rot[:c]), T(scale[:c]), T(sh[:c])]
        ctx.six_point_update(T(table), T(idx[:c].reshape(-1, k)), T(w[:c].reshape(-1, k)), out[0], T(scale[:c]),
                             T(static[:c]), *out[1:])
        torch.cuda.synchronize()
        return [o.cpu().numpy() for o in out]

    ctx.set_node_cache(cache)
    try:
        want = run(n)
        assert all(np.isfinite(a).all() for a in want)
        for c in (1, 63, 64, 65, 1001, 65536):
            for a, b in zip(run(c), want):
                assert np.array_equal(a, b[:c])
    finally:
        ctx.set_node_cache(True)
