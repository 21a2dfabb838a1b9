"""Cell lists at grid sizes around the 64 lanes of a row scan, of boxes from
one cell to the whole grid, built in one chunk and slab by slab, against the
oracle's (bit-exact)."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 700])
@pytest.mark.parametrize("G,chunk", [(1, 0), (5, 0), (63, 0), (64, 1), (65, 0), (65, 1), (130, 0)])
def test_cell_lists(ctx, G, chunk, n):
    import torch
    rng = np.random.default_rng(1000 * G + n)
    mn, step = np.array([-0.7, 0.1, -2.0], np.float32), np.float32(0.05)
    lo = mn + step * rng.uniform(-2.0, G + 1.0, size=(n, 3))   # some outside the grid
    size = step * np.where(rng.random((n, 1)) < 0.02, G * rng.random((n, 3)), 4.0 * rng.random((n, 3)))
    aabbs = np.concatenate([lo, lo + size], 1).astype(np.float32)
    a7 = np.concatenate([mn, mn + G * step, [step]]).astype(np.float32)
    ctx.set_grid_chunk(chunk)
    try:
        grid = ctx.grid_build(torch.from_numpy(aabbs).cuda(), a7, G, padding=1)
    finally:
        ctx.set_grid_chunk(0)
    prefix, lst, valid, _ = grid.arrays()
    rp, rl, rv, _ = O.grid_lists(aabbs, mn, step, G, padding=1)
    assert np.array_equal(prefix, rp) and np.array_equal(lst, rl) and np.array_equal(valid, rv)
    grid.close()


@pytest.mark.parametrize("chunk", [0, 1])
@pytest.mark.parametrize("G,n", [(1, 1024), (1, 1025), (5, 3000), (64, 40), (65, 40), (130, 6)])
def test_cell_lists_counted_from_corners(ctx, G, n, chunk):
    """More than 1024 pairs a cell, or 2^22 in all: the counts are prefix sums of the boxes' corners."""
    import torch
    rng = np.random.default_rng(G + n)
    mn, step = np.array([-0.7, 0.1, -2.0], np.float32), np.float32(0.05)
    lo = mn + step * G * rng.uniform(-0.5, 0.3, size=(n, 3))
    hi = mn + step * G * rng.uniform(0.7, 1.5, size=(n, 3))
    aabbs = np.concatenate([lo, hi], 1).astype(np.float32)
    a7 = np.concatenate([mn, mn + G * step, [step]]).astype(np.float32)
    ctx.set_grid_chunk(chunk)
    try:
        grid = ctx.grid_build(torch.from_numpy(aabbs).cuda(), a7, G, padding=0)
    finally:
        ctx.set_grid_chunk(0)
    prefix, lst, valid, _ = grid.arrays()
    rp, rl, rv, _ = O.grid_lists(aabbs, mn, step, G, padding=0)
    print(f"G={G} n={n}: {len(lst)} pairs", flush=True)
    assert (len(lst) > min(1 << 22, 1024 * G ** 3)) == (n != 1024)
    assert np.array_equal(prefix, rp) and np.array_equal(lst, rl) and np.array_equal(valid, rv)
    grid.close()
