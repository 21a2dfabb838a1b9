"""Tile lists of a render against the oracle's, bit for bit: the records by depth,
their tiles sorted by id, and the ranges.

The sizes are where the path turns: one tile, one column of tiles, tile ids of 8
and 9 bits (one pass of the sort or two), exactly 2^16 tiles and more (16-bit tile
ids or the 32-bit keys), no visible record, one instance, equal depths (record
order), rectangles of more tiles than a workgroup sorts, and instance counts on
both sides of the workgroup shapes.
"""
import numpy as np
import pytest

import oracle as O
from arapgs_amd import scenes as S

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def gaussians(n, size, ties):
    rng = np.random.default_rng(n + 7)
    pos = rng.uniform(-1.0, 1.0, (n, 3)).astype(np.float32)
    if ties:
        pos = pos[rng.integers(0, max(n // 16, 1), n)]  # 16 records a depth
    sh = rng.normal(0.0, 0.2, (n, 48)).astype(np.float32)
    scale = (size * rng.uniform(0.5, 1.5, (n, 3))).astype(np.float32)
    rot = rng.normal(size=(n, 4)).astype(np.float32)
    rot /= np.linalg.norm(rot, axis=1, keepdims=True)
    return pos, sh, rng.uniform(0.01, 0.3, n).astype(np.float32), scale, rot


# n, size, W, H, tile, views, equal depths
@pytest.mark.parametrize("n,size,W,H,tile,V,ties", [
    (1, 0.01, 16, 16, 16, 1, False),        # one tile, one pass of one-bit ids
    (300, 0.05, 16, 500, 16, 1, False),     # one column
    (500, 0.05, 256, 256, 16, 1, True),     # 256 tiles: 8 bits
    (500, 0.05, 256, 257, 16, 1, True),     # 272 tiles: 9 bits
    (3000, 0.02, 333, 217, 8, 3, True),     # several views, 3402 tiles
    (40, 3.0, 1600, 1200, 16, 1, False),    # every record covers all 7500 tiles: more than a workgroup's 2048
    (400, 3.0, 1600, 1200, 16, 1, False),   # the same with 3M instances
    (2400, 3.0, 1600, 1200, 16, 1, False),  # with the larger workgroups (18M instances)
    (300000, 0.002, 320, 180, 16, 8, True),  # 2.4M records: the larger workgroups for them
    (30000, 0.02, 2048, 2048, 8, 1, False),  # 65,536 tiles
    (3000, 0.02, 2048, 2056, 8, 1, True),   # 65,792 tiles: 32-bit keys
    (40, 3.0, 524288, 8, 8, 1, False),      # 65,536 tiles in one row: a width of 2^16
    (40, 3.0, 524280, 8, 8, 1, False),      # 65,535 of them
    (60000, 0.004, 640, 360, 16, 8, False),  # 480,000 records
    (90000, 0.004, 640, 360, 16, 8, True),  # 720,000: the records' counts are scanned by a launch of their own
])
def test_tile_lists_match_oracle(ctx, n, size, W, H, tile, V, ties):
    import torch
    pos, sh, op, scale, rot = gaussians(n, size, ties)
    cams = [S.look_at_camera((0.4 * v, -4.0 + 0.3 * v, 0.8), (0.0, 0.0, 0.0), 50.0, W, H) for v in range(V)]
    if W > 100000:  # one row: the covariances as a camera of this opening has them, so that they span it
        cams[0].tanfovx = 0.4
    bg = np.array([0.1, 0.2, 0.3], np.float32)
    nt = ((W + tile - 1) // tile) * ((H + tile - 1) // tile)
    keys, vals, ranges, at = [], [], [], 0
    for v, c in enumerate(cams):
        r = O.raster(pos, sh, op, scale, rot, c.view, c.proj, c.campos, c.tanfovx, c.tanfovy, W, H, bg, tile=tile)
        keys.append(r["keys"] + (np.uint64(v * nt) << np.uint64(32)))
        vals.append(r["vals"] + np.uint32(v * n))
        filled = r["ranges"][:, 1] > r["ranges"][:, 0]
        ranges.append(np.where(filled[:, None], r["ranges"] + at, 0))
        at += len(r["keys"])
    outs = [torch.empty((3, H, W), device="cuda") for _ in cams]
    cd = [dict(view=T(c.view), proj=T(c.proj), campos=T(c.campos), tx=c.tanfovx, ty=c.tanfovy) for c in cams]
    got = ctx.render_views(T(pos), T(sh), T(op), T(scale), T(rot), cd, W, H, T(bg), outs, tile=tile)
    assert got == at > 0
    k, x, rg = ctx.render_debug(at, nt * V)
    assert np.array_equal(x, np.concatenate(vals))
    assert np.array_equal(k, np.concatenate(keys))
    assert np.array_equal(rg.astype(np.int64), np.concatenate(ranges).astype(np.int64))


def test_no_visible_record(ctx):
    pos, sh, op, scale, rot = gaussians(100, 0.05, False)
    pos[:, 1] -= 40.0  # behind the camera
    W, H = 300, 200
    cam = S.look_at_camera((0.0, -4.0, 0.8), (0.0, 0.0, 0.0), 50.0, W, H)
    bg = np.array([0.1, 0.2, 0.3], np.float32)
    out = ctx.render(T(pos), T(sh), T(op), T(scale), T(rot), T(cam.view), T(cam.proj), T(cam.campos), cam.tanfovx,
                     cam.tanfovy, W, H, T(bg))
    assert out["num_rendered"] == 0
    assert np.array_equal(out["image"].cpu().numpy(), np.broadcast_to(bg[:, None, None], (3, H, W)))
