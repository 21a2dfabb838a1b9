"""The realignment's gradients (its sign kernel, cells merged) against the density
VJP of the same output gradients (one cell at a time), over grids of odd and even
edge, lists from one entry to several merge windows, lists that share all, most
or none of their entries, and cells left out as static.

Adam's first step with a huge epsilon moves a raw parameter by lr / eps times its
gradient, so the gradient can be read off the step."""
import numpy as np
import pytest

from arapgs_amd import arapgs
from arapgs_amd import scenes as S

pytestmark = pytest.mark.gpu


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def H(t):
    return t.detach().cpu().numpy().astype(np.float64)


# n, G, Gaussian size in cells, share of the Gaussians that move (None: all)
@pytest.mark.parametrize("n,G,size,moved", [
    (1, 1, 0.1, None), (1, 8, 0.5, None), (15, 2, 2.0, None), (17, 3, 2.0, None),
    (511, 2, 2.0, None), (512, 2, 2.0, None), (513, 3, 2.0, None), (1025, 3, 3.0, None),
    (2600, 4, 3.0, None),    # every cell lists nearly all: several windows
    (4000, 16, 0.05, None),  # lists share little
    (6000, 13, 0.4, None), (6000, 12, 0.4, 0.02),
])
@pytest.mark.parametrize("ada", [False, True])
def test_gradients_match_the_density_vjp(ctx, n, G, size, moved, ada):
    """dL/dSH: relative to the sum of the absolute values of its terms (|exponent|
    <= 64 gives 64 x 2^-23, sums of up to 64 x 64 terms in blocks of 64 with
    atomic adds of up to 64 cells (64 + 64) x 2^-24: 1.6e-5, on either side:
    4e-5 asserted). The others' terms change sign: relative to the largest."""
    import torch
    rng = np.random.default_rng(n + G)
    corner = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]], np.float32)
    a7 = ctx.scene_aabb(T(corner), G)
    mn, step = np.asarray(a7[:3]), float(a7[6])
    pos = (mn + step * G * rng.uniform(0.02, 0.98, (n, 3))).astype(np.float32)
    g = S.random_gaussians(rng, pos, log_scale_mean=np.log(size * step / 3), log_scale_std=0.4)
    g.opacity = rng.uniform(0.3, 0.9, size=g.n).astype(np.float32)
    p = [T(g.pos), T(g.rot), T(np.log(g.scale).astype(np.float32)),
         T(np.log(g.opacity / (1 - g.opacity)).astype(np.float32)), T(g.sh)]
    scale, op = torch.exp(p[2]), torch.sigmoid(p[3])
    grid = ctx.grid_build(ctx.gaussian_aabbs(p[0], p[1], scale, op), a7, G, padding=0)
    prefix, lst, valid, samples = grid.arrays()
    lpf = float(np.float32((0.2 * step) ** 2))
    if ada:
        grid.set_ada_lpf(0.6, samples=T((samples + 0.02 * step * np.sin(9.0 * samples[:, [1, 2, 0]])).astype(np.float32)))
    feat, dens = grid.density(p[0], p[1], scale, op, p[4], lpf)
    # aims above, below and at the values
    sf, sd = rng.integers(-1, 2, feat.shape), rng.integers(-1, 2, dens.shape)
    w = 0.3
    df, dd = sf.astype(np.float32), (w * sd).astype(np.float32)
    r = arapgs.Realign(ctx, grid, n, lr_pos=1e20, lr_rot=1e20, lr_scale=1e20, lr_opacity=1e20, lr_sh=1e20, eps=1e12,
                       w_density=w)
    if moved is not None:
        mv = (rng.random(n) < moved).astype(np.uint8)
        mvt = T(mv)
        r.set_options(moved=mvt)
        static = np.array([not mv[lst[(prefix[c - 1] if c else 0):prefix[c]]].any() for c in valid])
        assert static.any() and not static.all()
        df[np.repeat(static, 64)] = 0
        dd[np.repeat(static, 64)] = 0
    loss = torch.zeros(1, dtype=torch.float64, device="cuda")
    ref = grid.density_backward(p[0], p[1], scale, op, p[4], lpf, dfeat=T(df), dopac=T(dd), samples=T(samples))
    mag = grid.density_backward(p[0], p[1], scale, op, p[4], lpf, dfeat=T(np.abs(df)), dopac=T(np.abs(dd)),
                                samples=T(samples))
    ref = [H(ref[0]), H(ref[1]), H(ref[2] * scale), H(ref[3] * op * (1 - op)), H(ref[4])]
    r.step(T(samples), feat - T(1e3 * sf.astype(np.float32)), dens - T(1e3 * sd.astype(np.float32)), lpf, *p, loss=loss)
    torch.cuda.synchronize()
    grid.set_ada_lpf(0.0)
    r.close()
    want = 1e3 * (np.abs(sf).sum() + w * np.abs(sd).sum())
    assert abs(float(loss) - want) <= 1e-4 * want  # the aims are rounded to 2^-24 of 1e3
    got = [H(x) / -1e8 for x in p]
    sel = np.ones(n, bool) if moved is None else mv.astype(bool)
    worst = {}
    for name, a, b in zip(("pos", "rot", "scale", "opacity"), got, ref):
        worst[name] = np.abs(a - b)[sel].max() / max(np.abs(b).max(), 1e-20)
    worst["sh"] = (np.abs(got[4] - ref[4])[sel] / (H(mag[4])[sel] + 1e-3 * H(mag[4]).max())).max()
    print(f"n={n} G={G} size={size} ada={ada} moved={moved}: {worst}", flush=True)
    assert max(worst.values()) <= 4e-5


@pytest.mark.parametrize("special", ["coefficient", "weight", "none"])
def test_gradients_of_large_operands(ctx, special):
    """An infinite SH coefficient, or a density weight that is not split: the gradients are
    those of the density VJP (4e-5 as above), and not finite only where those are not."""
    import torch
    n, G = 700, 5
    rng = np.random.default_rng(12)
    corner = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]], np.float32)
    a7 = ctx.scene_aabb(T(corner), G)
    mn, step = np.asarray(a7[:3]), float(a7[6])
    pos = (mn + step * G * rng.uniform(0.02, 0.98, (n, 3))).astype(np.float32)
    g = S.random_gaussians(rng, pos, log_scale_mean=np.log(step / 3), log_scale_std=0.4)
    g.opacity = rng.uniform(0.3, 0.9, size=g.n).astype(np.float32)
    p = [T(g.pos), T(g.rot), T(np.log(g.scale).astype(np.float32)),
         T(np.log(g.opacity / (1 - g.opacity)).astype(np.float32)), T(g.sh)]
    scale, op = torch.exp(p[2]), torch.sigmoid(p[3])
    grid = ctx.grid_build(ctx.gaussian_aabbs(p[0], p[1], scale, op), a7, G, padding=0)
    samples = grid.arrays()[3]
    lpf = float(np.float32((0.2 * step) ** 2))
    feat, dens = grid.density(p[0], p[1], scale, op, p[4], lpf)
    # no aim at the value itself: cells with an infinity are summed in another order
    sf, sd = 2 * rng.integers(0, 2, feat.shape) - 1, 2 * rng.integers(0, 2, dens.shape) - 1
    w, k = (2.0 ** 61 if special == "weight" else 0.3), 7
    if special == "coefficient":
        p[4][100, k] = np.inf
        touched = ~torch.isfinite(grid.density(p[0], p[1], scale, op, p[4], lpf)[0]).cpu().numpy()
        sf[touched] = 1  # the differences are infinite
    df, dd = sf.astype(np.float32), (w * sd).astype(np.float32)
    ref = grid.density_backward(p[0], p[1], scale, op, p[4], lpf, dfeat=T(df), dopac=T(dd), samples=T(samples))
    ref = [H(ref[0]), H(ref[1]), H(ref[2] * scale), H(ref[3] * op * (1 - op)), H(ref[4])]
    r = arapgs.Realign(ctx, grid, n, lr_pos=1e20, lr_rot=1e20, lr_scale=1e20, lr_opacity=1e20, lr_sh=1e20, eps=1e12,
                       w_density=w)
    before = [H(x) for x in p]
    r.step(T(samples), feat - T(1e3 * sf.astype(np.float32)), dens - T(1e3 * sd.astype(np.float32)), lpf, *p)
    torch.cuda.synchronize()
    r.close()
    for name, a, b0, b in zip(("pos", "rot", "scale", "opacity", "sh"), p, before, ref):
        with np.errstate(invalid="ignore"):  # infinite before and after
            step_, fine = H(a) - b0, np.isfinite(b)
        if special == "weight" and name != "sh":
            # the gradients' squares overflow Adam's second moment, or their size its epsilon: the signs are left
            if name == "opacity":
                large = np.abs(b) > 1e-3 * np.abs(b).max()
                assert np.array_equal(np.sign(step_[large]), -np.sign(b[large]))
            continue
        if name == "sh" and special == "coefficient":
            fine[100, k] = False  # minus anything, it stays infinite
        assert np.isfinite(step_)[fine].all(), name
        assert name == "sh" or not np.isfinite(step_)[~fine].any(), name
        assert special == "coefficient" or fine.all()
        got = (step_ if name != "sh" else H(a)) / -1e8
        err = np.abs(got - b)[fine].max() / np.abs(b[fine]).max()
        print(f"{special} {name}: {err:.2e}, {int((~fine).sum())} not finite", flush=True)
        assert err <= 4e-5


def test_a_cell_whose_filter_leaves_no_inverse(ctx):
    """Two cells that are merged, and the second one's own filter is zero: a Gaussian
    without extent, which only the first lists, has no inverse there and keeps the
    gradients of its own cell."""
    import torch
    G, rng = 4, np.random.default_rng(3)
    corner = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]], np.float32)
    a7 = ctx.scene_aabb(T(corner), G)
    mn, step = np.asarray(a7[:3]), float(a7[6])
    at = np.repeat([[1, 1, 0], [1, 1, 1]], 20, axis=0)
    pos = (mn + step * (at + rng.uniform(0.4, 0.6, (40, 3)))).astype(np.float32)
    g = S.random_gaussians(rng, pos, log_scale_mean=np.log(0.03 * step), log_scale_std=0.1)
    g.opacity = rng.uniform(0.3, 0.9, size=g.n).astype(np.float32)
    ls = np.log(g.scale).astype(np.float32)
    ls[:5] = -np.inf
    p = [T(g.pos), T(g.rot), T(ls), T(np.log(g.opacity / (1 - g.opacity)).astype(np.float32)), T(g.sh)]
    scale, op = torch.exp(p[2]), torch.sigmoid(p[3])
    grid = ctx.grid_build(ctx.gaussian_aabbs(p[0], p[1], scale, op), a7, G, padding=0)
    prefix, lst, valid, samples = grid.arrays()
    assert len(valid) == 2 and valid[1] == valid[0] + 1 and valid[0] % 2 == 0
    moved = samples.copy()
    moved[64:] = samples[64]  # the second cell's samples in one place
    grid.set_ada_lpf(0.6, samples=T(moved))
    assert np.abs(grid.ada_lpf()[0]).max() > 0 and np.abs(grid.ada_lpf()[1]).max() == 0
    feat, dens = grid.density(p[0], p[1], scale, op, p[4], 0.0)
    sf, sd = rng.integers(-1, 2, feat.shape), rng.integers(-1, 2, dens.shape)
    w = 0.3
    ref = grid.density_backward(p[0], p[1], scale, op, p[4], 0.0, dfeat=T(sf.astype(np.float32)),
                                dopac=T((w * sd).astype(np.float32)), samples=T(samples))
    r = arapgs.Realign(ctx, grid, g.n, lr_pos=1e20, lr_rot=1e20, lr_scale=1e20, lr_opacity=1e20, lr_sh=1e20, eps=1e12,
                       w_density=w)
    r.step(T(samples), feat - T(1e3 * sf.astype(np.float32)), dens - T(1e3 * sd.astype(np.float32)), 0.0, *p)
    torch.cuda.synchronize()
    grid.set_ada_lpf(0.0)
    r.close()
    for name, a, b in (("pos", p[0], ref[0]), ("sh", p[4], ref[4])):
        a, b = H(a) / -1e8, H(b)
        assert np.isfinite(b).all(), name
        assert np.isfinite(a).all(), name
        assert np.abs(a - b).max() <= 4e-5 * np.abs(b).max(), name
