"""The matrix-core density sample and its backward at cell-list lengths around
their tiles (32 and 16 Gaussians a step, 64 a batch), with the scalar and the
adaptive filter, against FP64 sums of the definition."""
import numpy as np
import pytest

from arapgs_amd import scenes as S

pytestmark = pytest.mark.gpu

COUNTS = (1, 2, 3, 4, 5, 12, 13, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 193, 260)


def T(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def H(t):
    return t.detach().cpu().numpy().astype(np.float64)


@pytest.fixture(scope="module")
def cells(ctx):
    """A grid (padding 0) with COUNTS[i] small Gaussians in the i-th of its occupied cells."""
    G, rng = 8, np.random.default_rng(3)
    corner = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]], np.float32)
    a7 = ctx.scene_aabb(T(corner), G)
    mn, step = a7[:3], a7[6]
    at = [(2 * (i // 9) + 1, 2 * (i // 3 % 3) + 1, 2 * (i % 3) + 1) for i in range(len(COUNTS))]
    pos = np.concatenate([mn + step * (np.array(c) + rng.uniform(0.35, 0.65, size=(n, 3)))
                          for c, n in zip(at, COUNTS)]).astype(np.float32)
    g = S.random_gaussians(rng, pos, log_scale_mean=np.log(0.03 * step), log_scale_std=0.2)
    g.sh = rng.uniform(0.5, 1.5, size=g.sh.shape).astype(np.float32)
    g.opacity = rng.uniform(0.3, 0.9, size=g.n).astype(np.float32)
    grid = ctx.grid_build(ctx.gaussian_aabbs(T(g.pos), T(g.rot), T(g.scale), T(g.opacity)), a7, G, padding=0)
    prefix, lst, valid, samples = grid.arrays()
    ends = prefix[valid]
    begs = np.concatenate([[0], ends[:-1]])
    assert tuple(ends - begs) == COUNTS
    return dict(g=g, grid=grid, samples=samples.astype(np.float64), lists=[lst[b:e] for b, e in zip(begs, ends)],
                lpf=float(np.float32((0.2 * step) ** 2)))


def fp64(c, L, dfeat=None, ddens=None):
    """Features and densities, and with the output gradients their VJP, cell by cell in FP64."""
    g = c["g"]
    q = g.rot.astype(np.float64)
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    w, x, y, z = q.T
    R = np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y), 2 * (x * y + w * z),
                  1 - 2 * (x * x + z * z), 2 * (y * z - w * x), 2 * (x * z - w * y), 2 * (y * z + w * x),
                  1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)
    Sg = np.einsum("nik,nk,njk->nij", R, g.scale.astype(np.float64) ** 2, R)
    feat, dens = [], []
    dmu, dsh, dop = np.zeros((g.n, 3)), np.zeros((g.n, 48)), np.zeros(g.n)
    dx = np.zeros_like(c["samples"])
    for v, ids in enumerate(c["lists"]):
        Q = np.linalg.inv(Sg[ids] + L[v])
        d = c["samples"][64 * v: 64 * v + 64, None] - g.pos[ids].astype(np.float64)
        Qd = np.einsum("nij,snj->sni", Q, d)
        ex = np.exp(-0.5 * (d * Qd).sum(-1))
        a = ex * g.opacity[ids]
        feat.append(a @ g.sh[ids].astype(np.float64))
        dens.append(a.sum(1))
        if dfeat is not None:
            df, dd = dfeat[64 * v: 64 * v + 64], ddens[64 * v: 64 * v + 64]
            da = df @ g.sh[ids].T.astype(np.float64) + dd[:, None]
            dsh[ids] += a.T @ df
            dop[ids] += (ex * da).sum(0)
            e = -(a * da)[..., None] * Qd
            dx[64 * v: 64 * v + 64] = e.sum(1)
            dmu[ids] -= e.sum(0)
    return np.concatenate(feat), np.concatenate(dens), dmu, dop, dsh, dx


def filters(c, ada):
    nv = c["grid"].n_valid
    if ada is None:
        return np.tile(c["lpf"] * np.eye(3), (nv, 1, 1))
    L = np.zeros((nv, 3, 3))
    for k, (i, j) in enumerate(((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2))):
        L[:, i, j] = L[:, j, i] = ada[:, k]
    return L


@pytest.mark.parametrize("ada", [False, True])
def test_density_at_tile_edges(ctx, cells, ada):
    """All terms are positive, so every value is within the sum of its rounding
    steps, relative: |exponent| <= 64 gives 64 x 2^-23, the sum of 260 terms at
    most 260 x 2^-24: 2.4e-5 (3e-5 asserted)."""
    g, grid = cells["g"], cells["grid"]
    if ada:
        x = cells["samples"]
        grid.set_ada_lpf(0.6, samples=T((x + 0.05 * np.sin(4.0 * x[:, [1, 2, 0]])).astype(np.float32)))
    feat, dens = grid.density(T(g.pos), T(g.rot), T(g.scale), T(g.opacity), T(g.sh), cells["lpf"])
    rf, rd, *_ = fp64(cells, filters(cells, grid.ada_lpf()))
    grid.set_ada_lpf(0.0)
    big = rd > 1e-30  # below: FP32 underflows
    ef = np.abs(H(feat) - rf)[big] / rf[big]
    ed = np.abs(H(dens) - rd)[big] / rd[big]
    print(f"density ada={ada}: max rel err features {ef.max():.2e}, densities {ed.max():.2e}", flush=True)
    assert ef.max() <= 3e-5 and ed.max() <= 3e-5


@pytest.mark.parametrize("ada", [False, True])
@pytest.mark.parametrize("which", ["both", "feat", "dens"])
def test_density_backward_at_tile_edges(ctx, cells, ada, which):
    """Each Gaussian's gradients against the FP64 VJP, relative to the sums of
    the absolute values of their terms (64 samples, one cell each: 64 x 2^-24
    for the sums, 64 x 2^-23 for the exponent, 48 x 2^-23 for the products with
    the output gradient: 1.7e-5; 4e-5 asserted)."""
    g, grid = cells["g"], cells["grid"]
    rng = np.random.default_rng(5)
    S = cells["samples"].shape[0]
    df = rng.normal(size=(S, 48)).astype(np.float32) if which != "dens" else None
    dd = rng.normal(size=S).astype(np.float32) if which != "feat" else None
    if ada:
        x = cells["samples"]
        grid.set_ada_lpf(0.6, samples=T((x + 0.05 * np.sin(4.0 * x[:, [1, 2, 0]])).astype(np.float32)))
    L = filters(cells, grid.ada_lpf())
    args = [T(g.pos), T(g.rot), T(g.scale), T(g.opacity), T(g.sh), cells["lpf"]]
    kw = dict(dfeat=None if df is None else T(df), dopac=None if dd is None else T(dd))
    out = grid.density_backward(*args, **kw, want_samples=True)
    again = grid.density_backward(*args, **kw)
    grid.set_ada_lpf(0.0)
    f = np.zeros((S, 48)) if df is None else df.astype(np.float64)
    o = np.zeros(S) if dd is None else dd.astype(np.float64)
    ref = fp64(cells, L, f, o)
    mag = fp64(cells, L, np.abs(f), np.abs(o))
    # with and without the sample gradients: two kernels, whose exponents are
    # associated differently (each within the bound above)
    for got in (out, again):
        worst = {}
        for name, i, r, m in (("dop", 3, ref[3], mag[3]), ("dsh", 4, ref[4], mag[4])):
            worst[name] = (np.abs(H(got[i]) - r) / (m + 1e-30)).max()
        # the position gradients' terms are signed by Q d: relative to the largest
        for name, i, r in (("dmu", 0, ref[2]), ("dx", 5, ref[5])):
            if i < len(got):
                worst[name] = np.abs(H(got[i]) - r).max() / np.abs(r).max()
        print(f"density backward ada={ada} {which}: {worst}", flush=True)
        assert max(worst.values()) <= 4e-5


def same_class(got, ref):
    """Infinities and NaN where the reference (as float) has them, with their signs."""
    with np.errstate(over="ignore"):
        ref = np.asarray(ref, np.float32).astype(np.float64)
    odd = ~np.isfinite(ref)
    return odd, np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got[odd & ~np.isnan(ref)],
                                                                                  ref[odd & ~np.isnan(ref)])


LARGE = [np.inf, -np.inf, 3.4e38, -1e25, np.nan]


@pytest.mark.parametrize("ada", [False, True])
def test_density_of_large_coefficients(ctx, cells, ada):
    """An infinite coefficient, one above bf16's largest value and one whose square
    overflows: the features are the FP32 sums (3e-5, as above), infinite or NaN only
    where those are."""
    g, grid = cells["g"], cells["grid"]
    sh = g.sh.copy()
    where = []
    for i, x in enumerate(LARGE):  # in cells of 5, 13, 17, 33 and 129 Gaussians, the last of them
        ids = cells["lists"][(4, 7, 9, 12, 18)[i]]
        sh[ids[-1], 5 * i + 1] = x
        where.append(ids[-1])
    if ada:
        x = cells["samples"]
        grid.set_ada_lpf(0.6, samples=T((x + 0.05 * np.sin(4.0 * x[:, [1, 2, 0]])).astype(np.float32)))
    feat, dens = grid.density(T(g.pos), T(g.rot), T(g.scale), T(g.opacity), T(sh), cells["lpf"])
    keep, g.sh = g.sh, sh
    rf, rd, *_ = fp64(cells, filters(cells, grid.ada_lpf()))
    g.sh = keep
    grid.set_ada_lpf(0.0)
    odd, fine = same_class(H(feat), rf)
    assert odd.any() and fine
    ok = ~odd & (rd[:, None] > 1e-30)
    assert (np.abs(H(feat)[ok] - rf[ok]) / np.abs(rf[ok])).max() <= 3e-5
    assert np.isfinite(H(dens)).all()


@pytest.mark.parametrize("ada", [False, True])
@pytest.mark.parametrize("what", ["sh", "dfeat", "dopac", "none"])
def test_density_backward_of_large_operands(ctx, cells, ada, what):
    """Large coefficients and output gradients in the VJP: infinite or NaN where the sums
    are, everything else as without them (4e-5, as above)."""
    g, grid = cells["g"], cells["grid"]
    rng = np.random.default_rng(6)
    S = cells["samples"].shape[0]
    df = rng.uniform(0.5, 1.0, size=(S, 48)).astype(np.float32)
    dd = rng.uniform(0.5, 1.0, size=S).astype(np.float32)
    sh = g.sh.copy()
    for i, x in enumerate(LARGE if what != "none" else []):
        cell = (4, 7, 9, 12, 18)[i]
        x = np.float32(x)
        if what == "sh":
            sh[cells["lists"][cell][-1], 5 * i + 1] = x
        elif what == "dfeat":
            sh[cells["lists"][cell], 5 * i + 1] = 0.5  # (FP32's products with it do not overflow)
            df[64 * cell + 10 + i, 5 * i + 1] = x
        else:
            dd[64 * cell + 10 + i] = x
    if ada:
        x = cells["samples"]
        grid.set_ada_lpf(0.6, samples=T((x + 0.05 * np.sin(4.0 * x[:, [1, 2, 0]])).astype(np.float32)))
    L = filters(cells, grid.ada_lpf())
    args = [T(g.pos), T(g.rot), T(g.scale), T(g.opacity), T(sh), cells["lpf"]]
    kw = dict(dfeat=T(df), dopac=T(dd))
    outs = [grid.density_backward(*args, **kw, want_samples=True), grid.density_backward(*args, **kw)]
    grid.set_ada_lpf(0.0)
    keep, g.sh = g.sh, sh
    with np.errstate(invalid="ignore", over="ignore"):
        ref = fp64(cells, L, df.astype(np.float64), dd.astype(np.float64))
    g.sh = keep

    def off(got, want, where):
        return np.abs(got[where] - want[where]), np.abs(want[where])

    # the Gaussians of the cells without a large operand, and all of dL/dSH: no sum there mixes the two
    clean = np.ones(g.n, bool)
    for cell in (4, 7, 9, 12, 18):
        clean[cells["lists"][cell]] = False
    if what == "none":
        clean[:] = True
    for got in outs:
        odd, fine = same_class(H(got[4]), ref[4])
        assert fine and odd.any() == (what == "dfeat")
        e, r = off(H(got[4]), ref[4], ~odd)
        assert (e / r).max() <= 4e-5
        odd, fine = same_class(H(got[3]), ref[3])
        assert fine and odd.any() == (what != "none")
        e, r = off(H(got[3]), ref[3], ~odd)
        assert (e / r).max() <= 4e-5
        e, r = off(H(got[0]), ref[2], clean)
        assert e.max() <= 4e-5 * r.max()
        if len(got) > 5:
            rows = np.repeat([(clean[ids]).all() for ids in cells["lists"]], 64)
            e, r = off(H(got[5]), ref[5], rows)
            assert e.max() <= 4e-5 * r.max()
