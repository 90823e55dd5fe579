"""The splat and the projected render drawn on the matrix cores, at the edges of their tiles, groups, the
waves' shares of the items and item ranges, against the oracle; non-finite particles touch only their own footprint."""
import numpy as np
import pytest

from burn_automata_amd import kernels as K
from burn_automata_amd.config import RenderLossConfig, Splat2dConfig
from oracle import oracle as O
from tests.helpers import psnr, to_np

pytestmark = pytest.mark.gpu
f32 = np.float32
# The weights' exponent is evaluated by axis and the sums by matrix products: both sides round pixel
# coordinates (up to 2^-24 of the image size, times the weight's slope) and sums of a few hundred terms.
TOL = 1e-5


def _err(got, want):
    g, w = to_np(got).astype(np.float64), to_np(want).astype(np.float64).reshape(to_np(got).shape)
    return np.max(np.abs(g - w)) / max(np.max(np.abs(w)), 1e-30)


def _particles(n, seed, spread=1.0):
    rng = np.random.default_rng(seed)
    pos = np.zeros((n, 4), f32)
    pos[:, :3] = rng.uniform(-spread, spread, (n, 3))
    return pos, rng.random((n, 3)).astype(f32), rng.random(n).astype(f32), rng.uniform(0.5, 4.0, n).astype(f32)


@pytest.mark.parametrize("n,size,sigma,spread", [
    (1, 1, 0.4, 0.5), (3, 16, 1.0, 1.2), (500, 17, 2.0, 1.0), (8192, 64, 1.0, 1.0), (8193, 65, 0.7, 1.3), (20000, 300, 1.5, 1.0),
    (3000, 500, 0.05, 1.0), (900, 128, 9.0, 1.0), (4000, 1040, 2.0, 1.0), (9000, 40, 1.0, 0.02), (0, 33, 1.0, 1.0)])
def test_splat_matches_the_oracle(ctx, n, size, sigma, spread):
    pos, col, _, _ = _particles(n, size, spread)
    cfg = Splat2dConfig(image_size=size, sigma=sigma, pixel_size=2.0 / size)
    got = K.splat_particles_2d(pos, col, cfg, ctx=ctx)
    if n == 0:
        assert not to_np(got).any()
        return
    want = O.splat_particles_2d(pos, col, cfg)
    assert _err(got, want) <= TOL and psnr(got, to_np(want).reshape(to_np(got).shape)) >= 100
    np.testing.assert_array_equal(to_np(K.splat_particles_2d(pos, col, cfg, ctx=ctx)), to_np(got))


@pytest.mark.parametrize("batch,n,size,cols", [(5, 700, 48, 2), (64, 130, 128, 8), (7, 9000, 33, 3)])
def test_tiled_windows_match_single_ones(ctx, batch, n, size, cols):
    pos, col, _, _ = _particles(batch * n, batch)
    cfg = Splat2dConfig(image_size=size, sigma=1.2, pixel_size=2.0 / size)
    got = to_np(K.splat_particles_2d_tiled(pos, col, batch, n, cfg, cols, ctx=ctx))
    for b in range(batch):
        want = to_np(O.splat_particles_2d(pos[b * n:(b + 1) * n], col[b * n:(b + 1) * n], cfg)).reshape(size, size, 4)
        win = got[b // cols * size:(b // cols + 1) * size, b % cols * size:(b % cols + 1) * size]
        assert _err(win, want) <= TOL


@pytest.mark.parametrize("n,size,views", [(1, 5, (0,)), (1500, 64, (0, 1, 2, 3)), (9000, 65, (3,)), (2500, 200, (1, 2)),
                                          (700, 530, (0, 3))])
def test_render_matches_the_oracle(ctx, n, size, views):
    pos, col, op, sg = _particles(n, n, 1.1)
    cfg = RenderLossConfig(image_size=size)
    got = to_np(K.render_views(pos, col, op, sg, cfg, views, ctx=ctx))
    for k, v in enumerate(views):
        want = O.splat_projected(O.project_positions(v, pos, cfg.world_scale), col, op, sg, cfg)
        assert _err(got[k], want) <= TOL
    np.testing.assert_array_equal(to_np(K.render_views(pos, col, op, sg, cfg, views, ctx=ctx)), got)


def test_non_finite_values_stay_in_their_footprint(ctx):
    """A NaN or infinite colour reaches the pixels of its particle's footprint and no others; a particle at
    a NaN or infinite position is drawn as the oracle draws it."""
    pos, col, _, _ = _particles(300, 4)
    cfg = Splat2dConfig(image_size=96, sigma=0.8, pixel_size=2.0 / 96)
    col[7, 1] = np.nan
    col[100, 0] = np.inf
    col[200, 2] = -np.inf
    pos[30, 0] = np.nan
    pos[31, 1] = np.inf
    got = to_np(K.splat_particles_2d(pos, col, cfg, ctx=ctx))
    want = to_np(O.splat_particles_2d(pos, col, cfg)).reshape(got.shape)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isposinf(got), np.isposinf(want))
    np.testing.assert_array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    assert np.max(np.abs(got[fin] - want[fin])) <= TOL * np.max(np.abs(want[fin]))


def test_huge_finite_colours_stay_in_their_footprint(ctx):
    """Finite colours whose product with the particle's scale overflows, where the footprint is all but outside the
    image or falls between the pixels: finite in its own pixels, and nothing in any other."""
    pos, col, op, sg = _particles(60, 4, 0.9)
    size = 64
    px = lambda p: f32(2 * p / (size - 1) - 1)  # noqa: E731  (the inverse of the splat's pixel coordinates)
    pos[3, :2] = px(-3.6), px(size + 2.6)
    pos[4, :2] = px(20.0), px(-3.7)
    pos[5, :2] = px(size + 2.7), px(33.0)
    col[3], col[4, 1], col[5] = (1e31, 2e31, -1e31), 3e38, -3e38
    cfg = Splat2dConfig(image_size=size, sigma=0.8, pixel_size=2.0 / size)
    cfg_n = Splat2dConfig(image_size=size, sigma=0.1, pixel_size=2.0 / size)
    pos2, col2 = pos.copy(), col.copy()
    pos2[7, :2] = px(40.5), px(17.5)
    col2[7] = 1e32
    for p, c, cf in ((pos, col, cfg), (pos2, col2, cfg_n)):
        got = to_np(K.splat_particles_2d(p, c, cf, ctx=ctx))
        want = to_np(O.splat_particles_2d(p, c, cf)).reshape(got.shape)
        assert np.isfinite(want).all() and np.isfinite(got).all()
        for ch in range(4):
            g, w = got[..., ch].astype(np.float64), want[..., ch].astype(np.float64)
            np.testing.assert_allclose(g, w, rtol=2e-4, atol=1e-4)
    rc = RenderLossConfig(image_size=size)
    rpos, rcol = pos.copy(), col.copy()
    rpos[3, :2] = rc.world_scale * 1.13, -rc.world_scale * 1.13
    rcol[4], rcol[5] = 0.5, 0.5
    rcol[3] = 1e35
    got = to_np(K.render_views(rpos, rcol, op, np.full_like(sg, 0.9), rc, (0,), ctx=ctx))[0]
    want = O.splat_projected(O.project_positions(0, rpos, rc.world_scale), rcol, op, np.full_like(sg, 0.9), rc)
    want = to_np(want).reshape(got.shape)
    assert np.isfinite(want).all() and np.isfinite(got).all()
    np.testing.assert_allclose(got.astype(np.float64), want.astype(np.float64), rtol=2e-4, atol=1e-4)


def _splat64(pos, col, cfg):
    """The splat of a cloud in 64 bits, on the box of pixels it reaches: sum_p col_p scale_p e_p(y) e_p(x) with the
    32-bit pixel coordinates and sigma of the splat. Returns the box's first column and row and [y, x, 4]."""
    size, span = f32(cfg.image_size), f32(cfg.hi) - f32(cfg.lo)
    sigma = f32(cfg.sigma) * size * f32(cfg.pixel_size) / span
    r, t = max(1, int(np.ceil(f32(5) * sigma))), float(size * f32(cfg.pixel_size) / span)
    px = (pos[:, 0] - f32(cfg.lo)) / span * (size - f32(1))
    py = (size - f32(1)) - (pos[:, 1] - f32(cfg.lo)) / span * (size - f32(1))
    axes, at = [], []
    for p in (px, py):
        b = np.floor(p).astype(int)
        x = np.arange(max(0, b.min() - r), min(cfg.image_size - 1, b.max() + r) + 1)
        w = np.exp(-(x[None, :] - p[:, None].astype(np.float64)) ** 2 / (2 * float(sigma) ** 2))
        axes.append(w * (np.abs(x[None, :] - b[:, None]) <= r))
        at.append(x[0])
    wx, wy = axes
    scale = t * t / np.maximum(wx.sum(1) * wy.sum(1), 1e-8)
    v = np.concatenate([col.astype(np.float64), np.ones((len(col), 1))], 1) * scale[:, None]
    return at, np.stack([wy.T @ (wx * v[:, c:c + 1]) for c in range(4)], -1)


@pytest.mark.parametrize("n,size,spread,share", [
    (40000, 520, 0.02, 10000), (600000, 520, 0.01, 9400),  # groups of 2x2 tiles
    (6000, 1040, 0.01, 512), (600000, 1040, 0.01, 9400),   # of 4x4: a few ranges, and the most, whose lists are filled twice
    (9000, 2048, 0.04, 1200), (5000, 2033, 0.5, 5000)])
def test_crowded_splats(ctx, n, size, spread, share):
    """A cloud on a few tiles. Every 97th particle's colour is a thousand times the others', so a lost run of
    particles shows; a wave's sums take one rounding for four items, `share` of them at most."""
    pos, col, _, _ = _particles(n, size + n, spread)
    pos[:, 0] += f32(0.31)
    col[::97] *= 1000
    cfg = Splat2dConfig(image_size=size, sigma=1.0, pixel_size=2.0 / size)
    got = to_np(K.splat_particles_2d(pos, col, cfg, ctx=ctx)).reshape(size, size, 4)
    (x0, y0), want = _splat64(pos, col, cfg)
    box = got[y0:y0 + want.shape[0], x0:x0 + want.shape[1]].astype(np.float64)
    assert np.count_nonzero(got) == np.count_nonzero(box)
    for ch in range(4):
        e = np.max(np.abs(box[..., ch] - want[..., ch])) / np.max(np.abs(want[..., ch]))
        print(f"channel {ch}: {e:.2e}")
        assert e <= TOL + share / 4 * 2.0 ** -24
    for _ in range(2):  # the ranges' counters are left as they were found
        np.testing.assert_array_equal(to_np(K.splat_particles_2d(pos, col, cfg, ctx=ctx)).reshape(got.shape), got)


@pytest.mark.parametrize("n,size,views,spread", [(6000, 256, (0, 1, 2, 3), 0.03), (7000, 520, (0, 1, 2, 3), 0.05),
                                                 (5000, 530, (1,), 0.02), (3000, 1024, (3,), 0.3)])
def test_crowded_renders_match_the_oracle(ctx, n, size, views, spread):
    pos, col, op, sg = _particles(n, n, spread)
    pos[:, 0] -= f32(0.4)
    cfg = RenderLossConfig(image_size=size)
    got = to_np(K.render_views(pos, col, op, sg, cfg, views, ctx=ctx))
    for k, v in enumerate(views):
        want = O.splat_projected(O.project_positions(v, pos, cfg.world_scale), col, op, sg, cfg)
        assert _err(got[k], want) <= TOL
    np.testing.assert_array_equal(to_np(K.render_views(pos, col, op, sg, cfg, views, ctx=ctx)), got)


def test_crowded_windows(ctx):
    batch, n, size, cols = 4, 3000, 500, 2
    pos, col, _, _ = _particles(batch * n, 9, 0.02)
    pos[n:2 * n, :2] += f32(0.5)
    pos[3 * n:, 1] -= f32(0.98)
    cfg = Splat2dConfig(image_size=size, sigma=1.2, pixel_size=2.0 / size)
    got = to_np(K.splat_particles_2d_tiled(pos, col, batch, n, cfg, cols, ctx=ctx))
    for b in range(batch):
        want = to_np(O.splat_particles_2d(pos[b * n:(b + 1) * n], col[b * n:(b + 1) * n], cfg)).reshape(size, size, 4)
        win = got[b // cols * size:(b // cols + 1) * size, b % cols * size:(b % cols + 1) * size]
        assert _err(win, want) <= TOL


@pytest.mark.parametrize("size", [2032, 2033, 4096])  # 127 tiles an axis, 128 (rectangles in pairs of tiles), 256
@pytest.mark.parametrize("corner", [(-1, -1), (1, 1), (0.37, 1), (1, -0.2)])
def test_rectangles_of_wide_images(ctx, size, corner):
    pos, col, _, _ = _particles(300, size, 0.02)
    pos[:, :2] += np.asarray(corner, f32)
    cfg = Splat2dConfig(image_size=size, sigma=1.3, pixel_size=2.0 / size)
    got = to_np(K.splat_particles_2d(pos, col, cfg, ctx=ctx)).reshape(size, size, 4)
    (x0, y0), want = _splat64(pos, col, cfg)
    box = got[y0:y0 + want.shape[0], x0:x0 + want.shape[1]]
    assert np.count_nonzero(got) == np.count_nonzero(box)
    assert _err(box, want) <= TOL


def test_crowded_splat_replays_in_a_graph(ctx):
    """A captured drawing of crowded groups, replayed with eager drawings in between, equals the eager one."""
    import torch
    pos, col, _, _ = _particles(20000, 3, 0.02)
    pos, col = torch.from_numpy(pos).cuda(), torch.from_numpy(col).cuda()
    other = [torch.from_numpy(a).cuda() for a in _particles(9000, 5, 0.05)[:2]]
    cfg = Splat2dConfig(image_size=600, sigma=1.0, pixel_size=2.0 / 600)
    want = K.splat_particles_2d(pos, col, cfg, ctx=ctx).clone()
    want_other = K.splat_particles_2d(*other, cfg, ctx=ctx).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    home = torch.cuda.current_stream().cuda_stream
    try:
        with torch.cuda.graph(graph):
            ctx.set_stream(torch.cuda.current_stream().cuda_stream)
            got = K.splat_particles_2d(pos, col, cfg, ctx=ctx)
    finally:
        ctx.set_stream(home)
    for _ in range(3):
        got.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        assert torch.equal(K.splat_particles_2d(*other, cfg, ctx=ctx), want_other)
