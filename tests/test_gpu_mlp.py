"""The update MLP on explicit rows and the two-kernel step, bit for bit against the oracle at the edges
of its tiles: 16 rows per block, 64 hidden units per wave, chunks of 128 or 256 units, output groups of
16, feature counts that are not a multiple of four."""
import numpy as np
import pytest

from burn_automata_amd import synthetic as syn
from burn_automata_amd.config import Boundary, HashGridConfig, HashGridMode, NpaConfig
from burn_automata_amd.model import NpaModel
from helpers import to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu
f32 = np.float32


def _weights(m, seed):
    rng = np.random.default_rng(seed)
    F, H, Od = m.perception_dims(), m.hidden_dims, m.update_dims()
    w = {"w1": rng.normal(size=H * F), "b1": rng.normal(size=H), "w2": rng.normal(size=Od * H), "b2": rng.normal(size=Od)}
    return {k: (0.3 * v).astype(f32) for k, v in w.items()}


@pytest.mark.parametrize("rows,d,S,H,dgrad", [
    (1, 2, 16, 128, True), (15, 2, 16, 128, False), (16, 3, 24, 256, True), (17, 2, 1, 1, False), (33, 3, 32, 300, True),
    (31, 2, 13, 64, True), (40, 3, 29, 65, False), (5, 2, 4, 129, True), (64, 2, 32, 513, True), (18, 3, 5, 63, False)])
def test_mlp_forward_bit_exact(ctx, rows, d, S, H, dgrad):
    m = NpaConfig(spatial_dims=d, state_dims=S, hidden_dims=H, density_grad=dgrad)
    w = _weights(m, rows)
    rng = np.random.default_rng(rows + H)
    feats = rng.normal(size=(rows, m.perception_dims())).astype(f32)
    feats.reshape(-1)[::7] *= f32(1e-30)   # denormal products
    feats.reshape(-1)[::11] = f32(-0.0)
    feats.reshape(-1)[::13] *= f32(1e6)
    want_dx, want_ds = O.forward_from_features_with_eps(m, w, feats, 0.1)
    dx, ds = NpaModel(m, w).forward_from_features_with_eps(feats, 0.1, ctx=ctx)
    np.testing.assert_array_equal(to_np(dx), np.asarray(want_dx).reshape(rows, 4))
    np.testing.assert_array_equal(to_np(ds), np.asarray(want_ds).reshape(rows, S))


@pytest.mark.parametrize("rows,d,S,H,sgrad,dgrad", [
    (16385, 2, 1, 16, True, True), (16448, 2, 16, 4, True, True), (16400, 3, 8, 7, True, False), (20001, 3, 13, 4, True, True),
    (16449, 2, 32, 4, False, False), (16385, 3, 1, 1, False, False), (17000, 2, 4, 16, True, True)])
def test_narrow_networks_bit_exact(ctx, rows, d, S, H, sgrad, dgrad):
    """A thread per row: at most 400 products a row, more than 16,384 rows, feature counts on both sides of 64."""
    m = NpaConfig(spatial_dims=d, state_dims=S, hidden_dims=H, state_grad=sgrad, density_grad=dgrad)
    F = m.perception_dims()
    assert F <= 72 and (F + m.update_dims()) * H <= 400
    w = _weights(m, rows)
    feats = np.random.default_rng(rows + H).normal(size=(rows, F)).astype(f32)
    want_dx, want_ds = O.forward_from_features_with_eps(m, w, feats, 0.1)
    dx, ds = NpaModel(m, w).forward_from_features_with_eps(feats, 0.1, ctx=ctx)
    np.testing.assert_array_equal(to_np(dx), np.asarray(want_dx).reshape(rows, 4))
    np.testing.assert_array_equal(to_np(ds), np.asarray(want_ds).reshape(rows, S))


@pytest.mark.parametrize("d,S,H,n,periodic", [(2, 16, 256, 333, False), (2, 8, 129, 65, True), (3, 24, 256, 500, False),
                                              (3, 32, 300, 47, False), (2, 5, 1, 15, False)])
def test_two_kernel_step_bit_exact(ctx, d, S, H, n, periodic):
    m = NpaConfig(spatial_dims=d, state_dims=S, hidden_dims=H, density_grad=d == 2)
    g = HashGridConfig(d, Boundary.Periodic, HashGridMode.Grid, (10, 10, 10)[:d] + (1,) * (3 - d), 0.2, 32) if periodic \
        else HashGridConfig(d, Boundary.Clamped, HashGridMode.Particle, (16, 16, 16), 0.1, 32)
    w = _weights(m, n)
    pos = syn.uniform_disk(n, 3, 0.8) if d == 2 else syn.uniform_ball(n, 3, 0.4)
    st = syn.normal_states(n, S, 3)
    mask = (np.random.default_rng(1).random(n) < 0.6).astype(f32)
    want = O.step(m, w, pos, st, 1, n, g, 1.0, mask)
    got = NpaModel(m, w).step(pos, st, 1, n, g, 1.0, update_mask=mask, ctx=ctx)
    np.testing.assert_array_equal(to_np(got.next_positions), want.next_positions)
    np.testing.assert_array_equal(to_np(got.next_states), want.next_states)


@pytest.mark.parametrize("d,S,H", [(2, 16, 128), (3, 24, 256), (2, 5, 65)])
@pytest.mark.parametrize("scale,w2", [(1e-37, 0.3), (3e-39, 0.3), (3e-39, 1e-6), (1e-42, 0.3)])
def test_subnormal_products_bit_exact(ctx, d, S, H, scale, w2):
    """Without biases: features, products and hidden units below the smallest normal number keep their bits."""
    m = NpaConfig(spatial_dims=d, state_dims=S, hidden_dims=H)
    w = _weights(m, H)
    w["b1"], w["b2"], w["w2"] = 0 * w["b1"], 0 * w["b2"], w["w2"] * f32(w2 / 0.3)
    feats = (np.random.default_rng(S).normal(size=(40, m.perception_dims())) * scale).astype(f32)
    want_dx, want_ds = O.forward_from_features_with_eps(m, w, feats, 0.1)
    dx, ds = NpaModel(m, w).forward_from_features_with_eps(feats, 0.1, ctx=ctx)
    assert np.count_nonzero(want_ds)
    np.testing.assert_array_equal(to_np(dx), np.asarray(want_dx).reshape(40, 4))
    np.testing.assert_array_equal(to_np(ds), np.asarray(want_ds).reshape(40, S))


def test_more_rows_than_one_launch_takes(ctx):
    """Rows past 2^26 go to another launch: the same results as the same rows of a short call."""
    import torch
    m = NpaConfig(spatial_dims=2, state_dims=1, hidden_dims=130, state_grad=False, density_grad=False)
    mod = NpaModel(m, _weights(m, 3))
    F, short, rows = m.perception_dims(), 4001, (1 << 26) + 37
    feats = torch.randn(short, F, generator=torch.Generator().manual_seed(1)).cuda()
    dx, ds = mod.forward_from_features_with_eps(feats.repeat(rows // short + 1, 1)[:rows], 0.1, ctx=ctx)
    want_dx, want_ds = mod.forward_from_features_with_eps(feats, 0.1, ctx=ctx)
    for got, want in ((dx.reshape(rows, 4), want_dx.reshape(short, 4)), (ds.reshape(rows, 1), want_ds.reshape(short, 1))):
        for first in (0, rows // short * short - 3 * short, rows // short * short):
            n = min(short, rows - first)
            assert torch.equal(got[first:first + n], want[:n])
