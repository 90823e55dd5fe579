"""The perception adjoint over every gathered row width, over more neighbours than the per-particle lists
and the recorded chunks hold, and over bins that keep several cells, against the CPU oracle."""
import numpy as np
import pytest

from burn_automata_amd import kernels as K
from burn_automata_amd.config import Boundary, HashGridConfig, HashGridMode, PerceptionOptions
from oracle import oracle as O
from tests.helpers import rel_err, to_np

pytestmark = pytest.mark.gpu
f32 = np.float32
# the oracle sums each particle's terms in 32 bits in another order: a few hundred terms of either
# sign, 1e-6 of the output's peak each way, with room for the moment inverse's conditioning
TOL = 1e-4

CASES = {  # dim, S, n, box side, eps, grid size, batch, (state grad, density grad, hybrid, position features)
    "w4": (2, 1, 70, 1.0, 0.25, 16, 1, (1, 1, 1, 0)),
    "w8": (3, 7, 150, 0.7, 0.25, 8, 2, (1, 0, 1, 1)),
    "w24": (2, 24, 130, 1.0, 0.2, 16, 1, (1, 1, 0, 0)),
    "w24_3d": (3, 19, 200, 0.7, 0.25, 8, 1, (1, 1, 1, 1)),
    "w32": (3, 32, 97, 0.6, 0.25, 8, 1, (1, 1, 1, 0)),
    "w32_2d": (2, 25, 65, 1.0, 0.25, 16, 3, (1, 0, 1, 0)),
    "no_gradients": (2, 9, 80, 1.0, 0.25, 16, 1, (0, 0, 0, 0)),
    "density_only": (3, 4, 80, 0.6, 0.25, 8, 1, (0, 1, 0, 0)),
    "lists_overflow": (2, 5, 500, 0.3, 0.2, 16, 1, (1, 1, 1, 0)),    # about 300 neighbours each
    "chunks_overflow": (2, 3, 1500, 0.6, 0.2, 16, 1, (1, 1, 1, 0)),  # 9 cells of 170: 27 chunks of 64
    "chunks_overflow_3d": (3, 3, 900, 0.3, 0.15, 4, 1, (1, 1, 1, 0)),
    "shared_bins": (2, 3, 300, 6.0, 0.5, 2, 1, (1, 1, 1, 0)),        # 12 x 12 cells in 2 x 2 bins
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_adjoint_shapes_match_the_oracle(ctx, name):
    dim, S, n, side, eps, gs, batch, (sg, dg, hyb, pf) = CASES[name]
    cfg = HashGridConfig(dim, Boundary.Clamped, HashGridMode.Particle, (gs, gs, gs if dim == 3 else 1), eps, 32)
    rng = np.random.default_rng(n + S)
    pos = np.zeros((batch * n, 4), f32)
    pos[:, :dim] = rng.uniform(-side / 2, side / 2, (batch * n, dim))
    st = rng.normal(0, 0.5, batch * n * S).astype(f32)
    opts = PerceptionOptions(state_grad=bool(sg), density_grad=bool(dg), eps0=eps, hybrid_state_gradient=bool(hyb),
                             log_norm_grad=True, log_norm_density_grad=True, position_features=bool(pf))
    fa = rng.normal(0, 0.1, batch * n * opts.feature_dims(S, dim)).astype(f32)
    want = O.perceive_adjoint_with_options(pos, st, batch, n, S, cfg, opts, fa)
    got = K.perceive_adjoint_with_options(pos, st, batch, n, S, cfg, opts, fa, ctx=ctx)
    es, ep = rel_err(got.state, want.state), rel_err(to_np(got.position), want.position)
    print(f"{name}: state {es:.2e}, position {ep:.2e}")
    assert es <= TOL and ep <= TOL
    again = K.perceive_adjoint_with_options(pos, st, batch, n, S, cfg, opts, fa, ctx=ctx)
    np.testing.assert_array_equal(to_np(again.state), to_np(got.state))
    np.testing.assert_array_equal(to_np(again.position), to_np(got.position))


@pytest.mark.parametrize("dim,S", [(2, 16), (3, 5)])
def test_nearly_coincident_particles(ctx, dim, S):
    """Pairs from exactly coincident to 1e-15 apart, next to the origin, the squares of whose distances are
    subnormal or vanish. Below 1.5e-17 the oracle's position terms overflow in 32 bits; its state adjoint does not."""
    cfg = HashGridConfig(dim, Boundary.Clamped, HashGridMode.Particle, (8, 8, 8 if dim == 3 else 1), 0.25, 32)
    rng = np.random.default_rng(S)
    gaps = [0.0, 1e-30, 2e-23, 5e-23, 3e-20, 1e-19, 1.2e-19, 5e-18, 1e-16, 1e-15]
    B, N = len(gaps), 8  # one system per pair: its particles at 0 and at the gap, and six others around them
    pos = np.zeros((B, N, 4), f32)
    pos[:, 2:, :dim] = rng.uniform(-0.2, 0.2, (B, N - 2, dim))
    pos[:, 1, 0] = gaps
    pos = pos.reshape(B * N, 4)
    st = rng.normal(0, 0.5, B * N * S).astype(f32)
    opts = PerceptionOptions(state_grad=True, density_grad=True, eps0=0.25, hybrid_state_gradient=True,
                             log_norm_grad=False, log_norm_density_grad=False, position_features=False)
    fa = rng.normal(0, 0.1, B * N * opts.feature_dims(S, dim)).astype(f32)
    want = O.perceive_adjoint_with_options(pos, st, B, N, S, cfg, opts, fa)
    got = K.perceive_adjoint_with_options(pos, st, B, N, S, cfg, opts, fa, ctx=ctx)
    ws, gs = np.asarray(want.state).reshape(B, -1), to_np(got.state).reshape(B, -1)
    wp, gp = np.asarray(want.position).reshape(B, -1), to_np(got.position).reshape(B, -1)
    assert np.isfinite(ws).all() and np.isfinite(gs).all() and np.isfinite(gp).all()
    for k in range(B):
        es = rel_err(gs[k], ws[k])
        ep = rel_err(gp[k], wp[k]) if np.isfinite(wp[k]).all() else 0.0
        print(f"gap {gaps[k]:.1e}: state {es:.2e}, position {ep:.2e}")
        assert es <= TOL and ep <= TOL


def test_more_particles_than_one_launch_takes(ctx):
    """Past 2^24 particles a block takes several of them: 4,097 copies of one system give its result 4,097 times."""
    import torch
    B, N, S = 4097, 4096, 1
    cfg = HashGridConfig(2, Boundary.Clamped, HashGridMode.Particle, (16, 16, 1), 0.05, 32)
    rng = np.random.default_rng(5)
    pos = np.zeros((N, 4), f32)
    pos[:, :2] = rng.uniform(-0.9, 0.9, (N, 2))
    st = rng.normal(0, 0.5, N * S).astype(f32)
    opts = PerceptionOptions(state_grad=True, density_grad=False, eps0=0.05, hybrid_state_gradient=False)
    fa = rng.normal(0, 0.1, N * opts.feature_dims(S, 2)).astype(f32)
    want = O.perceive_adjoint_with_options(pos, st, 1, N, S, cfg, opts, fa)
    many = lambda a: torch.from_numpy(a).cuda().reshape(1, -1).expand(B, -1).contiguous()  # noqa: E731
    got = K.perceive_adjoint_with_options(many(pos).reshape(B * N, 4), many(st), B, N, S, cfg, opts, many(fa), ctx=ctx)
    for g, w in ((got.state, want.state), (got.position, want.position)):
        g = g.reshape(B, -1)
        assert rel_err(to_np(g[0]), w) <= TOL and torch.equal(g, g[:1].expand(B, -1))
