"""The fused update with the density gradient (the presets' option set), clamped and periodic, 2D and 3D,
in four-wave blocks (up to four items of four particles per CU) and sixteen-wave blocks, bit for bit
against the oracle; list and chunk capacities are passed in the crowded cases."""
import numpy as np
import pytest

from burn_automata_amd import synthetic as syn
from burn_automata_amd.config import Boundary, HashGridConfig, HashGridMode, NpaConfig
from burn_automata_amd.model import NpaModel
from oracle import oracle as O
from tests.helpers import to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,periodic,S,n,eps,side", [
    (2, False, 16, 1, 0.1, 0.8), (2, False, 13, 15, 0.1, 0.3), (2, False, 16, 1001, 0.1, 0.25), (2, False, 16, 4097, 0.05, 0.9),
    (2, True, 16, 17, 0.2, 1.9), (2, True, 9, 1500, 0.2, 1.0), (2, True, 16, 4200, 0.2, 1.99),
    (3, False, 16, 33, 0.1, 0.2), (3, False, 16, 900, 0.1, 0.25), (3, False, 12, 4100, 0.1, 0.6),
    (3, True, 16, 700, 0.2, 1.2), (3, True, 16, 4100, 0.2, 1.99)])
def test_density_gradient_step_bit_exact(ctx, d, periodic, S, n, eps, side):
    m = (NpaConfig.growing_2d() if d == 2 else NpaConfig.growing_3dgs()).replace(
        state_dims=S, hidden_dims=128, eps0=eps, alpha=0.5)
    g = HashGridConfig(d, Boundary.Periodic, HashGridMode.Grid, (10, 10, 10 if d == 3 else 1), eps, 32) if periodic else \
        HashGridConfig(d, Boundary.Clamped, HashGridMode.Particle, (32, 32, 32 if d == 3 else 1), eps, 32)
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :d] = rng.uniform(-side / 2, side / 2, (n, d))
    st = syn.normal_states(n, S, 3)
    w = syn.seeded_weights(m, 5)
    mask = (rng.random(n) < 0.5).astype(np.float32)
    want = O.step(m, w, pos, st, 1, n, g, 1.0, mask)
    got = NpaModel(m, w).step(pos, st, 1, n, g, 1.0, update_mask=mask, ctx=ctx)
    np.testing.assert_array_equal(to_np(got.next_positions), want.next_positions)
    np.testing.assert_array_equal(to_np(got.next_states), want.next_states)
    np.testing.assert_array_equal(to_np(got.density), want.density)
