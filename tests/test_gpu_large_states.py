"""States past 262,144 discs, which re-sort in place: their gradients, and
batches of many small instances."""
import numpy as np
import pytest

from demso_amd import scene as sc
from helpers import batch_of, bits_equal
from test_gpu_adjoint import gpu_grads

pytestmark = pytest.mark.gpu


def parting_pairs(n, seed):
    """Pairs of touching discs in a row on the floor that part within some
    five steps: runs of discs that feel a force at first and none later."""
    s = sc.column_collapse(seed=seed, cols=n, n=n, box=(n * 0.0125, 0.1), jitter=0.0)
    rng = np.random.default_rng(seed)
    k = np.arange(n // 2)
    a, b = s.radius[0::2].astype(np.float64), s.radius[1::2].astype(np.float64)
    apart = a + b - rng.uniform(4e-6, 2e-5, n // 2)
    s.pos[0::2, 0] = 0.0125 + 0.025 * k
    s.pos[1::2, 0] = s.pos[0::2, 0] + np.sqrt(apart ** 2 - (a - b) ** 2)
    s.pos[:, 1] = s.radius
    s.vel[0::2, 0], s.vel[1::2, 0] = -0.2, 0.2
    s.vel[:, 1] = rng.uniform(-0.05, 0.0, n)
    s.omega[:] = rng.normal(size=n).astype(np.float32)
    return s


@pytest.mark.parametrize("fused", [False, True])
def test_checkpoint_interval_of_large_states(gpu_ctx, fused):
    """Segments recomputed from their checkpoints start with a radix-sorted
    step after in-place ones, whose quiet runs are not that step's: the
    gradients are those of one recorded segment (of the state bit for bit; a
    parameter's sum of some 4,000 terms, in another order, far within 1e-9 of
    the largest)."""
    s = batch_of(parting_pairs(500, seed=3), 530)
    assert s.n > 262144
    gpu_ctx.set_step_variant(fused=fused, contact_lists=True)
    rng = np.random.default_rng(1)
    W, V = rng.normal(size=(s.n, 2)), rng.normal(size=(s.n, 2))
    steps = 8
    (gp, gv, par), final = gpu_grads(gpu_ctx, s, steps, W, V, K=steps)
    assert np.count_nonzero(par[:, 1]) == len(s.materials)
    for K in (2, 3):
        (gpk, gvk, park), finalk = gpu_grads(gpu_ctx, s, steps, W, V, K=K)
        assert bits_equal(finalk, final), K
        assert bits_equal(gpk, gp) and bits_equal(gvk, gv), K
        assert np.allclose(park, par, rtol=0, atol=1e-9 * np.abs(par).max(axis=0)), K
