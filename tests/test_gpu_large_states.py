"""States past 262,144 discs, which re-sort in place: their gradients, and
batches of many small instances."""
import numpy as np
import pytest

from demso_amd import api
from demso_amd import scene as sc
from helpers import batch_of, bits_equal, mixed_pack
from test_gpu_adjoint import gpu_grads
from test_gpu_kernel_edges import packed_rows

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


def test_adjoint_past_a_million_discs_lists_contacts(gpu_ctx):
    """Past 1,048,576 discs the adjoint lists the discs with contacts first: a
    batch of copies of one system (free, touching and heaped discs; rows of
    more than 64 candidates) against the system alone, which takes the
    one-kernel path: gradients of the state bit for bit, of the parameters to
    the order of their sums (some 4,000 terms)."""
    one = packed_rows(3001, seed=9)
    one.pos[1000:2000, 0] *= np.float32(1.02)
    one.pos[1000:2000, 1] += np.float32(0.2)  # (free discs)
    copies = 350
    many = batch_of(one, copies)
    assert many.n > 1048576
    rng = np.random.default_rng(0)
    W, V = rng.normal(size=(one.n, 2)), rng.normal(size=(one.n, 2))
    (gp1, gv1, par1), _ = gpu_grads(gpu_ctx, one, 3, W, V, K=2)
    (gpm, gvm, parm), _ = gpu_grads(gpu_ctx, many, 3, np.tile(W, (copies, 1)), np.tile(V, (copies, 1)), K=2)
    assert np.count_nonzero(par1) >= 3
    for k in (0, 1, 171, copies - 1):
        at = slice(k * one.n, (k + 1) * one.n)
        assert bits_equal(gpm[at], gp1) and bits_equal(gvm[at], gv1), k
    assert np.all(np.abs(parm - par1) <= 1e-9 * np.maximum(np.abs(par1), 1e-3 * np.abs(par1).max()))


def squeezed_batch(counts, seed):
    s = sc.ensemble(seed=seed, instances=len(counts), counts=counts)
    rng = np.random.default_rng(seed)
    s.pos[:] *= np.float32(0.86)
    s.vel[:] = (rng.normal(size=s.vel.shape) * 0.1).astype(np.float32)
    s.omega[:] = (rng.normal(size=s.n) * 10.0).astype(np.float32)
    return s


def type_radii(s):
    """The same discs with their material's radius, mass and inertia (the
    generator's materials have none)."""
    for m, r in zip(s.materials, np.random.default_rng(5).uniform(0.0048, 0.0054, len(s.materials))):
        m.radius = float(r)
        m.mass = m.areal * m.radius ** 2
        m.inertia = 0.4 * m.mass * m.radius ** 2
    s.radius = None
    return s


# waves inside one instance, waves across two or more (the last wave not
# full), and several materials in a wave of one instance; radii of the discs
# or of their materials
STATES = {
    "aligned": lambda: squeezed_batch([4416] * 60, 1),
    "ragged": lambda: squeezed_batch(np.random.default_rng(3).integers(1000, 5000, 90).tolist(), 3),
    "straddling": lambda: squeezed_batch(np.random.default_rng(2).integers(180, 420, 900).tolist(), 2),
    "straddling_type_radii": lambda: type_radii(squeezed_batch([299] * 900, 4)),
    "materials": lambda: mixed_pack(cols=521, rows=505),
}
FIELDS = ("hash", "index", "cellStart", "id", "type", "loc", "pos", "vel", "theta", "omega", "acc", "alpha", "pressure")


@pytest.mark.parametrize("name", list(STATES))
def test_large_states_step_alike_in_every_layout(oracle, name):
    """Past 262,144 discs: contact lists, split and fused, re-sorted in place,
    against the plain mode with the radix sort, and all against the oracle
    after one step."""
    s = STATES[name]()
    assert s.n > 262144
    ref = oracle.Sim(s, "f32")
    ref.step(1)
    want = ref.state()
    ref.close()
    assert np.count_nonzero(want["acc"]) > s.n // 4
    base = None
    for variant, mode in ((dict(contact_lists=False), 1), (dict(contact_lists=True), 2),
                          (dict(contact_lists=True, fused=True), 2)):
        ctx = api.Context(0)
        sim = api.Simulation(ctx, s)
        ctx.set_step_variant(**variant)
        sim.set_sort_mode(mode)
        sim.step(1)
        got = sim.download()
        for k in ("hash", "index", "pos", "vel", "theta", "omega", "acc", "alpha", "pressure"):
            assert bits_equal(got[k], want[k]), (variant, k)
        sim.step(2)
        sim.step_graph(6)
        got = sim.download()
        base = base or got
        for k in FIELDS:
            assert bits_equal(got[k], base[k]), (variant, k)
        sim.close()
        ctx.close()
