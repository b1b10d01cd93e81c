"""Kernels at the sizes where their work splits: waves and tiles that are
exactly full, one over and one short, and loads that gather in one place."""
import numpy as np
import pytest

from demso_amd import api
from demso_amd import scene as sc
from helpers import bits_equal, dev

pytestmark = pytest.mark.gpu

FIELDS = ("hash", "index", "cellStart", "cellEnd", "id", "type", "loc", "pos", "vel", "theta", "omega", "acc",
          "alpha", "pressure")

@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 5000])
def test_image_of_discs_past_its_end(gpu_ctx, oracle, n):
    """Discs above and right of the image clamp to its last pixel, which the
    highest index among them owns (some discs lie inside, some across)."""
    s = sc.settling(seed=n, side=71)
    s.pos, s.type, s.radius = s.pos[:n].copy(), s.type[:n], s.radius[:n].copy()
    rng = np.random.default_rng(n)
    lx, ly = s.instances[0].box
    s.pos[:, 0] = rng.uniform(0.0, 1.3 * lx, n)
    s.pos[:, 1] = rng.uniform(0.8 * ly, 3.0 * ly, n)
    s.pos[n // 2] = (lx * (1 - 1e-3), ly * (1 - 1e-3))
    zero = np.zeros(n, np.float32)
    gpu_ctx.load_scene(s)
    rp = api.render_params(s, image_height=300, view_rotations=False)
    import torch

    img = torch.zeros((rp["image_dim"][1], rp["image_dim"][0], 4), dtype=torch.uint8, device="cuda")
    api.plotParticles(gpu_ctx, img, dev(s.pos), dev(zero), dev(s.type), n, rp, dev(zero), radius=dev(s.radius))
    want = oracle.plot(s, rp, s.pos, zero, s.type, zero, radius=s.radius)
    assert np.array_equal(img.cpu().numpy(), want)


@pytest.mark.parametrize("n", [1, 255, 1023, 1025, 65537])
def test_pressure_scale_blocks(gpu_ctx, n):
    v = np.random.default_rng(n).normal(size=n).astype(np.float32)
    for at in (0, n // 2, n - 1):
        w = v.copy()
        w[at] = 9.5
        assert api.updatePressureScale(gpu_ctx, dev(w), n) == 9.5


def swept_row(n, seed=2):
    """n discs over two wide cell rows, a few of which hop between them every
    step, so that each hop shifts the slots of all the discs between."""
    s = sc.column_collapse(seed=seed, cols=n, n=n, box=(n * 0.012, 0.05), pitch=0.0115, jitter=0.0, dt=1e-4)
    s.pos[:, 1] = np.where(np.arange(n) % 2 == 0, 0.008, 0.025).astype(np.float32)
    rng = np.random.default_rng(seed)
    hop = rng.choice(n, max(2, n // 500), replace=False)
    s.vel[hop, 1] = np.where(s.pos[hop, 1] < 0.011, 100.0, -100.0)
    return s


@pytest.mark.parametrize("n", [64, 2047, 2048, 2049, 4097, 12289])
def test_long_lists_equal_radix(gpu_ctx, n):
    """Few movers that shift whole tiles of stayers: the in-place re-sort's
    lists against the radix sort."""
    s = swept_row(n)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    try:
        listed = []
        for _ in range(4):
            a.step(2)
            b.step(2)
            listed.append(b.resort_counts()["listed"])
            da, db = a.download(), b.download()
            for k in FIELDS:
                assert bits_equal(da[k], db[k]), k
        assert max(listed) > n // 8
    finally:
        a.close()
        b.close()


def packed_rows(n, seed, attract=0.0):
    """n discs in a few rows of overlapping neighbours, a wide empty gap in
    the middle (the wave across it has rows far apart) and, at its right
    end, a heap of discs in one cell (rows of more than 64 candidates)."""
    s = sc.column_collapse(seed=seed, cols=max(1, n // 4), n=n, box=(n * 0.012 + 6.0, 0.4), pitch=0.0098,
                           jitter=0.0009)
    s.pos[n // 2:, 0] += 4.0
    heap = slice(n - n // 5, n)
    rng = np.random.default_rng(seed)
    s.pos[heap] = s.pos[heap][:1] + rng.uniform(-0.004, 0.004, s.pos[heap].shape).astype(np.float32)
    s.vel[:] = (rng.normal(size=s.vel.shape) * 0.2).astype(np.float32)
    s.omega[:] = (rng.normal(size=n) * 30.0).astype(np.float32)
    s.materials[0].attract = attract
    return s


@pytest.mark.parametrize("attract", [0.0, 3.0])
@pytest.mark.parametrize("n", [5, 63, 64, 65, 129, 700])
def test_contact_lists_across_windows(gpu_ctx, oracle, n, attract):
    """The contact-list walk where a wave's rows fit its windows, where they
    do not, where a wave is not full and where a row has over 64 candidates,
    with and without attraction, against the oracle."""
    s = packed_rows(n, seed=n, attract=attract)
    gpu_ctx.set_step_variant(contact_lists=True)
    sim, ref = api.Simulation(gpu_ctx, s), oracle.Sim(s, "f32")
    try:
        for _ in range(3):
            sim.step(1)
            ref.step(1)
            got, want = sim.download(), ref.state()
            for k in ("hash", "index", "pos", "vel", "omega", "acc", "alpha", "pressure"):
                assert bits_equal(got[k], want[k]), k
    finally:
        sim.close()
        ref.close()


@pytest.mark.parametrize("key_bits", [8, 13, 24, 32])
@pytest.mark.parametrize("n", [2, 64, 4095, 4096, 4097, 8191, 8192, 8193, 10241, 1048576, 1048577])
@pytest.mark.parametrize("offset", [0, 1])
def test_sort_tile_edges(gpu_ctx, n, key_bits, offset):
    """The sort in one workgroup, in small and in large tiles, at their
    limits, from aligned and unaligned arrays; ties keep their order."""
    import torch

    g = 1 << min(key_bits, 16)
    s = sc.column_collapse(cols=8, rows=8)
    s.instances = [sc.Instance(box=(1.0, 1.0), extent=(1.0, 1.0), grid=(g, (1 << key_bits) // g - (key_bits == 32)))]
    gpu_ctx.load_scene(s)
    top = s.instances[0].cells
    k = np.random.default_rng(n).integers(0, top, n, dtype=np.uint64).astype(np.uint32)
    k[n // 3: n // 2] = k[0]
    v = np.arange(n, dtype=np.uint32)
    dk, dv = (torch.zeros(n + 4, dtype=torch.int32, device="cuda")[offset:offset + n] for _ in range(2))
    dk.copy_(torch.from_numpy(k.view(np.int32)))
    dv.copy_(torch.from_numpy(v.view(np.int32)))
    api.sortParticles(gpu_ctx, dk, dv, n)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(dk.cpu().numpy().view(np.uint32), k[order])
    assert np.array_equal(dv.cpu().numpy().view(np.uint32), order.astype(np.uint32))


def walkers(n, seed, cells, speed):
    """n discs strewn over cells x cells cells (mostly empty ones), moving
    fast enough that some change cell every step."""
    s = sc.column_collapse(seed=seed, cols=n, n=n, box=(cells * 0.011, cells * 0.011), dt=1e-4)
    rng = np.random.default_rng(seed)
    s.pos[:] = rng.uniform(0.02, cells * 0.011 - 0.02, s.pos.shape).astype(np.float32)
    s.vel[:] = (rng.normal(size=s.vel.shape) * speed).astype(np.float32)
    return s


# few discs in many cells (a mover's next occupied cell is far away), movers
# around the 512 whose order fits LDS, and far more of them
WHOLE = {
    "one": lambda: walkers(1, 1, 40, 50.0),
    "strewn": lambda: walkers(300, 2, 500, 20.0),
    "hundreds": lambda: walkers(6000, 3, 300, 4.0),
    "about_512": lambda: walkers(8200, 4, 200, 2.9),
    "most": lambda: walkers(3000, 5, 100, 90.0),
}


@pytest.mark.parametrize("name", list(WHOLE))
@pytest.mark.parametrize("fused", [False, True])
def test_whole_resort_equals_radix(gpu_ctx, name, fused):
    s = WHOLE[name]()
    gpu_ctx.set_step_variant(fused=fused, contact_lists=True)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    movers = []
    try:
        for steps in (1, 1, 1, 2, 4, 9):
            a.step(steps)
            (b.step_graph if steps > 1 else b.step)(steps)
            movers.append(b.mover_count())
            da, db = a.download(), b.download()
            for k in FIELDS:
                assert bits_equal(da[k], db[k]), (k, steps)
        print(name, fused, movers, flush=True)
        assert max(movers) > 0 or name == "one"
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("speed", [0.02, 2.0, 30.0])
@pytest.mark.parametrize("fused", [False, True])
def test_inplace_resort_of_large_states(gpu_ctx, speed, fused):
    """Past 262,144 discs re-sorted steps run in place: few movers, thousands
    (the movers workgroup's radix path beyond 4,096) and half the state."""
    s = walkers(262145 + 4096, 6, 700, speed)
    gpu_ctx.set_step_variant(fused=fused, contact_lists=True)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    try:
        for steps in (1, 1, 2, 3):
            a.step(steps)
            (b.step_graph if steps > 1 else b.step)(steps)
            da, db = a.download(), b.download()
            for k in FIELDS:
                assert bits_equal(da[k], db[k]), (k, steps)
        assert b.mover_count() > 0
    finally:
        a.close()
        b.close()


def test_variants_changed_between_steps(gpu_ctx):
    """A step's re-sort reads the movers as the step before listed them: the
    layouts in turn, eager and replayed, against radix-sorted steps."""
    s = walkers(5000, 7, 150, 5.0)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    try:
        for k in range(12):
            gpu_ctx.set_step_variant(fused=bool(k & 1), copy=k % 3 == 0, contact_lists=k % 4 != 0)
            a.step(3)
            (b.step_graph if k & 2 else b.step)(3)
            da, db = a.download(), b.download()
            for f in FIELDS:
                assert bits_equal(da[f], db[f]), (f, k)
    finally:
        a.close()
        b.close()


def test_adjoint_of_large_state_lists(gpu_ctx):
    """Past 262,144 discs the adjoint lists the particles with contacts first:
    88 copies of one system in a batch (boundaries of tiles and list groups
    everywhere in it; free, touching and heaped discs) against the system
    alone, which takes the one-kernel path: gradients of the state bit for
    bit, of the parameters to the order of their sums."""
    import dataclasses

    import torch

    one = packed_rows(3001, seed=9)
    one.pos[1000:2000, 0] *= np.float32(1.02)
    one.pos[1000:2000, 1] += np.float32(0.2)  # (free discs)
    copies = 88
    many = one.copy()
    for f in ("pos", "vel", "theta", "omega", "radius"):
        setattr(many, f, np.concatenate([getattr(one, f)] * copies))
    many.type = np.repeat(np.arange(copies, dtype=np.uint32), one.n)
    many.id = np.arange(copies * one.n, dtype=np.uint32)
    many.loc = many.id.copy()
    g = one.instances[0]
    many.instances = [dataclasses.replace(g, cell_base=k * g.cells) for k in range(copies)]
    many.materials = [dataclasses.replace(one.materials[0], instance=k) for k in range(copies)]
    assert many.n > 262144
    rng = np.random.default_rng(0)
    W, V = rng.normal(size=(one.n, 2)).astype(np.float32), rng.normal(size=(one.n, 2)).astype(np.float32)
    out = []
    for s, k in ((one, 1), (many, copies)):
        sim = api.Simulation(gpu_ctx, s)
        adj = api.Adjoint(sim, checkpoint_every=3)
        adj.forward(3)
        gp, gv, par = adj.backward(torch.from_numpy(np.tile(W, (k, 1))).cuda(), torch.from_numpy(np.tile(V, (k, 1))).cuda(),
                                   num_types=k)
        out.append((gp.cpu().numpy(), gv.cpu().numpy(), par.cpu().numpy()))
        adj.close()
        sim.close()
    (gp1, gv1, par1), (gpm, gvm, parm) = out
    assert np.count_nonzero(par1) >= 3
    for k in (0, 1, 40, copies - 1):
        at = slice(k * one.n, (k + 1) * one.n)
        assert bits_equal(gpm[at], gp1) and bits_equal(gvm[at], gv1), k
    # a sum of n terms in another order: n eps of the terms' magnitudes at most
    scale = np.abs(par1).max()
    assert np.all(np.abs(parm - par1) <= 1e-9 * np.maximum(np.abs(par1), 1e-3 * scale))


@pytest.mark.parametrize("flags", [1, 0])
@pytest.mark.parametrize("extent", [(8.0, 7.3), (1e-3, 123.456), (3.1415927, 0.7)])
def test_cell_keys_at_cell_borders(gpu_ctx, oracle, extent, flags):
    """Positions at the floats around every cell border (and their negatives
    and multiples beyond the grid): the quotient that decides the cell is the
    correctly rounded one."""
    from test_oracle_kat import one_type_scene

    grid = (64, 128)
    axes = []
    for e, g in zip(extent, grid):
        x = (np.arange(0, 2 * g + 1, dtype=np.float64) * e / g).astype(np.float32)
        near = [x]
        for way in (np.float32(-np.inf), np.float32(np.inf)):
            y = x
            for _ in range(3):
                y = np.nextafter(y, way)
                near.append(y)
        x = np.concatenate(near)
        axes.append(np.concatenate([x, -x]))
    n = max(map(len, axes))
    rng = np.random.default_rng(1)
    pos = np.stack([rng.permutation(np.resize(a, n)) for a in axes], 1).astype(np.float32)
    s = one_type_scene(pos, box=extent, grid=grid, flags=flags)
    gpu_ctx.load_scene(s)
    want, _ = oracle.calc_hash(oracle.System(s), s.pos, s.type)
    h, i = dev(np.zeros(n, np.uint32)), dev(np.zeros(n, np.uint32))
    api.calcHash(gpu_ctx, dev(s.pos), i, h, n)
    gpu_ctx.synchronize()
    assert np.array_equal(h.cpu().numpy().view(np.uint32), want)


def check_one_step(gpu_ctx, oracle, s):
    gpu_ctx.set_step_variant(contact_lists=True)
    sim, ref = api.Simulation(gpu_ctx, s), oracle.Sim(s, "f32")
    try:
        sim.step(1)
        ref.step(1)
        got, want = sim.download(), ref.state()
        for k in ("hash", "index", "pos", "vel", "omega", "acc", "alpha", "pressure"):
            assert bits_equal(got[k], want[k]), k
        assert np.count_nonzero(want["acc"]) > 0
    finally:
        sim.close()
        ref.close()


@pytest.mark.parametrize("attract", [0.0, 3.0])
@pytest.mark.parametrize("m", [31, 32, 33, 63, 64, 65, 95, 200])
def test_crowded_neighbourhoods(gpu_ctx, oracle, m, attract):
    """m discs in three by three cells (one or two words of marks, then passes
    over 31), one copy in a corner of the clamped grid, against the oracle."""
    n = 2 * m
    s = sc.column_collapse(seed=m, cols=n, n=n, box=(1.0, 0.5))
    g = s.instances[0]
    cell = np.array(g.box) / np.array(g.grid)
    rng = np.random.default_rng(m)
    at = rng.uniform(0.05, 2.95, (n, 2))
    s.pos[:] = ((at + np.where(np.arange(n)[:, None] < m, 4.0, 0.0)) * cell).astype(np.float32)
    s.vel[:] = (rng.normal(size=s.vel.shape) * 0.2).astype(np.float32)
    s.omega[:] = (rng.normal(size=n) * 30.0).astype(np.float32)
    s.materials[0].attract = attract
    check_one_step(gpu_ctx, oracle, s)


def test_contacts_at_the_ends_of_the_float_range(gpu_ctx, oracle):
    """Pairs whose squared distance is tiny or whose direction has a subnormal
    component: the law's roots and quotients round as sqrtf and a division."""
    xs = [1e-45, 3e-45, 7e-42, 1e-39, 3e-38, 1e-19, 5e-19, 3e-16, 1e-12, 1e-7]
    n = 2 * len(xs)
    s = sc.column_collapse(seed=1, cols=n, n=n, box=(0.4, 0.5))
    for k, x in enumerate(xs):
        y = 0.02 + 0.04 * k
        apart = 0.0 if x >= 1e-19 else 0.004 + 0.0001 * k
        s.pos[2 * k] = (0.0, y)
        s.pos[2 * k + 1] = (x, y + apart)
    rng = np.random.default_rng(2)
    s.vel[:] = (rng.normal(size=s.vel.shape) * 0.2).astype(np.float32)
    s.vel[4:8] *= np.float32(1e-25)
    s.omega[:] = 0.0
    check_one_step(gpu_ctx, oracle, s)


@pytest.mark.parametrize("n,cells", [(1, 40), (300, 130), (300, 1000), (5000, 4000)])
def test_sparse_grids_equal_radix(gpu_ctx, n, cells):
    """Small states re-sort as a whole while their grid has at most 64 cells a
    disc, and in place beyond."""
    s = walkers(n, 11, cells, 30.0)
    gpu_ctx.set_step_variant(fused=True, contact_lists=True)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    try:
        for steps in (1, 1, 2, 5):
            a.step(steps)
            (b.step_graph if steps > 1 else b.step)(steps)
            da, db = a.download(), b.download()
            for k in FIELDS:
                assert bits_equal(da[k], db[k]), (k, steps)
    finally:
        a.close()
        b.close()


def test_grid_of_nearly_2_to_the_32_cells(gpu_ctx):
    """The largest grids: no kernel's cell index wraps (51 GB of cell arrays)."""
    s = walkers(200000, 12, 700, 1.0)
    s.instances = [sc.Instance(box=(7.2e2, 7.2e2), extent=(7.2e2, 7.2e2), grid=(65535, 65536))]
    s.pos[:] = np.random.default_rng(12).uniform(1.0, 719.0, s.pos.shape).astype(np.float32)
    out = []
    for mode in (1, 2):
        sim = api.Simulation(gpu_ctx, s)
        try:
            sim.set_sort_mode(mode)
            sim.step(2)
            sim.step_graph(4)
            out.append(sim.download(extra=False))
            movers = sim.mover_count()
        finally:
            sim.close()
    assert movers > 0
    for k in ("id", "type", "loc", "pos", "vel", "theta", "omega"):
        assert bits_equal(out[0][k], out[1][k]), k


def hoppers(n, slots):
    """n discs a cell apart, of which those at the given sorted slots hop to
    the free cell on their right or above in the first step."""
    cols = int(np.ceil(np.sqrt(n)))
    s = sc.column_collapse(seed=1, cols=cols, n=n, box=((2 * cols + 4) * 0.011, (2 * cols + 4) * 0.011), dt=1e-4)
    k = np.arange(n)
    g = s.instances[0]
    cell = np.array(g.extent) / np.array(g.grid)
    s.pos[:] = ((np.stack([k % cols, k // cols], 1) * 2 + 0.5) * cell).astype(np.float32)
    s.radius[:] = 0.0045
    s.vel[slots, np.asarray(slots) % 2] = 110.0
    return s


# the small states' mover lists (a list takes every fourth wave's): one list
# exactly full for the ranking of few, one over, all four full, one over; whole
# runs of 1,024 movers; every disc
HOPS = {
    "one_list_64": (4099, np.arange(64)),
    "one_list_65": (4099, np.r_[np.arange(64), 256]),
    "lists_full": (4099, np.arange(256)),
    "lists_full_and_1": (4099, np.arange(257)),
    "first_and_last": (4099, np.array([0, 4098])),
    "random_1000": (20037, np.random.default_rng(0).choice(20037, 1000, replace=False)),
    "runs": (70001, np.r_[np.arange(1000, 5200), np.arange(66000, 70001)]),
    "all_300": (300, np.arange(300)),
    "all_5000": (5000, np.arange(5000)),
    "random_20000": (262143, np.random.default_rng(1).choice(262143, 20000, replace=False)),
    "all_262144": (262144, np.arange(262144)),
}


@pytest.mark.parametrize("name", list(HOPS))
@pytest.mark.parametrize("fused", [False, True])
def test_mover_lists_equal_radix(gpu_ctx, name, fused):
    n, slots = HOPS[name]
    s = hoppers(n, slots)
    gpu_ctx.set_step_variant(fused=fused, contact_lists=True)
    a, b = api.Simulation(gpu_ctx, s), api.Simulation(gpu_ctx, s)
    a.set_sort_mode(1)
    b.set_sort_mode(2)
    try:
        for k in range(4):
            a.step(1)
            b.step(1)
            da, db = a.download(), b.download()
            if k == 1:
                assert b.mover_count() == len(slots)
            for f in FIELDS:
                assert bits_equal(da[f], db[f]), (f, k)
        a.step(4)
        b.step_graph(4)
        da, db = a.download(), b.download()
        for f in FIELDS:
            assert bits_equal(da[f], db[f]), f
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("wrap", [False, True])
@pytest.mark.parametrize("m", [66, 100, 282, 600, 1500])
def test_crowded_rows(gpu_ctx, oracle, m, wrap):
    """Rows of 22 to 500 candidates (one to six chunks of 93, in parts of up
    to 31): a crowd inside the grid, one at its corner and one in a single
    cell, whose rows above and below are empty; clamped and wrapping."""
    from demso_amd import _lib

    rng = np.random.default_rng(m)
    s = sc.column_collapse(seed=m, cols=3 * m, n=3 * m, box=(0.352, 0.352))
    s.instances = [sc.Instance(box=(0.352, 0.352), extent=(0.352, 0.352), grid=(32, 32))]
    if wrap:
        s.flags &= ~_lib.DEM_GRID_CLAMP
    cell = 0.011
    s.pos[:m] = (rng.uniform(0.05, 2.95, (m, 2)) + 8.0) * cell
    s.pos[m:2 * m] = (rng.uniform(0.05, 2.95, (m, 2)) + (0.0 if not wrap else 29.0)) * cell
    s.pos[2 * m:] = (rng.uniform(0.05, 0.95, (m, 2)) + np.array([20.0, 25.0])) * cell
    s.radius[:] = rng.uniform(0.0005, 0.0055, s.n).astype(np.float32)
    s.vel[:] = (rng.normal(size=s.vel.shape) * 0.2).astype(np.float32)
    s.omega[:] = (rng.normal(size=s.n) * 30.0).astype(np.float32)
    check_one_step(gpu_ctx, oracle, s)
