"""Dry regions: the step kernels pass over cells that hold neither water nor
flux, row by row inside a launch and, from the second launch of a call on,
whole tasks.  The results are the restatement's bits, for water that stands,
spreads into dry ground, falls on it or flows in from a single wet cell, on
terrain and constants where a dry cell's flux underflows or overflows too."""
import numpy as np
from bitwise import same_bits
import pytest

pytestmark = pytest.mark.gpu

F32 = np.float32
LAUNCHES = [(8, 2), (8, 3), (8, 4), (8, 5), (8, 6), (8, 8), (3, 5), (4, 4), (5, 4), (6, 8), (7, 4)]


def ground(tws, H, W, seed):
    return tws.generate_fbm_terrain(W, H, seed=seed, height_scale=40.0)


def scenes(H, W, seed):
    """(name, depth, flux, rain) of states that are dry almost everywhere."""
    rng = np.random.default_rng(seed)
    zero = lambda: (np.zeros((H, W), F32), np.zeros((H, W, 4), F32))
    d, f = zero()
    yield "dry", d, f, None
    d, f = zero()
    d[H // 2:H // 2 + 9, W // 3:W // 3 + 7] = 20.0
    yield "dam", d, f, None
    d, f = zero()
    yield "rain", d, f, (0.8 * W, 0.3 * H, 1e-2, 30.0)
    # single wet cells and single cells that hold flux but no water, some on
    # the first and last rows and columns
    d, f = zero()
    for _ in range(6):
        d[rng.integers(H), rng.integers(W)] = rng.random() * 3.0
        f[rng.integers(H), rng.integers(W), rng.integers(4)] = rng.random()
    d[0, W - 1] = d[H - 1, 0] = 1.0
    yield "specks", d, f, None
    # a lake at the bottom edge and tiny depths at the top one
    d, f = zero()
    d[H - 20:] = 0.5
    d[:3, ::5] = 1e-41
    yield "edges", d, f, None
    d, f = zero()
    d[rng.random((H, W)) < 0.002] = F32(-0.0)
    d[H // 4, W // 2] = 2.0
    yield "negative zeros", d, f, None


def advance(tws, b, d, f, rain, p, kernel, k, calls):
    H, W = b.shape
    with tws.Simulation(W, H, p) as s:
        s.set_launch(kernel, k)
        s.upload(b, d, f)
        if rain:
            s.set_rain(*rain)
        for n in calls:
            s.step(n)
        return s.download()


@pytest.mark.parametrize("kernel,k", LAUNCHES)
def test_dry_scenes_bitwise(gpu, oracle, kernel, k):
    """Several launches per call, two calls, on a grid of several segments and
    strips (and, for the tile kernels, tiles)."""
    H, W = 611, 437
    p = gpu.params_physical(0.02, 9.81, 1.0, 1.0, 0.995)
    b = ground(gpu, H, W, 40 + k)
    for name, d, f, rain in scenes(H, W, k):
        out = advance(gpu, b, d, f, rain, p, kernel, k, (5 * k + 3, 4 * k))
        de, fe, _ = oracle.step(b, d, f, p.flow_friction, p.water_acceleration,
                                p.cell_area_inv_timescaled, n=9 * k + 3, rain=rain)
        assert same_bits(out["depth"], de), name
        assert same_bits(out["flux"], fe), name


@pytest.mark.parametrize("kernel,k", [(8, 6), (8, 4), (5, 4)])
@pytest.mark.parametrize("case", ["tiny heights", "tiny constants", "no area", "no acceleration",
                                  "flat", "huge heights"])
def test_dry_arithmetic_bitwise(gpu, oracle, kernel, k, case):
    """Dry ground where a flux underflows or overflows on its way to zero: such
    cells do hold flux after a step and are not passed over."""
    H, W = 300, 260
    rng = np.random.default_rng(3)
    b = (rng.random((H, W)) * 10.0).astype(F32)
    F, K, C = F32(0.99), F32(0.2), F32(0.02)
    if case == "tiny heights":
        b[100:160, 100:180] = (rng.random((60, 80)) * 1e-37).astype(F32)
    elif case == "tiny constants":
        K, C = F32(1e-30), F32(1e-15)
    elif case == "no area":
        C = F32(0.0)
    elif case == "no acceleration":
        K = F32(0.0)
    elif case == "flat":
        b[:] = 0.0
    else:
        b[50:60, 50:60] = (rng.random((10, 10)) * 1e25).astype(F32)
    d = np.zeros((H, W), F32)
    d[200:210, 30:50] = 1.0
    f = np.zeros((H, W, 4), F32)
    p = gpu.Params()
    p.flow_friction, p.water_acceleration, p.cell_area_inv_timescaled = F, K, C
    p.boundary, p.ghost_alpha = gpu.BOUNDARY_CLOSED, 0.0
    out = advance(gpu, b, d, f, None, p, kernel, k, (4 * k, 2 * k))
    de, fe, _ = oracle.step(b, d, f, F, K, C, n=6 * k)
    assert same_bits(out["depth"], de)
    assert same_bits(out["flux"], fe)


def test_dry_ground_changed_between_calls(gpu, oracle):
    """Nothing about dry ground outlives a call: water brushed, rained or
    uploaded onto it is stepped, as is terrain raised under it."""
    H, W = 700, 500
    p = gpu.params_physical(0.02, 9.81, 1.0, 1.0, 0.995)
    c = (p.flow_friction, p.water_acceleration, p.cell_area_inv_timescaled)
    b = ground(gpu, H, W, 9)
    d = np.zeros((H, W), F32)
    d[10:20, 10:20] = 3.0
    with gpu.Simulation(W, H, p) as s:
        s.set_launch(gpu.KERNEL_STREAM_128, 6)
        s.upload(b, d)
        s.step(30)
        de, fe, _ = oracle.step(b, d, None, *c, n=30)
        s.apply_brush(400.0, 600.0, 0.5, 40.0)
        de = oracle.brush(de, 400.0, 600.0, 0.5, 40.0)
        s.step(30)
        de, fe, _ = oracle.step(b, de, fe, *c, n=30)
        s.set_rain(250.0, 350.0, 1e-2, 90.0)
        s.step(30)
        rain = (250.0, 350.0, 1e-2, 90.0)
        de, fe, _ = oracle.step(b, de, fe, *c, n=30, rain=rain)
        out = s.download()
        assert same_bits(out["depth"], de) and same_bits(out["flux"], fe)
        b2 = ground(gpu, H, W, 10)
        s.upload(b2, out["depth"], out["flux"])
        s.step(30)
        de, fe, _ = oracle.step(b2, de, fe, *c, n=30, rain=rain)
        out = s.download()
        assert same_bits(out["depth"], de) and same_bits(out["flux"], fe)


@pytest.mark.parametrize("graphs,low", [(True, False), (False, False), (True, True)])
def test_dry_batch_bitwise(gpu, oracle, graphs, low):
    """A streaming batch of dry grids with a little water each, different step
    counts, replayed twice; with a grid too low to keep masks, too."""
    p = gpu.params_physical(0.02, 9.81, 1.0, 1.0, 0.995)
    c = (p.flow_friction, p.water_acceleration, p.cell_area_inv_timescaled)
    shapes = [(611, 437), (90, 1000), (1300, 60), (64, 64), (17, 300), (900, 900), (2100, 210)]
    if low:
        shapes.append((5, 300))
    with gpu.Batch(8, sum(gpu.grid_footprint(w, h) for h, w in shapes)) as batch:
        batch.set_launch(gpu.KERNEL_STREAM_128, 6)
        batch.use_graphs(graphs)
        state = {}
        for i, (h, w) in enumerate(shapes):
            gid = batch.add(w, h, p)
            b = ground(gpu, h, w, 60 + i)
            d = np.zeros((h, w), F32)
            d[h // 2, w // 3] = 5.0
            rain = (0.7 * w, 0.2 * h, 1e-2, 20.0) if i % 2 else None
            batch.upload(gid, b, d)
            if rain:
                batch.set_rain(gid, *rain)
            state[gid] = [b, d, None, rain]
        for turn in range(2):
            for gid in state:
                batch.set_steps(gid, 31 + 7 * (gid % 3))
            batch.run()
            for gid, st in state.items():
                n = 31 + 7 * (gid % 3)
                st[1], st[2], _ = oracle.step(st[0], st[1], st[2], *c, n=n, rain=st[3])
                out = batch.download(gid)
                assert same_bits(out["depth"], st[1]), (turn, gid)
                assert same_bits(out["flux"], st[2]), (turn, gid)
