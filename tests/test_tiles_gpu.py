"""Tile kernels: launches that pass over dry tiles (grids of many tiles), and
grids whose last rows and columns the reference's truncating dispatch shapes
leave as they are.  Bit for bit against the restatement."""
import numpy as np
from bitwise import same_bits
import pytest
from test_dry_gpu import ground, scenes

pytestmark = pytest.mark.gpu

F32 = np.float32
C, Z, D = "closed", "zero", "dispatch"


def boundary(gpu, oracle, name):
    return {C: (gpu.BOUNDARY_CLOSED, oracle.BOUNDARY_CLOSED),
            Z: (gpu.BOUNDARY_ZERO, oracle.BOUNDARY_ZERO),
            D: (gpu.BOUNDARY_REFERENCE_DISPATCH, oracle.BOUNDARY_DISPATCH)}[name]


def check(gpu, oracle, b, d, f, rain, kernel, k, edge, calls):
    H, W = b.shape
    ours, theirs = boundary(gpu, oracle, edge)
    p = gpu.params_physical(0.02, 9.81, 1.0, 1.0, 0.995, boundary=ours)
    with gpu.Simulation(W, H, p) as s:
        if kernel:
            s.set_launch(kernel, k)
        s.upload(b, d, f)
        if rain:
            s.set_rain(*rain)
        for n in calls:
            s.step(n)
        out = s.download()
    de, fe, _ = oracle.step(b, d, f, p.flow_friction, p.water_acceleration,
                            p.cell_area_inv_timescaled, n=sum(calls), boundary=theirs, rain=rain)
    assert same_bits(out["depth"], de) and same_bits(out["flux"], fe)


# 1024 tiles or more: 48 x 48 and 44 x 44 cells of 64x64 tiles at k = 4 and 5,
# 112 x 48 and 108 x 44 of 128x64 tiles
@pytest.mark.parametrize("kernel,k,shape", [(5, 4, (1601, 1570)), (5, 5, (1453, 1410)),
                                            (5, 4, (16500, 130)), (3, 4, (1700, 3333)),
                                            (3, 5, (1500, 3400))])
@pytest.mark.parametrize("edge", [C, Z, D])
def test_dry_tiles_bitwise(gpu, oracle, kernel, k, shape, edge):
    """Launches that pass over dry tiles, called twice: nothing is kept from
    one call to the next."""
    H, W = shape
    b = ground(gpu, H, W, 70 + k)
    for i, (_, d, f, rain) in enumerate(scenes(H, W, k)):
        if i % 3 == (C, Z, D).index(edge):
            check(gpu, oracle, b, d, f, rain, kernel, k, edge, (5 * k + 3, 4 * k))


@pytest.mark.parametrize("graphs", [True, False])
def test_dry_tiles_batch_bitwise(gpu, oracle, graphs):
    """The same in a batch, grids of different step counts."""
    p = gpu.params_physical(0.02, 9.81, 1.0, 1.0, 0.995)
    c = (p.flow_friction, p.water_acceleration, p.cell_area_inv_timescaled)
    shapes = [(900, 800), (1100, 1000), (700, 900), (64, 64)]
    with gpu.Batch(4, sum(gpu.grid_footprint(w, h) for h, w in shapes)) as batch:
        batch.set_launch(gpu.KERNEL_TILE_64x64, 4)
        batch.use_graphs(graphs)
        state = {}
        for i, (h, w) in enumerate(shapes):
            gid = batch.add(w, h, p)
            b = ground(gpu, h, w, 90 + i)
            d = np.zeros((h, w), F32)
            d[h // 2:h // 2 + 3, w // 3] = 5.0
            rain = (0.7 * w, 0.2 * h, 1e-2, 20.0) if i % 2 else None
            batch.upload(gid, b, d)
            if rain:
                batch.set_rain(gid, *rain)
            state[gid] = [b, d, None, rain]
        for turn in range(2):
            for gid in state:
                batch.set_steps(gid, 21 + 5 * (gid % 3))
            batch.run()
            for gid, st in state.items():
                st[1], st[2], _ = oracle.step(st[0], st[1], st[2], *c, n=21 + 5 * (gid % 3),
                                              rain=st[3])
                out = batch.download(gid)
                assert same_bits(out["depth"], st[1]), (turn, gid)
                assert same_bits(out["flux"], st[2]), (turn, gid)


# sides below 16 and 32 (nothing is updated, nothing rained on), multiples of 16
# and not, tails inside one tile and just past a tile's output
@pytest.mark.parametrize("shape", [(15, 300), (300, 31), (16, 16), (97, 113), (176, 240),
                                   (479, 331), (700, 1000)])
@pytest.mark.parametrize("kernel,k", [(0, 0), (2, 4), (3, 5), (4, 6), (5, 4), (6, 8), (7, 3), (8, 6)])
def test_truncated_dispatch_bitwise(gpu, oracle, shape, kernel, k):
    H, W = shape
    rng = np.random.default_rng(H * 7 + W)
    b = (rng.random((H, W)) * 4.0).astype(F32)
    d = (rng.random((H, W)) * 2.0).astype(F32)
    f = (rng.random((H, W, 4)) * 0.3).astype(F32)
    d[-1, -3:] = F32(-0.0)
    for rain in (None, (W - 10.0, H - 12.0, 1e-2, 900.0)):
        check(gpu, oracle, b, d, f, rain, kernel, k, D, (13, 5))
