"""The blocks the mip chain is made in: sides that leave a texel over at every
level, that end just before and after a block, and chains of 1, 2, 3 and more
than 4 levels; bit for bit against the restatement."""
import numpy as np
import pytest
from test_mips import rgba

pytestmark = pytest.mark.gpu

F32 = np.float32


@pytest.mark.parametrize("W,H", [(2, 1), (3, 3), (5, 2), (9, 15), (63, 64), (65, 127), (511, 513),
                                 (1023, 77), (129, 4099), (2047, 31), (1, 700), (960, 1056)])
@pytest.mark.parametrize("fill", [0.3, -0.0])
def test_mip_blocks_bitwise(gpu, oracle, W, H, fill):
    rng = np.random.default_rng(W * 5 + H)
    b = (rng.random((H, W)) * 40.0).astype(F32)
    d = (rng.random((H, W)) * 2.0 * (rng.random((H, W)) < 0.6)).astype(F32)
    with gpu.Simulation(W, H) as s:
        s.upload(b, d)
        ours = s.mips(fill)
    level0 = rgba(b, d)
    level0[..., 1:3] = F32(fill)
    want = oracle.mips(level0)
    assert len(ours) == len(want)
    for level, (a, w) in enumerate(zip(ours, want), 1):
        assert a.shape == w.shape
        assert np.array_equal(a.view(np.uint32), w.view(np.uint32)), level
