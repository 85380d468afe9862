"""The plane GEMM on its ring of LDS stages and the block order of its tiles, bit for bit against
the oracle: from one k step to past a turn of the ring and its remainders, outputs at the edges of
the 64 x 64, 128 x 128 and 256 x 128 tiles, odd widths, every size at which the choice of the tile
changes (64 rows, two workgroups a unit, one a unit, rounds of 256-row tiles), batches, splits over
k of one and several steps, both output rules."""
import numpy as np
import pytest

from gpu_util import dev16, host, poisoned16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def U():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cormorant_amd import units
    units.init()
    return units


SHAPES = [(33, 64 * s, 65, 1) for s in range(1, 11)] + [(130, 64 * s - 24, 66, 2) for s in (1, 2, 3, 4, 5, 9)] + [
    (63, 200, 64, 1), (64, 200, 63, 1), (65, 200, 129, 3), (128, 768, 127, 1), (127, 771, 130, 1),
    (40, 72, 33000, 1),                                   # at most 64 rows, more tiles than slots
    (2048, 136, 1024, 1), (2049, 136, 1024, 1),           # 512 tiles of 64 x 64, then one row more
    (2048, 72, 2048, 1), (2048, 72, 2049, 1),             # 256 tiles of 128 x 128, then past one a unit
    (2050, 72, 4100, 1), (513, 72, 2050, 5),              # rounds of 256-row tiles, a batch
    (64, 1600, 72, 1), (300, 2500, 200, 1), (2100, 2560, 1100, 1),   # wrap products split over k
    (1100, 3100, 1050, 1), (1500, 3100, 1000, 1),         # past 48 steps: 128 x 128 tiles on the ring in 3, two stages in 5
    (330, 6500, 1025, 2), (1270, 1500, 2040, 1),          # the ring in 4 of 26 steps; two stages in 3 of 8
    (600, 500, 8100, 1), (1024, 300, 8190, 1)]            # at most 8 steps: 128-row tiles, one round of 256-row ones


@pytest.mark.parametrize("wrap", [0, 1])
@pytest.mark.parametrize("n,k,m,batch", SHAPES)
def test_matmul_tiles(U, oracle_lib, n, k, m, batch, wrap):
    rng = np.random.default_rng(n + 3 * k + 5 * m + wrap)
    lim = 32768 if wrap else 3000
    a = rng.integers(-lim, lim, batch * n * k).astype(np.int16)
    b = rng.integers(-lim, lim, k * m).astype(np.int16)
    want = oracle_lib.matmul(a, b, n, k, m, batch, n * k, 0, n * m, 0, 0, wrap)
    c = poisoned16(batch * n * m + 8)
    U.matmul(dev16(a), dev16(b), c, n, k, m, batch=batch, a_bs=n * k, wrap32=bool(wrap))
    got = host(c)
    np.testing.assert_array_equal(got[:batch * n * m], np.asarray(want).reshape(-1))
    assert (got[batch * n * m:] == 0x5A5A).all()
