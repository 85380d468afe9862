"""NORM and the residual add at the edges of their short arithmetic, bit for bit against the oracle:
row magnitudes on both sides of the short sums' bound (2^21 .. 2^23 and far past it), one row short
and the next long in one call, output shifts on both sides of 32 / 33 and at 61, ties, both signs of
saturation; residual adds with and without the plain form (shifts, biases past 2^30
and shifted past the staged form's 40, RELU)."""
import numpy as np
import pytest

from gpu_util import dev8, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def U():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cormorant_amd import units
    units.init()
    return units


def _params(rng, n, sc_lo, sc_hi, sa=0, sb=0, bq=1 << 20):
    from cormorant_amd.rowops_nodes import param_block
    return np.ascontiguousarray(param_block(rng.integers(1 << 20, 1 << 30, n), rng.integers(-bq, bq, n), np.full(n, sa),
                                            np.full(n, sb), rng.integers(sc_lo, sc_hi + 1, n)), np.uint8).reshape(-1)


def _run(U, lib, jobs, out_bytes):
    """The jobs through cm_rowops_chain and one by one through the oracle: every output byte."""
    import torch
    d = [torch.full((nb,), 0x5A, dtype=torch.uint8, device="cuda") for nb in out_bytes]
    h = [np.full(nb, 0x5A, np.uint8) for nb in out_bytes]
    dj, prev_d, prev_h = [], None, None
    for i, j in enumerate(jobs):
        a, b, p = j.pop("a"), j.pop("b"), j.pop("p")
        dj.append(dict(j, a=dev8(a) if a is not None else prev_d, b=dev8(b) if b is not None else None, c=d[i], p=dev8(p)))
        lib.rowops(a if a is not None else prev_h, b, h[i], p, j["op"], j["n"], j["c1"], 1, j["a_s1"], 0, j["b_s1"], 0,
                   j["c_s1"], 0, eps=j.get("eps", 0), bq_sh=j.get("bq_sh", 0))
        prev_d, prev_h = d[i], h[i]
    U.rowops_jobs(dj)
    for x, y in zip(d, h):
        np.testing.assert_array_equal(host(x), y)


@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("rows,n,mag,sc", [
    (7, 768, 1 << 20, (34, 43)), (300, 768, (1 << 23) - 1, (33, 33)), (300, 512, 1 << 23, (40, 40)), (9, 520, 1 << 24, (36, 40)),
    (20, 2048, (1 << 21) - 1, (33, 61)), (20, 2304, 1 << 22, (38, 39)), (5, 4096, (1 << 31) - 1, (44, 50)),
    (40, 768, 1 << 18, (30, 34)), (33, 768, 1 << 18, (32, 32)), (300, 64, 5, (33, 40)), (16, 960, 1 << 12, (62, 63)),
    (300, 1024, 1 << 31, (44, 50)), (5, 4096, 1 << 31, (44, 50)), (5, 2048, 1 << 31, (44, 50))])     # a row of -2^31
def test_norm_magnitudes(U, oracle_lib, rows, n, mag, sc, rms):
    from cormorant_amd import rowops_nodes as rn
    rng = np.random.default_rng(rows + n + sc[0])
    x = rng.integers(-mag, mag + 1, (rows, n), dtype=np.int64)
    x[rows // 2] = rng.integers(-30, 30, n)                      # a short row among long ones
    x[rows - 1, :] = mag
    x = x.astype(np.int32)
    op = rn.opword(rn.RO_NORM, rn.K_I32, rn.K_I16, rn.K_I16) | (0 if rms else U.F_NORM_LN)
    _run(U, oracle_lib, [dict(a=x.reshape(-1).view(np.uint8), b=None, p=_params(rng, n, *sc), op=op, n=n, c1=rows, c2=1,
                              a_s1=4 * n, a_s2=0, b_s1=0, b_s2=0, c_s1=2 * n, c_s2=0, eps=1 << 20)], [rows * n * 2])


@pytest.mark.parametrize("rows,n,sa,sb,sc,bq,bq_sh,relu", [
    (300, 768, 0, 2, 0, 1 << 20, 5, False), (20, 768, 0, 15, 0, 1 << 18, 12, True), (300, 512, 0, 3, 0, 1 << 21, 11, False),
    (300, 768, 0, 16, 0, 1 << 10, 0, False), (9, 256, 1, 2, 0, 1 << 12, 0, False), (9, 256, 0, 2, 1, 1 << 12, 3, True),
    (3100, 768, 0, 4, 0, 1 << 16, 0, False), (9, 256, 0, 2, 0, 1 << 21, 40, False), (20, 512, 0, 2, 0, 3, 41, True)])
def test_residual_add_then_norm(U, oracle_lib, rows, n, sa, sb, sc, bq, bq_sh, relu):
    from cormorant_amd import rowops_nodes as rn
    rng = np.random.default_rng(rows + n + sb)
    x = rng.integers(-2 ** 31, 2 ** 31, (rows, n), dtype=np.int64).astype(np.int32)
    x[rows // 3:] >>= 10
    y = rng.integers(-32768, 32768, (rows, n)).astype(np.int16)
    op1 = rn.opword(rn.RO_ADDX, rn.K_I32, rn.K_I16, rn.K_I32, b_en=True) | (U.F_RELU if relu else 0)
    op2 = rn.opword(rn.RO_NORM, rn.K_I32, rn.K_I16, rn.K_I16) | U.F_NORM_LN
    p1 = _params(rng, n, sc, sc, sa, sb, bq)
    _run(U, oracle_lib, [dict(a=x.reshape(-1).view(np.uint8), b=y.reshape(-1).view(np.uint8), p=p1, op=op1, n=n, c1=rows, c2=1,
                              a_s1=4 * n, a_s2=0, b_s1=2 * n, b_s2=0, c_s1=4 * n, c_s2=0, bq_sh=bq_sh),
                         dict(a=None, b=None, p=_params(rng, n, 36, 44), op=op2, n=n, c1=rows, c2=1, a_s1=4 * n, a_s2=0,
                              b_s1=0, b_s2=0, c_s1=2 * n, c_s2=0, eps=1 << 12)], [rows * n * 4, rows * n * 2])
