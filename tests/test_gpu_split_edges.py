"""The operand splits at any element alignment, width and row length, bit for bit against the
oracle: operands that start 1 .. 7 elements past a 16-byte word, odd k and batch strides, every B
image at the edges of its 8-column and 32-column groups (fewer than 8 columns too), k at the edges
of a wavefront's 256 and a slab's 1024; the im2col split over channel remainders, strides,
dilation, asymmetric padding, several slabs of k and odd planes."""
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


def _image(b, k, m, layout):
    from cormorant_amd.packing import pack_matmul_b
    if layout == "packed":
        return np.asarray(pack_matmul_b(b.reshape(k, m))).reshape(-1)
    if layout == "trans":
        return np.ascontiguousarray(b.reshape(k, m).T).reshape(-1)
    return b


@pytest.mark.parametrize("layout", ["row", "packed", "gemv", "trans"])
@pytest.mark.parametrize("n,k,m,batch,ao,bo", [
    (35, 7, 5, 1, 1, 3), (33, 65, 8, 2, 3, 1), (40, 255, 9, 1, 0, 5), (70, 256, 31, 2, 7, 2), (34, 257, 33, 1, 2, 7),
    (50, 771, 63, 3, 5, 0), (36, 1023, 65, 1, 0, 1), (37, 1024, 39, 2, 6, 4), (65, 1025, 71, 1, 4, 6),
    (33, 1311, 127, 1, 1, 1), (129, 2049, 130, 1, 3, 3), (48, 80, 1, 1, 0, 0)])
def test_matmul_any_alignment(U, oracle_lib, n, k, m, batch, ao, bo, layout):
    if layout == "gemv":
        k = max(16, k // 16 * 16)
    rng = np.random.default_rng(n + k + m + len(layout))
    a_bs = n * k + (3 if batch > 1 else 0)
    a = rng.integers(-32768, 32768, (batch - 1) * a_bs + n * k).astype(np.int16)
    b = rng.integers(-32768, 32768, k * m).astype(np.int16)
    wide = np.zeros(batch * a_bs, np.int16)
    wide[:a.size] = a
    img = _image(b, k, m, layout)
    want = [oracle_lib.matmul(np.ascontiguousarray(wide[i * a_bs:i * a_bs + n * k]), b, n, k, m, 1, 0, 0, n * m, 0, 0, 1)
            for i in range(batch)]
    da = dev16(np.concatenate([np.full(ao, 77, np.int16), a]))[ao:]
    db = dev16(np.concatenate([np.full(bo, 77, np.int16), img]))[bo:]
    c = poisoned16(batch * n * m + 8)
    U.matmul(da, db, c, n, k, m, batch=batch, a_bs=a_bs if batch > 1 else 0, b_packed={"packed": 1, "trans": 2}.get(layout, 0),
             gemv_kw=1 if layout == "gemv" else 0, wrap32=True)
    got = host(c)
    np.testing.assert_array_equal(got[:batch * n * m], np.concatenate([np.asarray(w).reshape(-1) for w in want]))
    assert (got[batch * n * m:] == 0x5A5A).all()


@pytest.mark.parametrize("batch,in_ch,h,w,out_ch,kh,kw,sh,sw,dh,dw,pt,pl", [
    (2, 16, 9, 11, 33, 3, 3, 1, 1, 1, 1, 1, 1), (1, 20, 15, 14, 40, 3, 3, 2, 1, 1, 1, 0, 1),
    (3, 41, 7, 7, 20, 5, 3, 1, 2, 1, 1, 2, 0), (1, 64, 17, 19, 65, 3, 3, 1, 1, 2, 2, 2, 2),
    (2, 9, 12, 13, 70, 7, 7, 2, 2, 1, 1, 3, 3), (1, 130, 8, 9, 17, 3, 3, 1, 1, 1, 1, 1, 0),
    (2, 100, 6, 5, 48, 1, 1, 2, 2, 1, 1, 0, 0), (1, 24, 40, 41, 64, 3, 5, 1, 1, 1, 3, 4, 5)])
def test_conv_im2col(U, oracle_lib, batch, in_ch, h, w, out_ch, kh, kw, sh, sw, dh, dw, pt, pl):
    from cormorant_amd.packing import conv_weight_image
    rng = np.random.default_rng(in_ch + h + out_ch)
    oh, ow = (h + 2 * pt - dh * (kh - 1) - 1) // sh + 1, (w + pl - dw * (kw - 1) - 1) // sw + 1
    x = rng.integers(-4096, 4096, batch * in_ch * h * w).astype(np.int16)
    wt = rng.integers(-400, 400, (out_ch, in_ch, kh, kw)).astype(np.int16)
    img = np.asarray(conv_weight_image(wt, False)).reshape(-1)
    bias = rng.integers(-300, 300, out_ch).astype(np.int16)
    want = oracle_lib.conv(x, img, bias, batch * out_ch * oh * ow, batch, in_ch, h, w, out_ch, oh, ow, kh, kw, sh, sw, dh,
                           dw, pt, pl, 1, 0)
    y = poisoned16(batch * out_ch * oh * ow + 8)
    U.conv(dev16(x), dev16(img), dev16(bias), y, batch, in_ch, h, w, out_ch, oh, ow, kh, kw, sh, sw, dh, dw, pt, pl,
           has_bias=1)
    got = host(y)
    np.testing.assert_array_equal(got[:batch * out_ch * oh * ow], np.asarray(want).reshape(-1))
    assert (got[batch * out_ch * oh * ow:] == 0x5A5A).all()
