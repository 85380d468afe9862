"""The depthwise 3x3 kernels of strides 1 and 2, bit for bit against the oracle: few planes (a strip of one
column a lane) and as many as take the lanes of 8 input columns, rows that end anywhere in a lane's
columns, output rows past its strip, planes too small for its words, one plane and many (the words
beyond a plane's ends belong to its neighbours), paddings up to one past the kernel, both strides, both
output rules, activations, weights past the int32 bound, outputs on a y pattern."""
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


def _past_strips(batch, ch, w, oh, ow, stride):
    """The least channel count of at least ``ch`` past the lanes of the strip kernel (a lane one column of 8
    output rows, 4 at stride 2): 256 a compute unit, more over rows of at most 3 columns (over rows of 4 at
    stride 1 and planes of 5 x 5 there is no such count: many of its lanes)."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    most = (1200 if stride == 1 else 512) if w <= 3 else 256
    return max(ch, most * cus // (batch * -(-oh // (8 if stride == 1 else 4)) * ow) + 1)


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("act,wrap,lim", [(0, 0, 32768), (2, 0, 3000), (1, 1, 32768)])
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("batch,ch,h,w,pt,pl,pb,pr", [
    (1, 1, 1, 1, 1, 1, 1, 1), (1, 3, 2, 2, 1, 1, 1, 1), (2, 5, 3, 3, 0, 0, 0, 0), (1, 2, 3, 9, 1, 0, 0, 1),
    (2, 7, 7, 7, 1, 1, 1, 1), (1, 4, 14, 14, 1, 1, 1, 1), (3, 2, 15, 8, 0, 1, 1, 0), (1, 3, 9, 17, 2, 2, 2, 2),
    (1, 2, 8, 16, 1, 1, 1, 1), (1, 3, 6, 13, 2, 1, 2, 3), (2, 3, 28, 28, 1, 1, 1, 1), (1, 2, 56, 40, 0, 0, 1, 1), (1, 2, 5, 6, 3, 4, 3, 4), (1, 1, 4, 33, 1, 12, 1, 12)])
def test_dw3(U, oracle_lib, batch, ch, h, w, pt, pl, pb, pr, stride, act, wrap, lim, many):
    from cormorant_amd.packing import conv_weight_image
    oh, ow = (h + pt + pb - 3) // stride + 1, (w + pl + pr - 3) // stride + 1
    if many:
        ch = _past_strips(batch, ch, w, oh, ow, stride)
    rng = np.random.default_rng(ch + 7 * h + w + act + stride)
    x = rng.integers(-lim, lim, batch * ch * h * w).astype(np.int16)
    wt = rng.integers(-lim, lim, (ch, 1, 3, 3)).astype(np.int16)
    img = np.asarray(conv_weight_image(wt, True)).reshape(-1)
    bias = rng.integers(-300, 300, ch).astype(np.int16)
    n = batch * ch * oh * ow
    want = oracle_lib.conv(x, img, bias, n, batch, ch, h, w, ch, oh, ow, 3, 3, stride, stride, 1, 1, pt, pl, 1, 1, wrap32=bool(wrap))
    if act:
        want = np.clip(want, 0, 32767 if act == 1 else 6 << 8)
    y = poisoned16(n + 8)
    U.conv(dev16(x, extra=0), dev16(img), dev16(bias), y, batch, ch, h, w, ch, oh, ow, 3, 3, stride, stride, 1, 1, pt, pl,
           has_bias=1, is_depthwise=1, wrap32=bool(wrap), act=act)
    got = host(y)
    np.testing.assert_array_equal(got[:n], want)
    assert (got[n:] == 0x5A5A).all()


@pytest.mark.parametrize("many", [False, True])
@pytest.mark.parametrize("h,w", [(9, 7), (10, 16)])
def test_dw3_y_pattern(U, oracle_lib, h, w, many):
    """Output channel o at (o % 2) cs + (o / 2) gs."""
    from cormorant_amd.packing import conv_weight_image
    rng = np.random.default_rng(w)
    ch = _past_strips(1, 6, w, h, w, 1) + 1 & ~1 if many else 6
    plane = h * w
    cs, cn, gs = ch // 2 * (plane + 5), 2, plane + 5
    x = rng.integers(-2000, 2000, ch * plane).astype(np.int16)
    img = np.asarray(conv_weight_image(rng.integers(-2000, 2000, (ch, 1, 3, 3)).astype(np.int16), True)).reshape(-1)
    want = oracle_lib.conv(x, img, None, ch * plane, 1, ch, h, w, ch, h, w, 3, 3, 1, 1, 1, 1, 1, 1, 0, 1)
    y = poisoned16(ch * (plane + 5) + 8)
    U.conv(dev16(x, extra=0), dev16(img), None, y, 1, ch, h, w, ch, h, w, 3, 3, 1, 1, 1, 1, 1, 1, is_depthwise=1, y_cs=cs,
           y_cn=cn, y_gs=gs)
    full = np.full(ch * (plane + 5) + 8, 0x5A5A, np.int16)
    for o in range(ch):
        at = (o % cn) * cs + (o // cn) * gs
        full[at:at + plane] = want[o * plane:(o + 1) * plane]
    np.testing.assert_array_equal(host(y), full)
