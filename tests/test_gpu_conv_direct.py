"""1x1 convolutions whose workgroups split their own input (at most 512 output channels), bit for bit
against the oracle: planes from 4 pixels up that end anywhere in a 64-pixel tile and in a group of
4, channels at the edges of a 64-channel step and of the 16-channel weight tiles, one step and
several, output channels at the edges of the row tiles and past 512, biases, RELU and RELU6, both output
rules, full-range operands; the graph's choice of it over the few-tap path."""
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


@pytest.mark.parametrize("act,wrap,lim", [(0, 0, 32768), (2, 0, 3000), (1, 1, 32768)])
@pytest.mark.parametrize("batch,in_ch,h,w,out_ch", [
    (1, 8, 2, 2, 5), (3, 16, 1, 5, 64), (2, 63, 3, 3, 65), (1, 64, 7, 9, 17), (5, 65, 7, 7, 96), (2, 128, 8, 8, 64),
    (3, 129, 13, 5, 130), (2, 200, 14, 14, 33), (1, 320, 11, 11, 512), (2, 33, 9, 7, 520), (4, 96, 16, 12, 48),
    (1, 640, 5, 13, 70)])
def test_conv_direct(U, oracle_lib, batch, in_ch, h, w, out_ch, act, wrap, lim):
    from cormorant_amd.packing import conv_weight_image
    rng = np.random.default_rng(batch + in_ch + 7 * h + out_ch + act)
    x = rng.integers(-lim, lim, batch * in_ch * h * w).astype(np.int16)
    wt = rng.integers(-lim, lim, (out_ch, in_ch, 1, 1)).astype(np.int16)
    img = np.asarray(conv_weight_image(wt, False)).reshape(-1)
    bias = rng.integers(-300, 300, out_ch).astype(np.int16)
    n = batch * out_ch * h * w
    want = oracle_lib.conv(x, img, bias, n, batch, in_ch, h, w, out_ch, h, w, 1, 1, 1, 1, 1, 1, 0, 0, 1, 0, wrap32=bool(wrap))
    if act:
        want = np.clip(want, 0, 32767 if act == 1 else 6 << 8)
    planes = U.conv_w_planes(dev16(img), out_ch, in_ch, 1, 1)
    y = poisoned16(n + 8)
    U.conv_planes(dev16(x, extra=0), planes, dev16(bias), y, batch, in_ch, h, w, out_ch, h, w, 1, 1, has_bias=1,
                  wrap32=bool(wrap), act=act)
    got = host(y)
    np.testing.assert_array_equal(got[:n], want)
    assert (got[n:] == 0x5A5A).all()


@pytest.mark.parametrize("batch,hw", [(1, 6), (32, 33)])
def test_graph_pointwise(U, batch, hw):
    from cormorant_amd import graph as G
    from cormorant_amd.simulate import Simulator
    from oracle import graph_sim
    rng = np.random.default_rng(hw)
    x = G.TensorInfo("x", [batch, 24, hw, hw])
    w = G.TensorInfo("w", [40, 24, 1, 1], data=rng.uniform(-0.4, 0.4, (40, 24, 1, 1)))
    y = G.TensorInfo("y", [batch, 40, hw, hw])
    g = G.Graph([G.ConvNode([x, w], y)], [x], [y])
    feeds = {"x": np.round(rng.uniform(-4, 4, (batch, 24, hw, hw)) * 256) / 256}
    np.testing.assert_array_equal(Simulator(g).simulate(feeds)["y"], graph_sim.forward(g, feeds)["y"])
