"""1x1 convolutions that take their operand straight from the pixels, bit for bit against the
oracle: planes from one pixel up that end anywhere in a 32- or 64-pixel tile, channels at the edges of
the 16-channel loads and the 32-channel steps, one step and several, output channels at the edges
of the row tiles, the forms of one to three row tiles a wave, of one and two pixels a lane and of one,
two and four waves an output tile, outputs on a y pattern, biases, RELU and RELU6, both output
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
    (1, 640, 5, 13, 70), (3, 16, 1, 1, 16), (2, 1, 3, 1, 3), (16, 9, 64, 64, 150), (16, 17, 64, 64, 64), (2, 34, 64, 64, 33),
    (8, 72, 56, 56, 40), (8, 65, 33, 33, 128), (5, 100, 33, 33, 100), (1, 2048, 7, 7, 100), (3, 1025, 2, 2, 40)])
def test_conv_point(U, oracle_lib, batch, in_ch, h, w, out_ch, act, wrap, lim):
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


@pytest.mark.parametrize("in_ch", [24, 96])
@pytest.mark.parametrize("h,w", [(9, 7), (10, 6)])
def test_conv_point_y_pattern(U, oracle_lib, in_ch, h, w):
    """Output channel o of an image at (o % 4) cs + (o / 4) gs."""
    from cormorant_amd.packing import conv_weight_image
    rng = np.random.default_rng(in_ch + h)
    batch, out_ch, plane = 1, 40, h * w
    cs, cn, gs = 10 * (plane + 3), 4, plane + 3
    x = rng.integers(-2000, 2000, batch * in_ch * plane).astype(np.int16)
    img = np.asarray(conv_weight_image(rng.integers(-2000, 2000, (out_ch, in_ch, 1, 1)).astype(np.int16), False)).reshape(-1)
    want = oracle_lib.conv(x, img, None, out_ch * plane, batch, in_ch, h, w, out_ch, h, w, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0)
    y = poisoned16(40 * (plane + 3) + 8)
    U.conv_planes(dev16(x, extra=0), U.conv_w_planes(dev16(img), out_ch, in_ch, 1, 1), None, y, batch, in_ch, h, w, out_ch,
                  h, w, 1, 1, y_cs=cs, y_cn=cn, y_gs=gs)
    full = np.full(40 * (plane + 3) + 8, 0x5A5A, np.int16)
    for o in range(out_ch):
        at = (o % cn) * cs + (o // cn) * gs
        full[at:at + plane] = want[o * plane:(o + 1) * plane]
    np.testing.assert_array_equal(host(y), full)


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


def test_shared_weight_keeps_both_images(U, oracle_lib, monkeypatch):
    """One weight read by a pointwise and by a stride-2 node of few taps, in either order: the one on the
    matrix units, the other on its few-tap path."""
    from cormorant_amd import units
    from cormorant_amd.graph import ConvNode, Graph, TensorInfo
    from cormorant_amd.packing import conv_weight_image
    from cormorant_amd.simulate import Simulator
    rng = np.random.default_rng(3)
    x = TensorInfo("x", [2, 24, 6, 6])
    w = TensorInfo("w", [40, 24, 1, 1], data=rng.integers(-300, 300, (40, 24, 1, 1)) / 256.0)
    nodes = [ConvNode([x, w], TensorInfo("a", [2, 40, 6, 6])),
             ConvNode([x, w], TensorInfo("b", [2, 40, 3, 3]), stride_h=2, stride_w=2)]
    xr = rng.integers(-3000, 3000, x.numel).astype(np.int16)
    img = np.asarray(conv_weight_image((w.data * 256).astype(np.int16), False)).reshape(-1)
    want = {nd.output.onnx_name: oracle_lib.conv(xr, img, None, nd.output.numel, 2, 24, 6, 6, 40, nd.out_h, nd.out_w, 1, 1,
                                                 nd.stride_h, nd.stride_w, 1, 1, 0, 0, 0, 0) for nd in nodes}
    calls = []
    for name in ("conv", "conv_planes"):
        fn = getattr(units, name)
        monkeypatch.setattr(units, name, lambda *a, fn=fn, name=name, **k: (calls.append(name), fn(*a, **k))[1])
    for order in (nodes, nodes[::-1]):
        calls.clear()
        got = Simulator(Graph(nodes=list(order), input_tensors=[x], output_tensors=[n.output for n in order])).forward_raw(
            {"x": dev16(xr, extra=0)})
        assert calls == ["conv_planes" if nd is nodes[0] else "conv" for nd in order]
        for k, v in want.items():
            np.testing.assert_array_equal(host(got[k]).reshape(-1), v)


def test_no_workspace(U, oracle_lib):
    """Captured before any other call of its size (the workspace cannot grow during a capture): a 1x1
    convolution from its pixels has no planes of its input (412 MB of them here) to put there."""
    import torch
    rng = np.random.default_rng(11)
    batch, h, out_ch = 64, 224, 3
    n = batch * out_ch * h * h
    x = rng.integers(-3000, 3000, batch * h * h).astype(np.int16)
    from cormorant_amd.packing import conv_weight_image
    img = np.asarray(conv_weight_image(rng.integers(-3000, 3000, (out_ch, 1, 1, 1)).astype(np.int16), False)).reshape(-1)
    want = oracle_lib.conv(x, img, None, n, batch, 1, h, h, out_ch, h, h, 1, 1, 1, 1, 1, 1, 0, 0, 0, 0)
    planes, dx, y = U.conv_w_planes(dev16(img), out_ch, 1, 1, 1), dev16(x, extra=0), poisoned16(n)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        U.conv_planes(dx, planes, None, y, batch, 1, h, h, out_ch, h, h, 1, 1)
    for _ in range(2):
        y.fill_(0x5A5A)
        graph.replay()
        np.testing.assert_array_equal(host(y), want)
