"""cm_attention_strided bit for bit against the oracle's chain (q.K^T by the int32-wrap rule, the
keys-major softmax with its mask register, P.V): an encoder's rows in place at lengths on both
sides of a wavefront's 64-key step and of each instance's 256 keys, with o's byte planes; a
prompt's queries in the q.K^T image over group-major caches, causal from several positions and
with a fixed valid count; every register pair.  Then the graphs that take it: a prompt whose
scores nobody reads equals the node-by-node pass, and an encoder of an odd length the oracle's."""
import numpy as np
import pytest

from gpu_util import POISON16, dev16, host, poisoned16
from test_gpu_random import _attention_regs, rint16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def U():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from cormorant_amd import units
    units.init()
    return units


def _chain(lib, Q, K, V, cm, cfg, mask):
    nq, keys, hd = Q.shape[0], K.shape[0], Q.shape[1]
    s = lib.matmul(np.ascontiguousarray(K).ravel(), np.ascontiguousarray(Q.T).ravel(), keys, hd, nq, 1, 0, 0, keys * nq, 0,
                   0, True)
    kp = (keys + 7) & ~7
    p = lib.vectorop(s, None, nq * kp, keys, 11, nq, nq, kp, 0, 0, cm, cfg, mask)
    return lib.matmul(np.ascontiguousarray(p.reshape(nq, kp)[:, :keys]).ravel(), np.ascontiguousarray(V).ravel(), nq, keys,
                      hd, 1, 0, 0, nq * hd, 0, 0, True).reshape(nq, hd)


@pytest.mark.parametrize("B,T,H,regs,lim", [
    (1, 16, 1, 0, 32768), (2, 48, 3, 1, 4000), (1, 64, 2, 2, 32768), (1, 80, 2, 3, 2000), (3, 208, 2, 0, 3000),
    (1, 256, 1, 1, 32768), (1, 272, 2, 2, 3000), (1, 512, 1, 3, 32768), (1, 528, 1, 0, 1500), (1, 784, 1, 1, 3000),
    (1, 1024, 1, 2, 2500)])
def test_encoder_rows(U, oracle_lib, B, T, H, regs, lim):
    cm, cfg = _attention_regs()[regs]
    rng = np.random.default_rng(T * 10 + H + regs)
    D = 64 * H
    ld = 3 * D + 8
    offs = (8, 8 + D, 8 + 2 * D)
    x = rint16(rng, B * T * ld, -lim, lim).reshape(B * T, ld)
    want = np.empty((B * T, D), np.int16)
    for b in range(B):
        rows = x[b * T:(b + 1) * T]
        for h in range(H):
            Q, K, V = (rows[:, o + 64 * h:o + 64 * h + 64] for o in offs)
            want[b * T:(b + 1) * T, 64 * h:64 * h + 64] = _chain(oracle_lib, Q, K, V, cm, cfg, T)
    out = poisoned16(B * T * D + 8)
    planes = U.a_planes(B * T, D, H, "cuda")
    views = [(o, ld, T * ld, 64) for o in offs]
    d = dev16(x.ravel())
    U.attention_strided(d, d, d, out, T, T, B * H, H, *views, (0, D, T * D, 64), cm, cfg, T, planes=planes,
                        planes_rows=B * T)
    got = host(out)
    np.testing.assert_array_equal(got[:B * T * D].reshape(B * T, D), want)
    assert (got[B * T * D:] == POISON16).all()
    lines = (B * T + 255) // 256 * 256
    p = host(planes)
    w32 = want.astype(np.int32)
    np.testing.assert_array_equal(p[:lines * D].reshape(lines, D)[:B * T], ((w32 >> 8) & 0xFF).astype(np.uint8))
    np.testing.assert_array_equal(p[lines * D:2 * lines * D].reshape(lines, D)[:B * T], ((w32 & 0xFF) ^ 0x80).astype(np.uint8))
    sums = p[2 * lines * D:2 * lines * D + 4 * H * lines].view(np.int32).reshape(H, lines)[:, :B * T]
    np.testing.assert_array_equal(sums, w32.reshape(B * T, H, 64).sum(axis=2).T)


@pytest.mark.parametrize("KV,G,T,C,keys,mask,regs,lim", [
    (2, 3, 16, 64, 16, 1 | 16 << 16, 0, 3000), (1, 3, 32, 128, 64, 37 | 32 << 16, 1, 32768),
    (3, 1, 48, 320, 304, 250 | 48 << 16, 2, 3000), (2, 2, 64, 640, 592, 529 | 64 << 16, 3, 4000),
    (1, 2, 16, 1024, 1024, 1009 | 16 << 16, 0, 2000), (2, 2, 32, 96, 48, 39, 1, 3000), (1, 1, 32, 64, 64, 0, 0, 3000),
    (1, 2, 32, 128, 128, 500, 2, 32768)])
def test_prompt_over_caches(U, oracle_lib, KV, G, T, C, keys, mask, regs, lim):
    cm, cfg = _attention_regs()[regs]
    rng = np.random.default_rng(KV + 10 * G + T + C + keys)
    H = KV * G
    qx = rint16(rng, KV * 64 * G * T, -lim, lim).reshape(KV, 64, G * T)
    kc, vc = (rint16(rng, KV * C * 64, -lim, lim).reshape(KV, C, 64) for _ in range(2))
    want = np.empty((T, H * 64), np.int16)
    for h in range(H):
        kv, hp = divmod(h, G)
        want[:, 64 * h:64 * h + 64] = _chain(oracle_lib, qx[kv][:, hp * T:(hp + 1) * T].T, kc[kv, :keys], vc[kv, :keys], cm,
                                             cfg, mask)
    out = poisoned16(T * H * 64)
    cache = (0, 64, C * 64, 0)
    U.attention_strided(dev16(qx.ravel()), dev16(kc.ravel()), dev16(vc.ravel()), out, T, keys, H, G, (0, 1, 64 * G * T, T),
                        cache, cache, (0, H * 64, G * 64, 64), cm, cfg, mask, q_ds=G * T)
    np.testing.assert_array_equal(host(out).reshape(T, H * 64), want)


@pytest.mark.parametrize("T,n,pos", [(32, 32, 0), (64, 50, 37), (16, 9, 100)])
def test_prompt_graph_without_scores(U, T, n, pos):
    """Two layers over their caches, only the results kept: the chain in one launch gives the
    states of the pass that materializes every tensor."""
    from cormorant_amd import models
    from cormorant_amd.simulate import Simulator
    S = models.LlamaShape(layers=2, batch=1, d=256, heads=4, kv=2, hd=64, ff=256, vocab=512, ctx=128)
    w = models.smollm2_weights(S, 5)
    _, _, exps = models.smollm2_decode(S, seed=5, weights=w)
    pg = models.smollm2_prefill(S, T, exps, w)
    rng = np.random.default_rng(T + pos)
    feeds = {"ids": rng.integers(0, S.vocab, T).astype(float), "pos": np.array([pos]), "n": np.array([n])}
    st = {t.onnx_name: rng.integers(-3000, 3000, t.shape) / 2.0 ** float(np.max(t.exp)) if t.exp is not None else
          np.zeros(t.shape) for t in pg.state_tensors}
    full, lean = ({k: v.copy() for k, v in st.items()} for _ in range(2))
    sim = Simulator(pg)
    sim._forward_pass(feeds, states=full)
    sim._forward_pass(feeds, states=lean, keep=[])
    assert sim._attn_chain(next(i for i, nd in enumerate(pg.nodes) if type(nd).__name__ == "LlmAttnConvNode")) is not None
    for k in full:
        np.testing.assert_array_equal(lean[k], full[k], err_msg=k)


@pytest.mark.parametrize("batch,seq", [(3, 80), (1, 272)])
def test_encoder_odd_length(U, batch, seq):
    from cormorant_amd import models
    from cormorant_amd.simulate import Simulator
    from oracle import graph_sim
    g, inputs, _ = models.bert_encoder(models.BertShape(layers=1, batch=batch, seq=seq, d=128, heads=2, ff=256, vocab=64))
    want = graph_sim.forward(g, inputs)
    got = Simulator(g)._forward_pass(inputs)
    for name, v in got.items():
        np.testing.assert_array_equal(v, want[name].reshape(v.shape), err_msg=name)


def _off_word(t):
    """The same values in a buffer that starts two bytes past a 16-byte word."""
    import torch
    v = torch.empty(t.numel() + 8, dtype=t.dtype, device="cuda")[1:1 + t.numel()]
    return v.copy_(t.reshape(-1))


@pytest.mark.parametrize("keep", [None, []])
@pytest.mark.parametrize("planes", [False, True])
def test_encoder_unaligned_input(U, oracle_lib, keep, planes):
    """A caller's buffer off a 16-byte word, at a length only the strided kernel takes fused: the node by
    node pass, also where the next MatMul takes the output's planes."""
    import torch
    from cormorant_amd.graph import AttentionNode, Graph, MatmulNode, TensorInfo
    from cormorant_amd.simulate import Simulator
    rng = np.random.default_rng(5)
    B, T, H = 3, 48, 2
    x, o = TensorInfo("x", [B * T, 3 * 64 * H], exp=8), TensorInfo("o", [B * T, 64 * H], exp=8)
    nodes, out = [AttentionNode([x], o, batch=B, seq=T, heads=H, k_off=64 * H, v_off=128 * H)], o
    if planes:
        w = TensorInfo("w", [64 * H, 72], data=rng.integers(-40, 40, (64 * H, 72)) / 256.0, exp=8)
        out = TensorInfo("y", [B * T, 72], exp=8)
        nodes.append(MatmulNode([o, w], out))
    g = Graph(nodes=nodes, input_tensors=[x], output_tensors=[out])
    d = dev16(rint16(rng, x.numel, -2500, 2500), extra=0)
    want = Simulator(g).forward_raw({"x": d}, keep=keep)[out.onnx_name]
    got = Simulator(g).forward_raw({"x": _off_word(d)}, keep=keep)[out.onnx_name]
    assert torch.equal(got, want)


def test_prompt_unaligned_caches(U):
    """The attention chain alone over a caller's caches off a 16-byte word."""
    import torch
    from cormorant_amd import models
    from cormorant_amd.graph import AttnMergeNode, AttnSoftmaxNode, Graph, LlmAttnConvNode
    from cormorant_amd.simulate import Simulator
    S = models.LlamaShape(layers=1, batch=1, d=256, heads=4, kv=2, hd=64, ff=256, vocab=512, ctx=128)
    w = models.smollm2_weights(S, 5)
    _, _, exps = models.smollm2_decode(S, seed=5, weights=w)
    nodes = [nd for nd in models.smollm2_prefill(S, 32, exps, w).nodes
             if isinstance(nd, (LlmAttnConvNode, AttnSoftmaxNode, AttnMergeNode))]
    kc, qx, vc = nodes[0].inputs[0], nodes[0].inputs[1], nodes[2].inputs[1]
    g = Graph(nodes=nodes, input_tensors=[kc, qx, vc] + list(nodes[0].inputs[2:]), output_tensors=[nodes[-1].output])
    rng = np.random.default_rng(8)
    d = {t.onnx_name: dev16(rint16(rng, t.numel, -3000, 3000), extra=0) for t in (kc, qx, vc)}
    host_in = {"pos": np.array([37]), "n": np.array([32])}
    sim = Simulator(g)
    want = sim.forward_raw({**d, **host_in}, keep=[])[nodes[-1].output.onnx_name]
    got = sim.forward_raw({**{k: _off_word(v) for k, v in d.items()}, **host_in}, keep=[])[nodes[-1].output.onnx_name]
    assert torch.equal(got.reshape(-1), want.reshape(-1))
