"""The work a user of this framework has it do, as cases that can be prepared, run and timed.

Each case is a plain dict.  ``prepare`` makes what a program holds before the call (the weights laid
out once, the simulator with its captured forward, the raw inputs on the GPU), ``run`` is one pass:
a replay of the captured forward for whole graphs and layers (how a program serves a graph of small
launches: the capture is made once, inputs are written into its buffers), or the unit calls
themselves for single operations.  Every output is an integer the units define bit for bit, or such
an integer scaled by a power of two, so outputs are compared exactly.

Kinds:
  cnn        the small CNN, one image (models.small_cnn)
  mobilenet  MobileNetV2 in Q8.8 (models.mobilenet_v2)
  encoder    one encoder layer in pow2 numerics (models.bert_encoder with one layer)
  decode     one decode layer and a short head (models.smollm2_decode with one layer)
  prefill    one layer's prefill of one sequence (models.smollm2_prefill with one layer)
  matmul     the Matmul unit on operands of the call (both split per call)
  conv       the Conv unit with its weights laid out once
  head       a decode step's output projection and the dequantization of its logits
  rows       the residual add and the normalisation of its rows on the row-ops unit
"""
import math

import numpy as np
import torch

from cormorant_amd import models, units
from cormorant_amd import rowops_nodes as rn
from cormorant_amd.graph import TensorInfo
from cormorant_amd.packing import pack_matmul_b
from cormorant_amd.simulate import Simulator

MAX_MACS = 4 * 512 * 4096 * 4096          # the largest listed case's multiply-adds


def listed():
    return [
        # the smallest call: one image through a seven-launch network, launch latency alone
        {"name": "cnn_b1", "kind": "cnn"},
        # an image batch through a whole network: standard, pointwise and depthwise convolutions
        {"name": "mobilenet_b32", "kind": "mobilenet", "batch": 32, "res": 224},
        # the headline configuration's layer: a batch of full-length sequences
        {"name": "encoder_b8_s384", "kind": "encoder", "batch": 8, "seq": 384, "heads": 12},
        # one short query: every linear has few tiles
        {"name": "encoder_b1_s128", "kind": "encoder", "batch": 1, "seq": 128, "heads": 12},
        # a ragged batch: a sequence length that is no multiple of 64, an odd number of sequences
        {"name": "encoder_b5_s208", "kind": "encoder", "batch": 5, "seq": 208, "heads": 12},
        # a decode step's layer at the serving batch and a full cache
        {"name": "decode_b16_c1024", "kind": "decode", "batch": 16, "ctx": 1024, "d": 960, "heads": 15, "kv": 5,
         "ff": 2560, "vocab": 4096},
        # a prompt through a layer: the causal attention over a cache that holds earlier rows
        {"name": "prefill_t256", "kind": "prefill", "T": 256, "ctx": 1024, "pos": 300, "d": 960, "heads": 15, "kv": 5,
         "ff": 2560},
        # the largest product: Q8.8, the weight in the packed image, shared by the batch
        {"name": "matmul_b4_512x4096x4096", "kind": "matmul", "batch": 4, "n": 512, "k": 4096, "m": 4096,
         "wrap": False, "packed": True},
        # an odd product: no size a multiple of a tile, row-major operands, pow2 numerics
        {"name": "matmul_b3_1000x771x1235", "kind": "matmul", "batch": 3, "n": 1000, "k": 771, "m": 1235,
         "wrap": True, "packed": False},
        # an ordinary standard convolution (more taps than the short ones of the networks above)
        {"name": "conv3x3_b8_64x56", "kind": "conv", "batch": 8, "in_ch": 64, "out_ch": 128, "h": 56, "w": 56,
         "ksize": 3, "stride": 1},
        # the head of a decode step: 16 rows against a weight that HBM has to deliver once
        {"name": "head_b16_49152", "kind": "head", "batch": 16, "d": 960, "vocab": 49152},
        # many rows through the residual add and LayerNorm
        {"name": "add_norm_24576x768", "kind": "rows", "rows": 24576, "n": 768, "rms": False},
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _draw_one(rng):
    kind = rng.choice(["mobilenet", "encoder", "encoder", "decode", "decode", "prefill", "matmul", "matmul", "conv",
                       "conv", "head", "rows", "rows"])
    if kind == "mobilenet":
        return {"kind": kind, "batch": _log(rng, 1, 32), "res": 32 * rng.randint(2, 7)}
    if kind == "encoder":
        return {"kind": kind, "batch": _log(rng, 1, 16), "seq": 16 * rng.randint(2, 32), "heads": rng.choice([4, 8, 12, 16])}
    if kind == "decode":
        d, heads, kv, ff = rng.choice([(960, 15, 5, 2560), (576, 9, 3, 1536), (512, 8, 4, 1408)])
        return {"kind": kind, "batch": _log(rng, 1, 24), "ctx": 16 * rng.randint(4, 64), "d": d, "heads": heads, "kv": kv,
                "ff": ff, "vocab": 8 * rng.randint(100, 512)}
    if kind == "prefill":
        d, heads, kv, ff = rng.choice([(960, 15, 5, 2560), (576, 9, 3, 1536)])
        T, ctx = 16 * rng.randint(1, 20), 16 * rng.randint(24, 64)
        return {"kind": kind, "T": T, "ctx": ctx, "pos": rng.randint(0, ctx - T), "d": d, "heads": heads, "kv": kv, "ff": ff}
    if kind == "matmul":
        return {"kind": kind, "batch": _log(rng, 1, 8), "n": _log(rng, 1, 4096), "k": _log(rng, 16, 6000),
                "m": _log(rng, 16, 6000), "wrap": rng.random() < 0.5, "packed": rng.random() < 0.5}
    if kind == "conv":
        ksize = rng.choice([1, 3, 3, 5, 7])
        h = rng.randint(7, 112)
        return {"kind": kind, "batch": _log(rng, 1, 32), "in_ch": _log(rng, 8, 512), "out_ch": _log(rng, 8, 512), "h": h,
                "w": max(7, h + rng.randint(-5, 5)), "ksize": ksize, "stride": rng.choice([1, 1, 2])}
    if kind == "head":
        return {"kind": kind, "batch": _log(rng, 1, 16), "d": 64 * rng.randint(5, 32), "vocab": 8 * _log(rng, 250, 6400)}
    return {"kind": kind, "rows": _log(rng, 1, 32768), "n": 8 * _log(rng, 16, 256), "rms": rng.random() < 0.5}


def draw(rng):
    while True:
        c = _draw_one(rng)
        w = work(c)
        if w["flops"] <= 2 * MAX_MACS and w["bytes"] <= 400e6:
            return c


# ------------------------------------------------------------------ sizes
def _bert(c):
    return models.BertShape(layers=1, batch=c["batch"], seq=c["seq"], d=64 * c["heads"], heads=c["heads"],
                            ff=256 * c["heads"], vocab=1024)


def _llama(c, batch):
    return models.LlamaShape(layers=1, batch=batch, d=c["d"], heads=c["heads"], kv=c["kv"], hd=64, ff=c["ff"],
                             vocab=c.get("vocab", 1024), ctx=c["ctx"])


def _conv_geo(c):
    pad = c["ksize"] // 2
    oh = (c["h"] + 2 * pad - c["ksize"]) // c["stride"] + 1
    ow = (c["w"] + 2 * pad - c["ksize"]) // c["stride"] + 1
    return pad, oh, ow


def _mobilenet_sizes(batch, res):
    """(multiply-adds, weights) of MobileNetV2 1.0 with 1000 classes."""
    macs = weights = 0

    def conv(cin, cout, k, stride, h, dw=False):
        nonlocal macs, weights
        oh = (h + 2 * (k // 2) - k) // stride + 1
        w = cout * (1 if dw else cin) * k * k
        macs += batch * oh * oh * w
        weights += w
        return oh

    h = conv(3, 32, 3, 2, res)
    cin = 32
    for t, ch, n, s in models.MOBILENET_V2_BLOCKS:
        for i in range(n):
            mid = cin * t
            if t != 1:
                h = conv(cin, mid, 1, 1, h)
            h = conv(mid, mid, 3, s if i == 0 else 1, h, True)
            h = conv(mid, ch, 1, 1, h)
            cin = ch
    conv(320, 1280, 1, 1, h)
    return macs + batch * 1280 * 1000, weights + 1280 * 1000


def work(c):
    """Each input and weight read once, each output written once, two operations a multiply-add."""
    kind = c["kind"]
    if kind == "cnn":
        macs = 8 * 784 * 9 + 16 * 196 * 72 + 784 * 10
        return {"bytes": 2 * (784 + 8 * 9 + 16 * 72 + 7840 + 34 + 10), "flops": 2 * macs}
    if kind == "mobilenet":
        macs, weights = _mobilenet_sizes(c["batch"], c["res"])
        return {"bytes": 2 * (c["batch"] * (3 * c["res"] ** 2 + 1000) + weights), "flops": 2 * macs}
    if kind == "encoder":
        S = _bert(c)
        rows = S.batch * S.seq
        return {"bytes": rows * (4 + 4 * S.d) + 2 * (4 * S.d * S.d + 2 * S.d * S.ff) + 4 * min(rows, S.vocab) * S.d,
                "flops": 2 * S.macs()}
    if kind == "decode":
        S = _llama(c, c["batch"])
        cache = 2 * S.batch * S.kv * S.ctx * S.hd
        return {"bytes": S.weight_bytes() + 2 * cache + 4 * S.batch * S.vocab, "flops": 2 * S.macs()}
    if kind == "prefill":
        A, K, T, keys = c["heads"] * 64, c["kv"] * 64, c["T"], c["pos"] + c["T"]
        weights = c["d"] * (A + 2 * K) + A * c["d"] + 3 * c["d"] * c["ff"]
        return {"bytes": 2 * weights + 4 * T * c["d"] + 2 * 2 * keys * K, "flops": 2 * (T * weights + 2 * T * keys * A)}
    if kind == "matmul":
        b, n, k, m = c["batch"], c["n"], c["k"], c["m"]
        return {"bytes": 2 * (b * n * k + k * m + b * n * m), "flops": 2 * b * n * k * m}
    if kind == "conv":
        _, oh, ow = _conv_geo(c)
        b, w = c["batch"], c["out_ch"] * c["in_ch"] * c["ksize"] ** 2
        return {"bytes": 2 * (b * c["in_ch"] * c["h"] * c["w"] + w + c["out_ch"] + b * c["out_ch"] * oh * ow),
                "flops": 2 * b * oh * ow * w}
    if kind == "head":
        return {"bytes": 2 * c["d"] * (c["vocab"] + c["batch"]) + 6 * c["batch"] * c["vocab"],
                "flops": 2 * c["batch"] * c["d"] * c["vocab"]}
    return {"bytes": 12 * c["rows"] * c["n"] + 32 * c["n"], "flops": 12 * c["rows"] * c["n"]}


def tolerance(c):
    return "exact"                            # the units' arithmetic is integer: every bit is defined


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal16(g, numel, std):
    """int16 lanes of a normal distribution (a tensor at its own exponent, std in lanes)."""
    x = torch.randn(numel, generator=g, device="cuda", dtype=torch.float32) * std
    return x.round_().clamp_(-32768, 32767).to(torch.int16)


def _raw(t, values):
    """A graph input's lanes on the device: int32 / int16 at the tensor's exponent (Q8.8 without one)."""
    f = 8 if t.exp is None else t.exp
    v = np.rint(np.asarray(values, np.float64) * 2.0 ** np.asarray(f, np.float64))
    return torch.from_numpy(v.astype(np.int32 if t.kind == "i32" else np.int16)).cuda().reshape(-1)


def _matmul_inputs(c, seed):
    g = _gen(seed)
    b, n, k, m = c["batch"], c["n"], c["k"], c["m"]
    # Q8.8: activations N(0, 1) clipped at 8, weights N(0, 0.05); pow2: activations that fill the
    # lanes to a few deviations, weights at the exponent that keeps the output there too
    if c["wrap"]:
        a, w = _normal16(g, b * n * k, 4000.0), _normal16(g, k * m, max(2.0, 400.0 / math.sqrt(k)))
    else:
        a, w = _normal16(g, b * n * k, 256.0).clamp_(-2048, 2048), _normal16(g, k * m, 12.8)
    return a.view(b, n, k), w.view(k, m)


def _conv_inputs(c, seed):
    g = _gen(seed)
    x = _normal16(g, c["batch"] * c["in_ch"] * c["h"] * c["w"], 256.0).clamp_(0, 1536)      # after a RELU6
    fan = c["in_ch"] * c["ksize"] ** 2
    w = _normal16(g, c["out_ch"] * fan, 256.0 * math.sqrt(2.0 / fan))
    bias = _normal16(g, c["out_ch"], 25.0)
    return x.view(c["batch"], c["in_ch"], c["h"], c["w"]), w.view(c["out_ch"], c["in_ch"], c["ksize"], c["ksize"]), bias


def _conv_image(w):
    """The conv unit's weight image: per output channel, 16-lane input-channel tiles, the last of
    8 or 16 lanes; inside a tile [kh][kw][lane]."""
    out_ch, in_ch, kh, kw = w.shape
    parts = []
    for c0 in range(0, in_ch, 16):
        lanes = 16 if in_ch - c0 > 8 else 8
        t = torch.zeros((out_ch, lanes, kh, kw), dtype=w.dtype, device=w.device)
        t[:, :min(lanes, in_ch - c0)] = w[:, c0:c0 + lanes]
        parts.append(t.permute(0, 2, 3, 1).reshape(out_ch, -1))
    return torch.cat(parts, dim=1).reshape(-1).contiguous()


HEAD_EXP = 11                                  # the logits' exponent


def _head_inputs(c, seed):
    g = _gen(seed)
    return (_normal16(g, c["batch"] * c["d"], 4000.0).view(c["batch"], c["d"]),
            _normal16(g, c["d"] * c["vocab"], 20.0).view(c["d"], c["vocab"]))


# ------------------------------------------------------------------ captured graphs
def _captured(graph, feeds, keep):
    """The simulator of ``graph`` and its forward captured over ``feeds`` (name: device tensor):
    the first calls lay the weights out and grow the library's workspace, as bench.py does."""
    sim = Simulator(graph)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            sim.forward_raw(feeds, keep=keep)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    hg = torch.cuda.CUDAGraph()
    with torch.cuda.graph(hg):
        raw = sim.forward_raw(feeds, keep=keep)
    return {"sim": sim, "graph": hg, "out": {n: raw[n] for n in keep}}


def prepare(c, seed):
    kind = c["kind"]
    units.init()
    if kind == "cnn":
        g, inputs = models.small_cnn(seed)
        return _captured(g, {"input": _raw(g.input_tensors[0], inputs["input"])}, ["probs"])
    if kind == "mobilenet":
        g, inputs, _ = models.mobilenet_v2(c["batch"], c["res"], seed)
        return _captured(g, {"input": _raw(g.input_tensors[0], inputs["input"])}, ["logits"])
    if kind == "encoder":
        g, inputs, _ = models.bert_encoder(_bert(c), seed=seed)
        return _captured(g, {"ids": _raw(g.input_tensors[0], inputs["ids"])}, [g.output_tensors[0].onnx_name])
    if kind == "decode":
        g, inputs, _ = models.smollm2_decode(_llama(c, c["batch"]), seed=seed)
        feeds = {t.onnx_name: _raw(t, inputs[t.onnx_name]) for t in g.input_tensors}
        return _captured(g, feeds, ["logits", "l0.kc", "l0.vc"])
    if kind == "prefill":
        S = _llama(c, 1)
        w = models.smollm2_weights(S, seed)
        _, _, exps = models.smollm2_decode(S, seed=seed, weights=w)
        g = models.smollm2_prefill(S, c["T"], exps, w)
        rng = np.random.default_rng(seed)
        feeds = {"pos": np.array([c["pos"]], np.int64), "n": np.array([c["T"]], np.int64)}
        for t in g.input_tensors:
            if t.onnx_name == "ids":
                feeds["ids"] = _raw(t, rng.integers(0, S.vocab, c["T"]))
        for t in g.state_tensors:
            if t.onnx_name == "h_last":
                feeds["h_last"] = torch.zeros(t.numel, dtype=torch.int32, device="cuda")
            else:                              # group-major cache rows: the first pos of them written
                rows = np.zeros((S.kv, S.ctx, S.hd))
                rows[:, :c["pos"]] = rng.standard_normal((S.kv, c["pos"], S.hd)) * 0.6
                feeds[t.onnx_name] = _raw(t, rows)
        return _captured(g, feeds, ["h_last", "l0.kc", "l0.vc"])
    if kind == "matmul":
        a, w = _matmul_inputs(c, seed)
        img = torch.from_numpy(pack_matmul_b(w.cpu().numpy())).cuda() if c["packed"] else w.reshape(-1)
        out = torch.empty(c["batch"] * c["n"] * c["m"], dtype=torch.int16, device="cuda")
        return {"a": a.reshape(-1), "b": img, "c": out, "case": dict(c)}
    if kind == "conv":
        x, w, bias = _conv_inputs(c, seed)
        pad, oh, ow = _conv_geo(c)
        img = _conv_image(w)
        small = units.conv_small(c["in_ch"], c["ksize"], c["ksize"], c["out_ch"], c["batch"])
        if not small:                          # the weight's GEMM operand, laid out once
            img = units.conv_w_planes(img, c["out_ch"], c["in_ch"], c["ksize"], c["ksize"])
        y = torch.empty(c["batch"] * c["out_ch"] * oh * ow, dtype=torch.int16, device="cuda")
        return {"x": x.reshape(-1), "w": img, "small": small, "bias": bias, "y": y, "geo": (pad, oh, ow), "case": dict(c)}
    if kind == "head":
        a, w = _head_inputs(c, seed)
        n, k, m = c["batch"], c["d"], c["vocab"]
        chunk = next(x for x in range(4096, 0, -8) if m % x == 0)
        rows = n * m // chunk
        deq = rn.DequantRoNode([TensorInfo("q", [rows, chunk], exp=HEAD_EXP)], TensorInfo("f", [rows, chunk], kind="f32"))
        job = deq.jobs()[0]
        p = torch.from_numpy(np.ascontiguousarray(job.params, np.uint8)).cuda()
        q = torch.empty(n * m, dtype=torch.int16, device="cuda")
        f = torch.empty(n * m, dtype=torch.float32, device="cuda")
        return {"a": a.reshape(-1), "w": units.matmul_b_planes(w.reshape(-1), k, m), "q": q, "f": f, "case": dict(c),
                "job": dict(a=q.view(torch.uint8), b=None, c=f.view(torch.uint8), p=p, op=job.op, n=chunk, c1=rows, c2=1,
                            a_s1=2 * chunk, a_s2=0, b_s1=0, b_s2=0, c_s1=4 * chunk, c_s2=0)}
    # rows
    g = _gen(seed)
    rows, n = c["rows"], c["n"]
    rng = np.random.default_rng(seed)
    h = (torch.randn(rows * n, generator=g, device="cuda") * 2.0 ** 15).round_().to(torch.int32)
    d = _normal16(g, rows * n, 4000.0)
    ht, dt = TensorInfo("h", [rows, n], exp=15, kind="i32"), TensorInfo("d", [rows, n], exp=13)
    h1, y = TensorInfo("h1", [rows, n], exp=15, kind="i32"), TensorInfo("y", [rows, n], exp=12)
    gamma = 1.0 + 0.02 * rng.standard_normal(n)
    if c["rms"]:
        add, norm = rn.ResAddRoNode([ht, dt], h1), rn.RMSNormRoNode([h1], y, gamma=gamma, eps=1e-5)
    else:
        add = rn.ResAddBiasRoNode([ht, dt], h1, bias=0.02 * rng.standard_normal(n))
        norm = rn.LayerNorm32RoNode([h1], y, gamma=gamma, beta=0.02 * rng.standard_normal(n), eps=1e-12)
    out1 = torch.empty(rows * n, dtype=torch.int32, device="cuda")
    out2 = torch.empty(rows * n, dtype=torch.int16, device="cuda")
    jobs = []
    for node, a, b, o in ((add, h, d, out1), (norm, out1, None, out2)):
        j = node.jobs()[0]
        p = torch.from_numpy(np.ascontiguousarray(j.params, np.uint8)).cuda()
        jobs.append(dict(a=a.view(torch.uint8), b=b.view(torch.uint8) if b is not None else None,
                         c=o.view(torch.uint8), p=p, op=j.op, n=n, c1=rows, c2=1, a_s1=4 * n, a_s2=0,
                         b_s1=2 * n if b is not None else 0, b_s2=0, c_s1=n * o.element_size(), c_s2=0, eps=j.eps,
                         aux=j.aux, bq_sh=j.bq_sh))
    return {"jobs": jobs, "out": {"h": out1, "y": out2}}


def run(s):
    if "graph" in s:                          # a captured forward
        s["graph"].replay()
        return s["out"]
    if "jobs" in s:
        units.rowops_jobs(s["jobs"])
        return s["out"]
    c = s["case"]
    if c["kind"] == "matmul":
        n, k, m = c["n"], c["k"], c["m"]
        units.matmul(s["a"], s["b"], s["c"], n, k, m, batch=c["batch"], a_bs=n * k, c_bs=n * m,
                     b_packed=1 if c["packed"] else 0, wrap32=c["wrap"])
        return s["c"]
    if c["kind"] == "conv":
        pad, oh, ow = s["geo"]
        fn = units.conv if s["small"] else units.conv_planes
        fn(s["x"], s["w"], s["bias"], s["y"], c["batch"], c["in_ch"], c["h"], c["w"], c["out_ch"], oh, ow, c["ksize"],
           c["ksize"], c["stride"], c["stride"], pad_top=pad, pad_left=pad, has_bias=1)
        return s["y"]
    units.matmul_skinny_planes(s["a"], c["batch"], c["d"], [s["w"]], [s["q"]], [c["vocab"]])
    units.rowops_jobs([s["job"]])
    return {"q": s["q"], "logits": s["f"]}


# ------------------------------------------------------------------ 64-bit references
def _floor8(acc):
    """floor(acc / 2^8) saturated to int16: acc holds whole numbers below 2^53 exactly."""
    return torch.floor(acc / 256.0).clamp_(-32768, 32767).to(torch.int16)


def exact(c, seed):
    """The products in float64 (whole numbers below 2^53, exact; no sum here reaches 2^31, so the
    pow2 rule's 32-bit wrap never acts).  The layers, networks and row jobs are chains of the
    units' own integer rules, which plain torch has no counterpart of."""
    if c["kind"] == "matmul":
        a, w = _matmul_inputs(c, seed)
        return _floor8(torch.matmul(a.reshape(-1, c["k"]).double(), w.double())).reshape(-1)
    if c["kind"] == "conv":
        x, w, bias = _conv_inputs(c, seed)
        pad, oh, ow = _conv_geo(c)
        out = []
        for i in range(c["batch"]):
            cols = torch.nn.functional.unfold(x[i:i + 1].double(), c["ksize"], padding=pad, stride=c["stride"])[0]
            out.append(_floor8(torch.matmul(w.double().reshape(c["out_ch"], -1), cols) + 256.0 * bias.double()[:, None]))
        return torch.stack(out).reshape(-1)
    if c["kind"] == "head":
        a, w = _head_inputs(c, seed)
        q = _floor8(torch.matmul(a.double(), w.double())).reshape(-1)
        return {"q": q, "logits": q.double() * 2.0 ** -HEAD_EXP}
    return None
