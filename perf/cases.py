"""Performance cases of the framework: what its users run, through its public entry points (the
HipExecutionProvider operators and the ComputationalGraph runtime), over the sizes they run it at.

listed() names the cases, draw() gives others of the same ranges.  Tensors are torch allocations wrapped as
DeviceTensors, as a program does that holds its data on the GPU; graphs are built, fused and, where the program
captures them, captured in prepare(), which a user does once per model and input shape.  exact() evaluates the
same computation in 64 bits with plain torch."""
import math

import numpy as np
import torch

import onnx_amd
from onnx_amd import DeviceTensor, HipExecutionProvider as HIP
from onnx_amd.graph import ComputationalGraph

FLOAT = 1  # TensorElementType code of the Cast target
SQRT2 = np.float32(math.sqrt(2.0))


def listed():
    return [
        # A bias Add and a scalar Mul on one short sequence's activations: two eager operator calls whose time is
        # the call and the launch (the smallest work a program asks for).
        {"name": "bias_scale_128x384", "kind": "bias_scale", "rows": 128, "cols": 384},
        # The decomposed LayerNorm of a BERT-base layer, 8 sequences of 512 tokens.
        {"name": "layernorm_4096x768", "kind": "layernorm", "rows": 4096, "hidden": 768},
        # Attention probabilities of 16 sequences of 512 tokens, 12 heads: scale, padding mask, Softmax.
        {"name": "softmax_16x12x512", "kind": "softmax", "batch": 16, "heads": 12, "queries": 512, "keys": 512},
        # The headline step: GELU over 201M activations, then a sum over an axis and the mean of 268M values.
        {"name": "gelu_reduce_201m", "kind": "gelu_reduce", "batch": 32, "seq": 2048, "ff": 3072, "outer": 256,
         "mid": 4096, "inner": 256},
        # Integer features: an Int64 broadcast Add, its Float copy and its sums over an axis.
        {"name": "int64_64x256x4096", "kind": "int64", "outer": 64, "mid": 256, "inner": 4096},
        # The data movement of an exported model: embedding rows by token id, the Q part of a joint QKV
        # projection, its heads, and the three parts joined again.
        {"name": "movement_8x512x768", "kind": "movement", "batch": 8, "seq": 512, "heads": 12, "width": 64,
         "vocab": 30522},
        # The feed-forward block of a BERT-base layer over 8 sequences of 512 tokens.
        {"name": "ffn_4096x768x3072", "kind": "ffn", "tokens": 4096, "hidden": 768, "ff": 3072},
        # A batched Float MatMul of the tensor library's own benchmark suite.
        {"name": "matmul_f32_12x384", "kind": "matmul", "dtype": "float32", "batch": 12, "m": 384, "k": 384, "n": 384},
        # The same suite's six matrices in Int32 (wrapping).
        {"name": "matmul_i32_6x384", "kind": "matmul", "dtype": "int32", "batch": 6, "m": 384, "k": 384, "n": 384},
        # One BERT-base layer as a graph, sequences padded to the longest of the batch (197 tokens).
        {"name": "bert_layer_4x197", "kind": "encoder", "batch": 4, "seq": 197, "hidden": 768, "heads": 12, "ff": 3072,
         "layers": 1, "vocab": 0, "captured": False},
        # A short query through a multilingual-e5-small-shaped encoder: captured once, replayed per query.
        {"name": "encoder_1x8", "kind": "encoder", "batch": 1, "seq": 8, "hidden": 384, "heads": 12, "ff": 1536,
         "layers": 12, "vocab": 30522, "captured": True},
        # Documents through the same encoder, 8 of 512 tokens, executed eagerly.
        {"name": "encoder_8x512", "kind": "encoder", "batch": 8, "seq": 512, "hidden": 384, "heads": 12, "ff": 1536,
         "layers": 12, "vocab": 30522, "captured": False},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of its range."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["bias_scale", "layernorm", "softmax", "gelu_reduce", "int64", "movement", "ffn", "matmul",
                       "matmul", "encoder", "encoder", "encoder"])
    if kind == "bias_scale":
        return {"kind": kind, "rows": _size(rng, 1, 1024), "cols": _size(rng, 32, 3072)}
    if kind == "layernorm":
        return {"kind": kind, "rows": _size(rng, 8, 16384), "hidden": rng.choice([_size(rng, 64, 4096), 384, 768, 1024])}
    if kind == "softmax":
        s = _size(rng, 8, 512)
        return {"kind": kind, "batch": _size(rng, 1, 16), "heads": rng.choice([8, 12, 16]), "queries": s, "keys": s}
    if kind == "gelu_reduce":
        return {"kind": kind, "batch": _size(rng, 1, 32), "seq": _size(rng, 8, 2048), "ff": rng.choice([1536, 3072]),
                "outer": _size(rng, 1, 256), "mid": _size(rng, 8, 4096), "inner": _size(rng, 8, 256)}
    if kind == "int64":
        return {"kind": kind, "outer": _size(rng, 1, 64), "mid": _size(rng, 4, 256), "inner": _size(rng, 16, 4096)}
    if kind == "movement":
        return {"kind": kind, "batch": _size(rng, 1, 8), "seq": _size(rng, 8, 512), "heads": 12,
                "width": rng.choice([32, 64]), "vocab": 30522}
    if kind == "ffn":
        h = rng.choice([384, 768, _size(rng, 64, 768)])
        return {"kind": kind, "tokens": _size(rng, 8, 4096), "hidden": h, "ff": 4 * h}
    if kind == "matmul":
        dtype = rng.choice(["float32", "float32", "float32", "float64", "int32"])
        if rng.random() < 0.5:  # square-ish batches as the benchmark suite's
            n = _size(rng, 32, 512)
            return {"kind": kind, "dtype": dtype, "batch": rng.choice([1, 6, 12]), "m": n, "k": n, "n": n}
        top = 2048 if dtype == "float32" else 768
        return {"kind": kind, "dtype": dtype, "batch": 1, "m": _size(rng, 1, top), "k": _size(rng, 16, top),
                "n": _size(rng, 1, top)}
    seq = _size(rng, 8, 512)
    if rng.random() < 0.3:
        return {"kind": kind, "batch": _size(rng, 1, max(1, 2048 // seq)), "seq": seq, "hidden": 768, "heads": 12,
                "ff": 3072, "layers": 1, "vocab": 0, "captured": rng.random() < 0.5}
    return {"kind": kind, "batch": _size(rng, 1, max(1, 3072 // seq)), "seq": seq, "hidden": 384, "heads": 12,
            "ff": 1536, "layers": 12, "vocab": 30522, "captured": rng.random() < 0.5}


# ---- inputs ---------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda:0")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    return torch.randn(*shape, device="cuda:0", generator=g, dtype=dtype) * scale


def _data(c, seed):
    """The inputs of a case as torch tensors by name."""
    g, k = _gen(seed), c["kind"]
    if k == "bias_scale":
        return {"x": _randn(g, 1, c["rows"], c["cols"]), "bias": _randn(g, c["cols"], scale=0.1),
                "scale": torch.tensor(0.125, device="cuda:0")}
    if k == "layernorm":
        return {"x": _randn(g, c["rows"], c["hidden"], scale=2.0), "gamma": 1 + _randn(g, c["hidden"], scale=0.02),
                "beta": _randn(g, c["hidden"], scale=0.02)}
    if k == "softmax":
        b, s = c["batch"], c["keys"]
        lens = torch.randint(max(1, s - s // 4), s + 1, (b, 1), device="cuda:0", generator=g)
        mask = torch.where(torch.arange(s, device="cuda:0").view(1, s) < lens, 0.0, -10000.0).float()
        return {"s": _randn(g, b, c["heads"], c["queries"], s, scale=8.0), "mask": mask.view(b, 1, 1, s).contiguous(),
                "scale": torch.tensor(8.0, device="cuda:0")}
    if k == "gelu_reduce":
        y = torch.rand(c["outer"], c["mid"], c["inner"], device="cuda:0", generator=g)
        return {"x": _randn(g, c["batch"], c["seq"], c["ff"]), "y": y.mul_(2).sub_(1)}
    if k == "int64":
        a = torch.randint(-(2**20), 2**20 + 1, (c["outer"], 1, c["inner"]), device="cuda:0", generator=g)
        b = torch.randint(1, 1025, (1, c["mid"], c["inner"]), device="cuda:0", generator=g)
        return {"a": a, "b": b}
    if k == "movement":
        h = c["heads"] * c["width"]
        return {"table": _randn(g, c["vocab"], h),
                "ids": torch.randint(0, c["vocab"], (c["batch"], c["seq"]), device="cuda:0", generator=g),
                "qkv": _randn(g, c["batch"], c["seq"], 3 * h)}
    if k == "ffn":
        t, h, f = c["tokens"], c["hidden"], c["ff"]
        return {"x": _randn(g, t, h), "w1": _randn(g, h, f, scale=h ** -0.5), "b1": _randn(g, f, scale=0.02),
                "w2": _randn(g, f, h, scale=f ** -0.5), "b2": _randn(g, h, scale=0.02)}
    if k == "matmul":
        sa, sb = (c["batch"], c["m"], c["k"]), (c["batch"], c["k"], c["n"])
        if c["dtype"] == "int32":
            return {n: torch.randint(-(2**15), 2**15, s, device="cuda:0", generator=g, dtype=torch.int32)
                    for n, s in (("a", sa), ("b", sb))}
        dt = getattr(torch, c["dtype"])
        return {"a": _randn(g, *sa, dtype=dt), "b": _randn(g, *sb, dtype=dt)}
    # encoder: weights, then token ids (or, without a vocabulary, hidden states) and an attention mask that
    # pads the later sequences of the batch
    b, s, h, f = c["batch"], c["seq"], c["hidden"], c["ff"]
    d = {}
    if c["vocab"]:
        d["word_emb"], d["pos_emb"], d["tt_row"] = (_randn(g, *sh, scale=0.5) for sh in ((c["vocab"], h), (512, h), (h,)))
        d["gamma_emb"], d["beta_emb"] = 1 + _randn(g, h, scale=0.02), _randn(g, h, scale=0.02)
    for i in range(c["layers"]):
        for n, sh in (("wq", (h, h)), ("wk", (h, h)), ("wv", (h, h)), ("wo", (h, h)), ("w1", (h, f)), ("w2", (f, h)),
                      ("bq", (h,)), ("bk", (h,)), ("bv", (h,)), ("bo", (h,)), ("b1", (f,)), ("b2", (h,)),
                      ("beta1", (h,)), ("beta2", (h,))):
            d[f"{n}_{i}"] = _randn(g, *sh, scale=0.02)
        for n in ("gamma1", "gamma2"):
            d[f"{n}_{i}"] = 1 + _randn(g, h, scale=0.02)
    lens = torch.randint(max(1, s - s // 4), s + 1, (b, 1), device="cuda:0", generator=g)
    lens[0] = s
    d["attention_mask"] = (torch.arange(s, device="cuda:0").view(1, s) < lens).to(torch.int64)
    if c["vocab"]:
        d["input_ids"] = torch.randint(0, c["vocab"], (b, s), device="cuda:0", generator=g)
    else:
        d["hidden_states"] = _randn(g, b, s, h)
    return d


# ---- the encoder graph, node by node as an exported BERT-class model ---------------------------------------------
def _layernorm_nodes(add, x, y, sfx):
    add("ReduceMean", [x, "axes"], [f"mean{sfx}"])
    add("Sub", [x, f"mean{sfx}"], [f"d{sfx}"])
    add("Pow", [f"d{sfx}", "two"], [f"p{sfx}"])
    add("ReduceMean", [f"p{sfx}", "axes"], [f"var{sfx}"])
    add("Add", [f"var{sfx}", "eps"], [f"ve{sfx}"])
    add("Sqrt", [f"ve{sfx}"], [f"sd{sfx}"])
    add("Div", [f"d{sfx}", f"sd{sfx}"], [f"n{sfx}"])
    add("Mul", [f"n{sfx}", f"gamma{sfx}"], [f"m{sfx}"])
    add("Add", [f"m{sfx}", f"beta{sfx}"], [y])


def _encoder_graph(c, d):
    b, s, h, heads = c["batch"], c["seq"], c["hidden"], c["heads"]
    gr = ComputationalGraph(13)
    inputs = ("input_ids" if c["vocab"] else "hidden_states", "attention_mask")
    for n in inputs:
        gr.AddInput(n, np.float32 if n == "hidden_states" else np.int64, tuple(d[n].shape))
    f32 = np.float32
    consts = {"heads_shape": np.array([b, s, heads, h // heads], np.int64), "hidden_shape": np.array([b, s, h], np.int64),
              "scale": np.array(math.sqrt(h // heads), f32), "axes": np.array([-1], np.int64), "two": np.array(2.0, f32),
              "eps": np.array(1e-12, f32), "sqrt2": np.array(SQRT2, f32), "one": np.array(1.0, f32),
              "half": np.array(0.5, f32), "unsq_axes": np.array([1, 2], np.int64), "neg": np.array(-10000.0, f32)}
    if c["vocab"]:
        consts["position_ids"] = np.arange(s, dtype=np.int64).reshape(1, s)
    for n, v in list(consts.items()) + [(n, t.cpu().numpy()) for n, t in d.items() if n not in inputs]:
        gr.AddInitializer(n, v)

    def add(op, ins, outs, **attrs):
        gr.AddNode(op, ins, outs, name=f"{op}_{outs[0]}", **attrs)

    x = "hidden_states"
    if c["vocab"]:
        add("Gather", ["word_emb", "input_ids"], ["we"], axis=0)
        add("Gather", ["pos_emb", "position_ids"], ["pe"], axis=0)
        add("Add", ["we", "pe"], ["e0"])
        add("Add", ["e0", "tt_row"], ["e1"])
        _layernorm_nodes(add, "e1", "h_0", "_emb")
        x = "h_0"
    add("Unsqueeze", ["attention_mask", "unsq_axes"], ["m0"])
    add("Cast", ["m0"], ["m1"], to=FLOAT)
    add("Sub", ["one", "m1"], ["m2"])
    add("Mul", ["m2", "neg"], ["mask"])
    for i in range(c["layers"]):
        y = f"h_{i + 1}" if i + 1 < c["layers"] else "last_hidden_state"
        for t, perm in (("q", [0, 2, 1, 3]), ("k", [0, 2, 3, 1]), ("v", [0, 2, 1, 3])):
            add("MatMul", [x, f"w{t}_{i}"], [f"{t}0_{i}"])
            add("Add", [f"{t}0_{i}", f"b{t}_{i}"], [f"{t}1_{i}"])
            add("Reshape", [f"{t}1_{i}", "heads_shape"], [f"{t}2_{i}"])
            add("Transpose", [f"{t}2_{i}"], [f"{t}h_{i}"], perm=perm)
        add("MatMul", [f"qh_{i}", f"kh_{i}"], [f"s0_{i}"])
        add("Div", [f"s0_{i}", "scale"], [f"s1_{i}"])
        add("Add", [f"s1_{i}", "mask"], [f"s2_{i}"])
        add("Softmax", [f"s2_{i}"], [f"probs_{i}"], axis=-1)
        add("MatMul", [f"probs_{i}", f"vh_{i}"], [f"c0_{i}"])
        add("Transpose", [f"c0_{i}"], [f"c1_{i}"], perm=[0, 2, 1, 3])
        add("Reshape", [f"c1_{i}", "hidden_shape"], [f"c2_{i}"])
        add("MatMul", [f"c2_{i}", f"wo_{i}"], [f"o0_{i}"])
        add("Add", [f"o0_{i}", f"bo_{i}"], [f"o1_{i}"])
        add("Add", [f"o1_{i}", x], [f"r1_{i}"])
        _layernorm_nodes(add, f"r1_{i}", f"a_{i}", f"1_{i}")
        add("MatMul", [f"a_{i}", f"w1_{i}"], [f"f0_{i}"])
        add("Add", [f"f0_{i}", f"b1_{i}"], [f"f1_{i}"])
        add("Div", [f"f1_{i}", "sqrt2"], [f"g0_{i}"])
        add("Erf", [f"g0_{i}"], [f"g1_{i}"])
        add("Add", [f"g1_{i}", "one"], [f"g2_{i}"])
        add("Mul", [f"f1_{i}", f"g2_{i}"], [f"g3_{i}"])
        add("Mul", [f"g3_{i}", "half"], [f"g4_{i}"])
        add("MatMul", [f"g4_{i}", f"w2_{i}"], [f"f2_{i}"])
        add("Add", [f"f2_{i}", f"b2_{i}"], [f"f3_{i}"])
        add("Add", [f"f3_{i}", f"a_{i}"], [f"r2_{i}"])
        _layernorm_nodes(add, f"r2_{i}", y, f"2_{i}")
        x = y
    gr.AddOutput("last_hidden_state")
    gr.Fuse()
    return gr


class _View:
    """A graph output's device memory for torch (read in place; valid until the graph's next execution)."""

    def __init__(self, t):
        self.t = t  # keeps the graph
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": t.dtype.str, "data": (t.h.data, False), "version": 2}


def _graph_output(gr, name):
    return torch.as_tensor(_View(gr.Output(name)), device="cuda:0")


# ---- prepare and run ----------------------------------------------------------------------------------------------
def prepare(case, seed):
    onnx_amd.init(0)
    c, d = case, _data(case, seed)
    k = c["kind"]
    s = {"case": c, "keep": d}

    def out(name, shape, dtype=torch.float32):
        s[name] = torch.empty(*shape, device="cuda:0", dtype=dtype)
        s["w" + name] = DeviceTensor.wrap_torch(s[name])

    if k == "encoder":
        inputs = ("input_ids" if c["vocab"] else "hidden_states", "attention_mask")
        torch.cuda.synchronize()
        s["graph"] = _encoder_graph(c, d)
        s["inputs"] = {n: DeviceTensor.wrap_torch(d[n]) for n in inputs}
        s["keep"] = {n: d[n] for n in inputs}
        if c["captured"] and not s["graph"].Capture(s["inputs"]):
            raise RuntimeError(s["graph"].LastError)
        return s
    s["in"] = {n: DeviceTensor.wrap_torch(t) for n, t in d.items()}
    if k == "bias_scale":
        out("h", d["x"].shape)
        out("y", d["x"].shape)
    elif k in ("layernorm", "softmax"):
        out("y", d["x" if k == "layernorm" else "s"].shape)
    elif k == "gelu_reduce":
        out("y", d["x"].shape)
        out("sums", (c["outer"], 1, c["inner"]))
        out("mean", (1, 1, 1))
    elif k == "int64":
        sh = (c["outer"], c["mid"], c["inner"])
        out("y", sh, torch.int64)
        out("f", sh)
        out("sums", (c["outer"], 1, c["inner"]), torch.int64)
    elif k == "movement":
        b, q, n, w = c["batch"], c["seq"], c["heads"], c["width"]
        out("emb", (b, q, n * w))
        out("part", (b, q, n * w))
        out("heads", (b, n, q, w))
        out("joined", (b, q, 3 * n * w))
        s["part4"] = s["wpart"].reshape((b, q, n, w))
    elif k == "ffn":
        out("mid", (c["tokens"], c["ff"]))
        out("y", (c["tokens"], c["hidden"]))
    elif k == "matmul":
        out("y", (c["batch"], c["m"], c["n"]), getattr(torch, c["dtype"]))
    torch.cuda.synchronize()
    return s


def _ok(*results):
    for r in results:
        if r.Code:
            raise RuntimeError(r.Message)


def run(state):
    s, c = state, state["case"]
    k = c["kind"]
    if k == "encoder":
        gr = s["graph"]
        if not (gr.Replay() if c["captured"] else gr.Execute(s["inputs"])):
            raise RuntimeError(gr.LastError)
        return _graph_output(gr, "last_hidden_state")
    i = s["in"]
    if k == "bias_scale":
        _ok(HIP.Add(i["x"], i["bias"], out=s["wh"]), HIP.Mul(s["wh"], i["scale"], out=s["wy"]))
        return s["y"]
    if k == "layernorm":
        _ok(HIP.LayerNormDecomposed(i["x"], i["gamma"], i["beta"], 1e-12, out=s["wy"]))
        return s["y"]
    if k == "softmax":
        _ok(HIP.ScaleAddSoftmax(i["s"], i["scale"], True, i["mask"], -1, out=s["wy"]))
        return s["y"]
    if k == "gelu_reduce":
        _ok(HIP.GeluErf(i["x"], out=s["wy"]), HIP.ReduceSum(i["y"], [1], 1, out=s["wsums"]),
            HIP.ReduceMean(i["y"], None, 1, out=s["wmean"]))
        return [s["y"], s["sums"], s["mean"]]
    if k == "int64":
        _ok(HIP.Add(i["a"], i["b"], out=s["wy"]), HIP.Cast(s["wy"], FLOAT, out=s["wf"]),
            HIP.ReduceSum(s["wy"], [1], 1, out=s["wsums"]))
        return [s["y"], s["f"], s["sums"]]
    if k == "movement":
        h = c["heads"] * c["width"]
        _ok(HIP.Gather(i["table"], i["ids"], 0, out=s["wemb"]),
            HIP.Slice(i["qkv"], [0], [h], [-1], None, out=s["wpart"]),
            HIP.Transpose(s["part4"], [0, 2, 1, 3], out=s["wheads"]),
            HIP.Concat([s["wpart"], s["wemb"], s["wpart"]], -1, out=s["wjoined"]))
        return [s["emb"], s["part"], s["heads"], s["joined"]]
    if k == "ffn":
        _ok(HIP.MatMulAddGelu(i["x"], i["w1"], i["b1"], out=s["wmid"]),
            HIP.MatMulAdd(s["wmid"], i["w2"], i["b2"], i["x"], out=s["wy"]))
        return [s["mid"], s["y"]]
    _ok(HIP.MatMul(i["a"], i["b"], out=s["wy"]))
    return s["y"]


# ---- work, tolerance, exact ---------------------------------------------------------------------------------------
def work(case):
    c, k = case, case["kind"]
    if k == "bias_scale":
        n = c["rows"] * c["cols"]
        return {"bytes": 4 * (2 * n + c["cols"] + 1), "flops": 2 * n}
    if k == "layernorm":
        n = c["rows"] * c["hidden"]
        return {"bytes": 4 * (2 * n + 2 * c["hidden"]), "flops": 8 * n}
    if k == "softmax":
        n = c["batch"] * c["heads"] * c["queries"] * c["keys"]
        return {"bytes": 4 * (2 * n + c["batch"] * c["keys"] + 1), "flops": 6 * n}
    if k == "gelu_reduce":
        n, m = c["batch"] * c["seq"] * c["ff"], c["outer"] * c["mid"] * c["inner"]
        # the reduced tensor is read by two operator calls; once is what they cannot do without
        return {"bytes": 4 * (2 * n + m + c["outer"] * c["inner"] + 1), "flops": 20 * n + 2 * m}
    if k == "int64":
        n = c["outer"] * c["mid"] * c["inner"]
        return {"bytes": 12 * n + 8 * (c["mid"] * c["inner"] + 2 * c["outer"] * c["inner"]), "flops": 2 * n}
    if k == "movement":
        n = c["batch"] * c["seq"] * c["heads"] * c["width"]
        # embedding rows and the Q part read, the four results written
        return {"bytes": 4 * 8 * n + 8 * c["batch"] * c["seq"], "flops": 0}
    if k == "ffn":
        t, h, f = c["tokens"], c["hidden"], c["ff"]
        return {"bytes": 4 * (2 * t * h + 2 * h * f + f + h + t * f), "flops": 4 * t * h * f}
    if k == "matmul":
        e = 8 if c["dtype"] == "float64" else 4
        b, m, kk, n = c["batch"], c["m"], c["k"], c["n"]
        return {"bytes": e * b * (m * kk + kk * n + m * n), "flops": 2 * b * m * kk * n}
    t, h, f, s = c["batch"] * c["seq"], c["hidden"], c["ff"], c["seq"]
    weights = c["layers"] * (4 * h * h + 2 * h * f + 9 * h + f)
    emb = t * h + s * h if c["vocab"] else t * h
    return {"bytes": 4 * (weights + emb + t * h) + 8 * t,
            "flops": c["layers"] * (2 * t * (4 * h * h + 2 * h * f) + 4 * t * s * h)}


def tolerance(case):
    k = case["kind"]
    if k in ("int64", "movement") or (k == "matmul" and case["dtype"] == "int32"):
        return "exact"
    if k == "bias_scale":
        return {"rel": 2e-7, "max": 1e-6}      # two separately rounded float32 operations
    if k == "layernorm":
        return {"rel": 3e-7, "max": 1e-5}      # float32 row sums in another order (6e-8 off 64 bits)
    if k == "softmax":
        return {"rel": 4e-7, "max": 2e-4}      # exp of float32 differences, row sums in another order (6e-8)
    if k == "gelu_reduce":
        return {"rel": 1e-5, "max": 1e-4}      # sums of up to 268M signed float32 values in another order (8e-7)
    if k == "matmul" and case["dtype"] == "float64":
        return {"rel": 1e-14, "max": 1e-12}
    if k in ("ffn", "matmul"):
        return {"rel": 3e-6, "max": 1e-4}      # float32 dot products of up to 3072 terms in another order (6e-7)
    return {"rel": 4e-6, "max": 4e-4}          # up to 12 layers of them (6e-7)


def _norm64(t, g, b):
    m = t.mean(-1, keepdim=True)
    v = (t - m).square().mean(-1, keepdim=True)
    return (t - m) / torch.sqrt(v + 1e-12) * g + b


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x / math.sqrt(2.0)))


def exact(case, seed):
    c, d = case, _data(case, seed)
    k = c["kind"]
    if k in ("int64", "movement") or (k == "matmul" and c["dtype"] == "int32"):
        return None  # whole numbers and copies: compared bit for bit
    if k != "gelu_reduce":
        d = {n: t.double() if t.is_floating_point() else t for n, t in d.items()}
    if k == "bias_scale":
        return (d["x"] + d["bias"]) * d["scale"]
    if k == "layernorm":
        return _norm64(d["x"], d["gamma"], d["beta"])
    if k == "softmax":
        return torch.softmax(d["s"] / d["scale"] + d["mask"], -1)
    if k == "gelu_reduce":
        y = d["y"].double()
        return [_gelu64(d["x"].double()), y.sum(1, keepdim=True), y.mean().reshape(1, 1, 1)]
    if k == "ffn":
        mid = _gelu64(d["x"] @ d["w1"] + d["b1"])
        return [mid, mid @ d["w2"] + d["b2"] + d["x"]]
    if k == "matmul":
        return torch.matmul(d["a"], d["b"]) if c["dtype"] == "float32" else None  # Double is 64 bits already
    b, s, heads = c["batch"], c["seq"], c["heads"]

    def split(t):
        return t.reshape(b, s, heads, -1).transpose(1, 2).contiguous()

    if c["vocab"]:
        x = _norm64(d["word_emb"][d["input_ids"]] + d["pos_emb"][:s] + d["tt_row"], d["gamma_emb"], d["beta_emb"])
    else:
        x = d["hidden_states"]
    mask = (1.0 - d["attention_mask"].double()).reshape(b, 1, 1, s) * -10000.0
    for i in range(c["layers"]):
        q, kk, v = (split(x @ d[f"w{t}_{i}"] + d[f"b{t}_{i}"]) for t in "qkv")
        p = torch.softmax(torch.matmul(q, kk.transpose(2, 3).contiguous()) / math.sqrt(c["hidden"] // heads) + mask, -1)
        ctx = torch.matmul(p, v).transpose(1, 2).reshape(b, s, -1)
        a = _norm64(ctx @ d[f"wo_{i}"] + d[f"bo_{i}"] + x, d[f"gamma1_{i}"], d[f"beta1_{i}"])
        g = _gelu64(a @ d[f"w1_{i}"] + d[f"b1_{i}"])
        x = _norm64(g @ d[f"w2_{i}"] + d[f"b2_{i}"] + a, d[f"gamma2_{i}"], d[f"beta2_{i}"])
    return x
