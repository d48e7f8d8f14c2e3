"""The Attention node of heads longer than one tile (more than 64 rows and 72 keys): scores, scaled masked Softmax and
context in one launch (lx_attention.hip), against float64 and against the three nodes it replaces.

Bar: the scores' float32 sums are within e_s = (6 ceil(D / 16) + 3) 2^-24 max_j sum |q k_j| / scale of the exact ones
(six roundings per step of 16, the scale, the mask and the maximum's subtraction); an error of e_s in every score
moves a probability by at most 2 e_s of itself, and the exponential, the sums and the context's own roundings
((6 ceil(SK / 16) + 16) 2^-24) add to that: |got - exact| <= (2 e_s + (6 ceil(SK / 16) + 32) 2^-24) sum_j p_j |v_j|."""
import time

import numpy as np
import pytest

import onnx_amd
import onnx_writer as W
from onnx_amd import DeviceTensor
from onnx_amd.graph import Model
from test_gpu_attention import attention_model

pytestmark = pytest.mark.gpu


def constants(model_args):
    """The mask and scale attention_model draws for these arguments (the same generator, in the same order)."""
    b, h, s, sk, d, dv, mask_kind, scale = model_args
    rng = np.random.default_rng(s * 1000 + sk * 100 + d + 7 * dv)
    mshape = {"b11s": (b, 1, 1, sk), "bhss": (b, h, s, sk), "b1ss": (b, 1, s, sk), "s": (sk,), "one": (1,)}[mask_kind]
    mask = np.where(rng.random(mshape) < 0.2, -10000.0, rng.normal(0, 0.5, mshape)).astype(np.float32)
    c = {"div": np.float32(np.sqrt(d)), "mul": np.float32(1.0 / np.sqrt(d)), None: np.float32(1)}[scale]
    return mask, c


def exact(q, k, v, mask, c, div):
    """softmax(q k^T scaled + mask) v in float64 and the bar, [b, s, h, dv]; the reference's maximum starts at 0."""
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    f = 1.0 / float(c) if div else float(c)
    s = q @ k.transpose(0, 1, 3, 2) * f + mask.astype(np.float64)
    mag = (np.abs(q) @ np.abs(k).transpose(0, 1, 3, 2) * abs(f)).max(-1, keepdims=True)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    e = (6 * -(-q.shape[-1] // 16) + 3) * 2.0 ** -24 * (mag + np.abs(np.where(mask < -1000, 0, mask)).max() + 1)
    bar = (2 * e + (6 * -(-k.shape[2] // 16) + 32) * 2.0 ** -24) * (p @ np.abs(v))
    return (p @ v).transpose(0, 2, 1, 3), bar.transpose(0, 2, 1, 3)


CASES = [  # b, h, s, sk, d, dv, mask, scale
    (2, 3, 128, 128, 32, 32, "b11s", "div"),    # whole tiles
    (2, 16, 512, 512, 64, 64, "b11s", "div"),   # BERT-base heads
    (2, 2, 197, 197, 64, 64, "b11s", "div"),    # rows and keys past the last tile, unaligned mask rows
    (1, 2, 65, 73, 64, 64, "bhss", "mul"),      # the smallest
    (1, 3, 130, 97, 33, 17, "bhss", "div"),     # ragged widths
    (2, 12, 77, 300, 20, 50, "b1ss", None),     # three mask row axes, no scale
    (1, 24, 129, 1030, 16, 33, "s", "mul"),     # many key tiles
    (1, 1, 100, 80, 1, 1, "b11s", "div"),
    (1, 160, 66, 1056, 8, 64, "one", "mul"),
]


def same_bits(x, y):
    """Heads that run the three nodes give their bits, the one-launch kernel does not (the sums' order)."""
    return np.array_equal(x.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:6])) + f"-{c[6]}-{c[7]}")
def test_long_heads(hip, case):
    b, h, s, sk, d, dv, mask_kind, scale = case
    model, ins = attention_model(*case)
    kept, _ = attention_model(*case, extra_outputs=("sc",))
    mask, c = constants(case)
    dev = {k: DeviceTensor.from_numpy(v) for k, v in ins.items()}
    g, g3 = Model.Load(model), Model.Load(kept)
    g.Fuse()
    g3.Fuse()
    assert [n.Op for n in g.Nodes] == ["Attention"] and len(g3.Nodes) == 3
    assert g.Execute(dev) and g3.Execute(dev), (g.LastError, g3.LastError)
    ref, bar = exact(ins["q"], ins["k"], ins["v"], mask, c, scale == "div")
    got, nodes = g.Output("y").to_numpy(), g3.Output("y").to_numpy()
    assert got.shape == ref.shape and np.isfinite(got).all() and not same_bits(got, nodes)
    assert np.all(np.abs(got - ref) <= bar), float((np.abs(got - ref) / bar).max())
    # no further from float64 than the three nodes (their own errors of the same size)
    assert np.linalg.norm(got - ref) <= 1.5 * np.linalg.norm(nodes - ref) + 1e-7 * np.linalg.norm(ref)
    assert g.Capture(dev), g.LastError
    for rep in range(3):
        q2 = (ins["q"] * (0.5 + rep)).astype(np.float32)
        dev["q"].upload(q2)
        assert g.Replay(), g.LastError
        got2 = g.Output("y").to_numpy().copy()
        ref2, bar2 = exact(q2, ins["k"], ins["v"], mask, c, scale == "div")
        assert np.all(np.abs(got2 - ref2) <= bar2), rep
    g.ReleaseCapture()
    g.EnableProfiling(True)
    assert g.Execute(dev), g.LastError
    assert [p["op"] for p in g.Profile] == ["Attention"]


def _run(q, k, v, mask, fused=True, scale=("Div", 8.0)):
    """Projection-layout inputs [b, s, h, d] through the transposed views, the mask an input, scores divided by 8."""
    b, s, h, d = q.shape
    nodes = [W.node("Transpose", ["q"], ["qt"], "tq", perm=[0, 2, 1, 3]),
             W.node("Transpose", ["k"], ["kt"], "tk", perm=[0, 2, 3, 1]),
             W.node("Transpose", ["v"], ["vt"], "tv", perm=[0, 2, 1, 3]),
             W.node("MatMul", ["qt", "kt"], ["sc"], "scores"), W.node(scale[0], ["sc", "c"], ["sd"], "scale"),
             W.node("Add", ["sd", "mask"], ["t"], "add"), W.node("Softmax", ["t"], ["p"], "softmax", axis=-1),
             W.node("MatMul", ["p", "vt"], ["ctx"], "context"),
             W.node("Transpose", ["ctx"], ["y"], "ty", perm=[0, 2, 1, 3])]
    ins = {"q": q, "k": k, "v": v, "mask": mask}
    g = Model.Load(W.model(nodes, [(n, np.float32, a.shape) for n, a in ins.items()], [("y", np.float32, ())],
                           [("c", np.array(scale[1], np.float32))]))
    if fused:
        g.Fuse()
        assert [n.Op for n in g.Nodes] == ["Attention"]
    assert g.Execute({n: DeviceTensor.from_numpy(a) for n, a in ins.items()}), g.LastError
    return g.Output("y").to_numpy()


def float32_chain(a, b, ranges=1):
    """a b with the products added one after another in float32, each exact before it is added, in equal ranges of the
    inner axis whose sums are added in order."""
    a64, b64, k = a.astype(np.float64), b.astype(np.float64), a.shape[-1]
    total = None
    for r in range(ranges):
        acc = np.zeros(a.shape[:-1] + (b.shape[-1],), np.float32)
        for j in range(r * k // ranges, (r + 1) * k // ranges):
            acc = (acc + a64[..., j:j + 1] * b64[..., j:j + 1, :]).astype(np.float32)
        total = acc if total is None else total + acc
    return total


@pytest.mark.parametrize("s,d,ranges", [(512, 64, 4), (197, 64, 1), (512, 32, 4), (128, 16, 2)])
@pytest.mark.parametrize("kind", ["normal", "relu_v", "positive", "sparse_v", "sparse", "few_keys"])
def test_long_heads_error_is_no_larger_than_the_nodes(hip, s, d, ranges, kind):
    """Against 64 bits: no further off than float32 products summed in chains (the context's K in the ranges a split
    product has there), a correctly rounded exponential and a division of every probability."""
    rng = np.random.default_rng(s + d)
    q, k, v = (rng.normal(0, 1, (2, s, 16 if s == 512 else 4, d)).astype(np.float32) for _ in range(3))
    mask = np.where(np.arange(s) < s - s // 6, 0.0, -10000.0).astype(np.float32).reshape(1, 1, 1, s)
    if kind == "relu_v":
        v = np.maximum(v, 0)
    elif kind == "positive":
        q, k, v = (np.maximum(t, 0) for t in (q, k, v))
    elif kind == "sparse_v":
        v = v * (rng.random(v.shape) < 0.02)
    elif kind == "sparse":
        q, k, v = (t * (rng.random(t.shape) < 0.1) for t in (q, k, v))
    elif kind == "few_keys":
        mask = np.where(rng.random((2, 1, 1, s)) < 0.03, 0.0, -10000.0).astype(np.float32)
        mask[..., 0] = 0
    q, k, v = (t.astype(np.float32) for t in (q, k, v))
    qh, kh, vh = (t.transpose(0, 2, 1, 3) for t in (q, k, v))
    ref, _ = exact(qh, kh, vh, mask, np.float32(8), True)
    t = float32_chain(qh, kh.transpose(0, 1, 3, 2)) / np.float32(8) + mask
    e = np.exp((t - np.maximum(t.max(-1, keepdims=True), 0)).astype(np.float64)).astype(np.float32)
    nodes = float32_chain(e / e.sum(-1, keepdims=True), vh, ranges).transpose(0, 2, 1, 3)
    assert np.linalg.norm(_run(q, k, v, mask) - ref) <= np.linalg.norm(nodes - ref)


@pytest.mark.parametrize("kind", ["plain", "masked_rows", "lowest", "first_keys", "infinite_mask", "tiny_v", "huge_v",
                                  "inf_v", "inf_k", "nan_q", "tiny_qk", "large_scores"])
def test_long_heads_special_values(hip, kind):
    """Rows masked whole (NaN: the maximum starts at 0), a mask of the type's lowest value, whole first tiles masked,
    an infinite mask, and operands the bf16 parts cannot hold, which run on the fp32 MFMA: the pattern of NaN and
    infinities of the unfused graph, and its values within 1e-5 of the context's magnitude."""
    rng = np.random.default_rng(5)
    b, s, h, d = 2, 99, 3, 64
    q, k, v = (rng.normal(0, 1, (b, s, h, d)).astype(np.float32) for _ in range(3))
    mask = np.zeros((b, 1, 1, s), np.float32)
    mask[0, 0, 0, 80:] = -10000.0
    if kind == "masked_rows":
        mask[1] = -10000.0
    elif kind == "lowest":
        mask[mask != 0] = np.finfo(np.float32).min
        mask[1, 0, 0, :40] = np.finfo(np.float32).min
    elif kind == "first_keys":
        mask[1, 0, 0, :70] = -10000.0
    elif kind == "infinite_mask":
        mask[mask != 0] = -np.inf
        mask[1, 0, 0, :32] = -np.inf
    elif kind == "tiny_v":
        v[0] = (v[0] * 1e-36).astype(np.float32)
    elif kind == "huge_v":
        v[0, 3] = 1e30
    elif kind == "inf_v":
        v[0, 3, 1, 5], v[1, 90, 0, 0] = np.inf, np.nan
    elif kind == "inf_k":
        k[0, 50, 1, 2], k[1, 98, 2, 0] = np.inf, -np.inf
    elif kind == "nan_q":
        q[0, 10, 0, 0], q[1, 98, 2, 63] = np.nan, np.inf
    elif kind == "tiny_qk":
        q, k = (q * 1e-30).astype(np.float32), (k * 1e-10).astype(np.float32)
    elif kind == "large_scores":
        q = q * np.float32(20)
    got, ref = _run(q, k, v, mask), _run(q, k, v, mask, fused=False)
    assert not same_bits(got, ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], ref[inf])
    fin = np.isfinite(ref)
    if kind == "masked_rows":
        assert not fin[1].any() and fin[0].all()
    scale = np.broadcast_to(np.abs(np.where(np.isfinite(v), v, 0)).max(1, keepdims=True), ref.shape)  # per head column
    tol = 3e-5 if kind == "large_scores" else 1e-5  # scores of +-60: their float32 spacing alone is 4e-6
    assert np.all(np.abs(got[fin] - ref[fin]) <= tol * scale[fin])


def test_long_heads_random(hip):
    """Random sizes around the tiles, permuted views, against float64."""
    rng = np.random.default_rng(21)
    for _ in range(12):
        b, h = int(rng.integers(1, 4)), int(rng.integers(4, 9))
        s, d = 4 * int(rng.integers(18, 72)) + int(rng.integers(1, 4)), int(rng.integers(1, 65))
        q, k, v = (rng.normal(0, 1, (b, s, h, d)).astype(np.float32) for _ in range(3))
        mask = np.where(rng.random((b, 1, 1, s)) < 0.3, -10000.0, 0.0).astype(np.float32)
        ref, bar = exact(*(t.transpose(0, 2, 1, 3) for t in (q, k, v)), mask, np.float32(8), True)
        got = _run(q, k, v, mask)
        assert np.all(np.abs(got - ref) <= bar), (b, h, s, d, float((np.abs(got - ref) / bar).max()))


@pytest.mark.parametrize("scale", [("Mul", 1e37), ("Mul", -3e20), ("Mul", 1e6), ("Div", 1e-30), ("Div", -7.3), ("Mul", 1e-20)])
def test_long_heads_scales(hip, scale):
    """Scale constants far from 1 over operands that bring the scores back to a few units, tiny ones included: the
    unfused graph's values within 1e-5 of the context's magnitude."""
    rng = np.random.default_rng(41)
    b, s, h, d = 1, 99, 3, 64
    q, k, v = (rng.normal(0, 1, (b, s, h, d)).astype(np.float32) for _ in range(3))
    f = 0.125 / abs(scale[1] if scale[0] == "Mul" else 1 / scale[1])
    q = (q * (f if f < 1 else f ** 0.5)).astype(np.float32)
    k = (k * (1 if f < 1 else f ** 0.5)).astype(np.float32)
    mask = np.where(np.arange(s) < 90, 0.0, -10000.0).astype(np.float32).reshape(1, 1, 1, s)
    got, ref = _run(q, k, v, mask, scale=scale), _run(q, k, v, mask, fused=False, scale=scale)
    assert not same_bits(got, ref)
    assert np.all(np.abs(got - ref) <= 1e-5 * np.abs(v).max())


@pytest.mark.parametrize("b,h,s,sk,d", [(1, 1, 128, 1024, 64), (1, 2, 2048, 2048, 64), (1, 1, 100, 512, 32), (12, 1, 100, 512, 48),
                                        (8, 12, 512, 512, 32), (4, 12, 197, 197, 64)])
def test_long_heads_take_the_faster_form(hip, b, h, s, sk, d):
    """Few heads over many keys run the three nodes, which spread over the chip (one head of 128 rows and 1024 keys: 22
    us, 57 in one launch), and bit for bit so; the fused graph is never much slower than its nodes."""
    model, ins = attention_model(b, h, s, sk, d, d, "b11s", "div")
    kept, _ = attention_model(b, h, s, sk, d, d, "b11s", "div", extra_outputs=("sc",))
    dev = {k: DeviceTensor.from_numpy(v) for k, v in ins.items()}
    g, g3 = Model.Load(model), Model.Load(kept)
    g.Fuse()
    g3.Fuse()
    assert g.Execute(dev) and g3.Execute(dev), (g.LastError, g3.LastError)
    assert same_bits(g.Output("y").to_numpy(), g3.Output("y").to_numpy()) == (b * h < 48)
    assert g.Capture(dev) and g3.Capture(dev)
    best = [1e9, 1e9]
    for _ in range(5):
        for i, x in enumerate((g, g3)):
            assert x.Replay()
            onnx_amd.synchronize()
            t = time.perf_counter()
            for _ in range(20):
                x.Replay()
            onnx_amd.synchronize()
            best[i] = min(best[i], time.perf_counter() - t)
    assert best[0] < 1.3 * best[1], best
