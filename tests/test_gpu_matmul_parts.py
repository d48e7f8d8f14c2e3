"""Float MatMul over K ranges of 256 and more, where every operand is split into three bf16 parts and multiplied on
the bf16 matrix unit (lx_matmul.hip, k_matmul_f32_b3).

Bar: every part product is exact and each of a step's six MFMAs rounds its accumulation once, so a dot product of K
terms is within (6 ceil(K / 16) + 1) 2^-24 sum_j |a_j b_j| of the exact one (the part products left out weigh 2^-25),
and within the MatMul bar of 1e-5 sum_j |a_j b_j|."""
import time

import numpy as np
import pytest

import onnx_amd
from onnx_amd import DeviceTensor, HipExecutionProvider as HIP, OpStatus

pytestmark = pytest.mark.gpu


def dev(a):
    return DeviceTensor.from_numpy(np.asarray(a))


def mm(a, b):
    r = HIP.MatMul(dev(a), dev(b))
    assert r.Status == OpStatus.Success, r.Message
    return r.Outputs[0].to_numpy()


def check(a, b, got=None):
    got = (mm(a, b) if got is None else got).astype(np.float64)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bar = min(1e-5, (6 * -(-a.shape[-1] // 16) + 1) * 2.0 ** -24)
    err, mag = np.abs(got - a64 @ b64), np.abs(a64) @ np.abs(b64)
    assert np.all(err <= bar * mag + 2.0 ** -140), float((err / (mag + 1e-300)).max())


# Every form of the kernel: the tiles with whole pairs of steps (128x128, 128x64, 64x64 several per CU, 64x64 with loading
# waves), K tails in 16-byte loads (128x128 and 64x64) and in scalar ones (both), the ranges of a split product
FORMS = [(4096, 256, 1024), (1100, 384, 960), (4096, 256, 1152), (1024, 576, 512), (1536, 516, 1600), (600, 516, 516),
         (1500, 533, 1601), (256, 533, 70), (640, 3072, 640)]
# and edges in both directions, single rows and few columns, the first K with a CU per tile
SHAPES = FORMS + [(4096, 384, 384), (1000, 320, 4100), (788, 768, 768), (129, 516, 65), (2000, 260, 2020), (700, 533, 260),
                  (127, 513, 33), (2048, 1001, 1030), (1, 4100, 500), (300, 1000, 36), (700, 768, 768), (5, 700, 37),
                  (1100, 516, 512), (100, 600, 70)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_parts_tiles_and_edges(hip, m, k, n):
    rng = np.random.default_rng(m + k + n)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    check(a, b)


def test_parts_batches(hip):
    rng = np.random.default_rng(3)
    for sa, sb in [((30, 1, 130, 256), (1, 2, 256, 132)), ((70, 65, 300), (70, 300, 67))]:
        check(rng.standard_normal(sa).astype(np.float32), rng.standard_normal(sb).astype(np.float32))


@pytest.mark.parametrize("m,k,n", FORMS + [(1090, 333, 1000)])
@pytest.mark.parametrize("kind", ["tiny", "tiny_times_huge", "one_tiny", "huge", "mixed", "not_finite"])
def test_parts_of_extreme_values(hip, m, k, n, kind):
    """Values whose parts bf16 cannot hold take the fp32 MFMA: subnormal operands, subnormal times huge, a row's only
    product that of a subnormal beside larger values, values that round to an infinite bf16, rows over 45 decades, and
    infinities and NaN (the same pattern as float32's)."""
    rng = np.random.default_rng(7)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    if kind == "tiny":
        a = (a * 1e-36).astype(np.float32)
    elif kind == "tiny_times_huge":
        a, b = (a * 1e-41).astype(np.float32), (b * np.float32(1e20)).astype(np.float32)
    elif kind == "one_tiny":
        a[::5], a[::5, 7], a[::5, 9] = 0, 1e-41, 1
        b[7], b[9] = b[7] * np.float32(1e15), 0
        b[:, ::7], b[7, ::7], b[9, ::7] = 0, 1e-41, 1  # columns likewise
        a[1::5, 7], a[1::5, 9] = 1e15, 0
    elif kind == "huge":
        a[::3, 5] = np.float32(3.4e38)
        b[5, :] = 0.25
    elif kind == "mixed":
        a = (a * 10.0 ** rng.uniform(-30, 15, a.shape)).astype(np.float32)
    else:
        a[0, 0], a[2, 5], b[7, 0] = np.nan, np.inf, -np.inf
        a[3, :], b[:, 2] = 0, 0
        got = mm(a, b)
        with np.errstate(all="ignore"):
            ref = a @ b
        assert np.array_equal(np.isnan(ref), np.isnan(got))
        inf = np.isinf(ref)
        assert np.array_equal(inf, np.isinf(got)) and np.array_equal(ref[inf], got[inf])
        rows = [i for i in range(m) if i not in (0, 2)]
        cols = [j for j in range(n) if j != 0]
        check(a[rows], b[:, cols], got[np.ix_(rows, cols)])
        return
    check(a, b)


def float32_chain(a, b):
    """The products one after another in float32, each exact before it is added (a chain of fused multiply-adds, which
    v_mfma_f32_32x32x2f32 is): float64 holds a product's 48 bits and adds it with an error far below a float32's."""
    acc = np.zeros((a.shape[0], b.shape[1]), np.float32)
    a, b = a.astype(np.float64), b.astype(np.float64)
    for j in range(a.shape[1]):
        acc = (acc + a[:, j:j + 1] * b[j]).astype(np.float32)
    return acc


# 128x64, 64x64, 128x128 tiles, loading waves, a split product, scalar loads with a tail
@pytest.mark.parametrize("m,k,n", [(1100, 384, 960), (600, 516, 516), (788, 768, 2500), (700, 768, 768), (640, 3072, 640),
                                   (1090, 333, 1000)])
@pytest.mark.parametrize("dense", [1.0, 0.5, 0.1, 0.02, "both", "positive", "small"])
def test_parts_error_is_no_larger_than_a_float32_chain(hip, m, k, n, dense):
    """Against 64 bits, dense and sparse operands (a float32 chain does not round on a zero)."""
    rng = np.random.default_rng(19)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    if dense == "positive":
        a, b = np.abs(a), np.abs(b)
    elif dense == "small":  # small part products of subnormal size, results just above where they run again
        a, b = a * np.float32(2.0 ** -58), b * np.float32(2.0 ** -58)
    elif dense == "both":
        a, b = a * (rng.random(a.shape) < 0.1), b * (rng.random(b.shape) < 0.1)
    else:
        a *= rng.random(a.shape) < dense
    got = mm(a.astype(np.float32), b.astype(np.float32)).astype(np.float64)
    rows, cols = slice(0, 64), slice(0, min(n, 512))
    exact, chain = a[rows].astype(np.float64) @ b[:, cols].astype(np.float64), float32_chain(a[rows], b[:, cols])
    assert np.linalg.norm(got[rows, cols] - exact) <= np.linalg.norm(chain - exact)


@pytest.mark.parametrize("m,k,n,r", [(60, 2560, 4096, 4), (256, 3072, 768, 4), (384, 3072, 768, 3)])
def test_short_ranges_of_a_split_product_keep_float32(hip, m, k, n, r):
    """Ranges of up to 1024 run on the fp32 MFMA, where they are faster: each partial product is the bits of a float32
    chain of steps of 16, k = j and then k = 8 + j of each (j = 0..7), and the partials are added in order."""
    rng = np.random.default_rng(23)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    order = np.arange(k).reshape(-1, 2, 8).transpose(0, 2, 1).reshape(-1)
    got, cols = mm(a, b), slice(n - 64, n)
    ref = np.zeros((8, 64), np.float32)
    for i in range(r):
        o = order[i * (k // r):(i + 1) * (k // r)]
        part = float32_chain(a[:8, o], b[o, cols])
        ref = part if i == 0 else ref + part
    assert np.array_equal(got[:8, cols], ref)


@pytest.mark.parametrize("b,m,k,n", [(96, 512, 512, 64), (96, 100, 640, 64), (4, 512, 512, 512)])
def test_narrow_and_lone_products_keep_float32(hip, b, m, k, n):
    """64 columns with K below 1024, and K up to 512 with a CU per tile, run on the fp32 MFMA: a float32 chain."""
    rng = np.random.default_rng(27)
    a, w = rng.standard_normal((b, m, k)).astype(np.float32), rng.standard_normal((b, k, n)).astype(np.float32)
    order = np.arange(k).reshape(-1, 2, 8).transpose(0, 2, 1).reshape(-1)
    got = mm(a, w)
    assert np.array_equal(got[1, :64], float32_chain(a[1, :64][:, order], w[1][order]))


@pytest.mark.parametrize("m,k,n", [(4096, 768, 768), (788, 768, 768), (1100, 384, 1000)])
def test_parts_time_does_not_depend_on_zeros(hip, m, k, n):
    """Exactly zero results of nonzero rows and columns (integers, sparse operands, a selection) and small values need
    no second run on the fp32 MFMA (which takes 3.4 to 5.5 times as long): the time of normal data, and integer
    products are exact."""
    rng = np.random.default_rng(17)
    normal = [rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n))]
    small = [rng.integers(-8, 9, s).astype(np.float32) for s in ((m, k), (k, n))]
    signs = [rng.integers(-1, 2, s).astype(np.float32) for s in ((m, k), (k, n))]
    one = np.zeros((m, k), np.float32)
    one[np.arange(m), rng.integers(0, k, m)] = 1
    half = (normal[1] * (rng.random((k, n)) < 0.5)).astype(np.float32)
    for a, b in (small, signs, [one, half]):
        assert np.array_equal(mm(a, b), a.astype(np.float64) @ b.astype(np.float64))
    y = DeviceTensor.empty((m, n), np.float32)
    calls = {}
    for name, (a, b) in {"normal": normal, "small": small, "signs": signs, "selected": (one, half),
                         "tiny": (normal[0], (normal[1] * 1e-24).astype(np.float32))}.items():
        calls[name] = (dev(a), dev(b))
    best = dict.fromkeys(calls, 1e9)
    for _ in range(5):
        for name, (a, b) in calls.items():
            HIP.MatMul(a, b, out=y)
            onnx_amd.synchronize()
            t = time.perf_counter()
            for _ in range(50):
                HIP.MatMul(a, b, out=y)
            onnx_amd.synchronize()
            best[name] = min(best[name], time.perf_counter() - t)
    assert max(best.values()) < 2 * best["normal"], best


def test_parts_results_do_not_depend_on_the_tile(hip):
    """The same bits alone and inside a larger product, extreme rows (which take the fp32 MFMA) included (parts of more
    than 256 tiles of 64x64: fewer keep the fp32 MFMA at this K, or split K and sum other ranges)."""
    rng = np.random.default_rng(11)
    a, b = rng.standard_normal((4096, 320)).astype(np.float32), rng.standard_normal((320, 1024)).astype(np.float32)
    a[10] *= np.float32(1e-38)
    a[70, 3], b[4, 500] = np.inf, np.float32(1e-40)
    whole = mm(a, b)
    for rows, cols in [(slice(0, 2048), slice(0, 576)), (slice(0, 2200), slice(448, 1024))]:
        part = mm(np.ascontiguousarray(a[rows]), np.ascontiguousarray(b[:, cols]))
        assert np.array_equal(part.view(np.uint32), whole[rows, cols].view(np.uint32))


def test_parts_of_a_long_k_do_not_depend_on_the_tile(hip):
    """K = 576: 64x64 tiles whole, its parts 128x128, 128x64 and 64x64 with loading waves; rows of subnormals and a few
    values that are not finite run on the fp32 MFMA in each."""
    rng = np.random.default_rng(12)
    a, b = rng.standard_normal((4096, 576)).astype(np.float32), rng.standard_normal((576, 1152)).astype(np.float32)
    a[10] *= np.float32(1e-38)
    a[900, 500], a[70, 3], b[4, 500], b[300, 20] = np.nan, np.inf, np.float32(1e-40), -np.inf
    whole = mm(a, b)
    for rows, cols in [(slice(0, 2048), slice(0, 1152)), (slice(0, 1024), slice(0, 1152)), (slice(0, 1024), slice(0, 512))]:
        part = mm(np.ascontiguousarray(a[rows]), np.ascontiguousarray(b[:, cols]))
        nan = np.isnan(whole[rows, cols])
        assert np.array_equal(np.isnan(part), nan)
        assert np.array_equal(part[~nan].view(np.uint32), whole[rows, cols][~nan].view(np.uint32))


@pytest.mark.parametrize("s,d", [(640, 256), (512, 320), (301, 515)])
def test_parts_of_a_right_operand_by_columns(hip, s, d):
    """A transposed right operand folded into the product is read by columns: bit for bit the Transpose and MatMul
    nodes (128x128 and 64x64 tiles, 16-byte and scalar loads, a K tail)."""
    import onnx_writer as W
    from onnx_amd.graph import Model
    rng = np.random.default_rng(13)
    ins = {t: rng.standard_normal((2, s, 4, d)).astype(np.float32) for t in "qk"}
    nodes = [W.node("Transpose", ["q"], ["qt"], "tq", perm=[0, 2, 1, 3]),
             W.node("Transpose", ["k"], ["kt"], "tk", perm=[0, 2, 3, 1]), W.node("MatMul", ["qt", "kt"], ["y"], "mm")]
    model = W.model(nodes, [(t, np.float32, v.shape) for t, v in ins.items()], [("y", np.float32, ())], [])
    d_in = {t: dev(v) for t, v in ins.items()}
    res = []
    for fuse in (False, True):
        g = Model.Load(model)
        if fuse:
            assert g.Fuse() == 1 and [x.Op for x in g.Nodes] == ["MatMulPermuted"]
        assert g.Execute(d_in), g.LastError
        res.append(g.Output("y").to_numpy())
    assert np.array_equal(res[0].view(np.uint32), res[1].view(np.uint32))
    check(ins["q"].transpose(0, 2, 1, 3), ins["k"].transpose(0, 2, 3, 1), res[1])


@pytest.mark.parametrize("b,m,k,n", [(192, 8, 384, 384), (600, 4, 320, 512), (40, 220, 1536, 96)])
@pytest.mark.parametrize("side", ["left", "result"])
def test_a_shared_right_operand_is_the_same_bits_folded_or_not(hip, b, m, k, n, side):
    """A product whose left matrices all meet one right matrix runs as one product of their rows where these are
    dense, and batch by batch where the Transpose before or after it is folded in: both choose their unit by the rows of
    the whole batch (the fp32 MFMA, parts of a short and of a long K)."""
    import onnx_writer as W
    from onnx_amd.graph import Model
    rng = np.random.default_rng(29)
    x = rng.standard_normal((m, b, k) if side == "left" else (b, m, k)).astype(np.float32)
    w = rng.standard_normal((k, n)).astype(np.float32)
    nodes = ([W.node("Transpose", ["x"], ["t"], "t", perm=[1, 0, 2]), W.node("MatMul", ["t", "w"], ["y"], "mm")]
             if side == "left" else
             [W.node("MatMul", ["x", "w"], ["t"], "mm"), W.node("Transpose", ["t"], ["y"], "t", perm=[1, 0, 2])])
    res = []
    for fuse in (False, True):
        g = Model.Load(W.model(nodes, [("x", np.float32, x.shape)], [("y", np.float32, ())], [("w", w)]))
        if fuse:
            assert g.Fuse() == 1 and [v.Op for v in g.Nodes] == ["MatMulPermuted"]
        assert g.Execute({"x": dev(x)}), g.LastError
        res.append(g.Output("y").to_numpy())
    assert np.array_equal(res[0].view(np.uint32), res[1].view(np.uint32))
    check(x.swapaxes(0, 1) if side == "left" else x, w, res[0] if side == "left" else res[0].swapaxes(0, 1))


@pytest.mark.parametrize("b,m,k,n", [(192, 8, 384, 384), (600, 4, 320, 512)])
def test_a_bias_row_per_batch_keeps_the_products_bits(hip, b, m, k, n):
    rng = np.random.default_rng(31)
    x, w = rng.standard_normal((b, m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    bias = rng.standard_normal((b, 1, n)).astype(np.float32)
    r = HIP.MatMulAdd(dev(x), dev(w), dev(bias))
    assert r.Status == OpStatus.Success, r.Message
    assert np.array_equal(r.Outputs[0].to_numpy(), mm(x, w) + bias)


def test_a_large_batch_runs_on_one_unit(hip):
    """Batches above 65535 run in several launches: the last, short one keeps the unit of the others."""
    rng = np.random.default_rng(37)
    a, b = rng.standard_normal((41, 1600, 1, 256)).astype(np.float32), rng.standard_normal((1600, 256, 33)).astype(np.float32)
    a[40] = a[0]
    got = mm(a, b)
    assert np.array_equal(got[40], got[0])
    check(a[0], b, got[0])
