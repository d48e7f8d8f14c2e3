"""Split float products of few rows in one launch (lx_matmul.hip, k_matmul_small): the bits of the ordered sum of the
products of their K ranges, each run whole by the fp32 MFMA, and the bits of the MatMul, Add and GELU calls that the
fused entry points stand for."""
import numpy as np
import pytest

from onnx_amd import DeviceTensor, HipExecutionProvider as HIP, OpStatus

pytestmark = pytest.mark.gpu


def dev(a):
    return DeviceTensor.from_numpy(np.asarray(a))


def out(r):
    assert r.Status == OpStatus.Success, r.Message
    return r.Outputs[0].to_numpy()


def same(x, y):
    assert x.shape == y.shape and np.array_equal(x.view(np.uint32), y.view(np.uint32))


# one row to the limit of 64 and the first past it (65: the tiles), ragged row groups and columns, two ranges (half a
# wave) to the limit of 64, a count that is no whole number of waves, the first K past the limit, a batch
SHAPES = [(1, 128, 4, 1), (3, 384, 36, 1), (8, 1536, 384, 1), (32, 384, 1536, 1), (33, 832, 100, 1), (64, 512, 132, 1),
          (65, 512, 132, 1), (1, 4096, 64, 1), (1, 4160, 64, 1), (5, 320, 20, 3)]


@pytest.mark.parametrize("m,k,n,batch", SHAPES)
def test_small_products_sum_their_ranges_in_order(hip, m, k, n, batch):
    rng = np.random.default_rng(m + k + n)
    a = (rng.standard_normal((batch, m, k)) * 10.0 ** rng.uniform(-3, 3, (batch, m, k))).astype(np.float32)
    b = rng.standard_normal((batch, k, n)).astype(np.float32)
    a[..., k // 2] = 0
    got = out(HIP.MatMul(dev(a), dev(b)))
    # each range as a product of its own: K = 64 does not split
    tiles = -(-m // 64) * -(-n // 64) * batch
    r = max(r for r in range(1, k // 64 + 1) if (k // 64) % r == 0 and tiles * r <= 256)
    assert k // r == 64
    ref = None
    for i in range(r):
        part = out(HIP.MatMul(dev(a[..., 64 * i:64 * i + 64]), dev(np.ascontiguousarray(b[:, 64 * i:64 * i + 64]))))
        ref = part if ref is None else (ref + part).astype(np.float32)
    same(got, ref)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - a64 @ b64) <= 1e-5 * (np.abs(a64) @ np.abs(b64)))


@pytest.mark.parametrize("m,k,n", [(8, 384, 384), (7, 1536, 60), (64, 384, 1536)])
def test_small_products_with_epilogues(hip, m, k, n):
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32) / 8
    bias, res = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    mm = out(HIP.MatMul(dev(a), dev(b)))
    add = out(HIP.MatMulAdd(dev(a), dev(b), dev(bias)))
    same(add, mm + bias)
    same(out(HIP.MatMulAdd(dev(a), dev(b), dev(bias), dev(res))), (mm + bias) + res)
    same(out(HIP.MatMulAddGelu(dev(a), dev(b), dev(bias))), out(HIP.GeluErf(dev(add))))


def test_small_products_of_not_finite_values(hip):
    rng = np.random.default_rng(6)
    a, b = rng.standard_normal((9, 384)).astype(np.float32), rng.standard_normal((384, 40)).astype(np.float32)
    a[0, 0], a[2, 100], b[200, 3], a[4, :], b[7, 7] = np.nan, np.inf, -np.inf, 0, 1e-44
    got = out(HIP.MatMul(dev(a), dev(b)))
    with np.errstate(all="ignore"):
        ref = a @ b
    assert np.array_equal(np.isnan(ref), np.isnan(got))
    inf = np.isinf(ref)
    assert np.array_equal(inf, np.isinf(got)) and np.array_equal(ref[inf], got[inf])


@pytest.mark.parametrize("m,n,batch", [(8, 384, 1), (64, 256, 1), (5, 192, 3)])
def test_small_products_over_their_operands(hip, m, n, batch):
    """A result stored over the left operand, or over the residual: the bits of a result of its own."""
    rng = np.random.default_rng(8)
    for _ in range(5):
        a, b = (rng.standard_normal((batch, r, n)).astype(np.float32) for r in (m, n))
        bias, ref = rng.standard_normal(n).astype(np.float32), out(HIP.MatMul(dev(a), dev(b)))
        x, r = dev(a), dev(a)
        same(out(HIP.MatMul(x, dev(b), out=x)), ref)
        x = dev(a)
        same(out(HIP.MatMulAdd(x, dev(b), dev(bias), x, out=x)), (ref + bias) + a)
        same(out(HIP.MatMulAdd(dev(a), dev(b), dev(bias), r, out=r)), (ref + bias) + a)
