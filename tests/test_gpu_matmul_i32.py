"""Int32 MatMul, mostly on the int8 matrix unit (lx_matmul.hip, k_matmul_i32 and k_matmul_i32_few): whole wrapping
products, bit for bit against int64 sums modulo 2^32."""
import numpy as np
import pytest

from onnx_amd import DeviceTensor, HipExecutionProvider as HIP, OpStatus

pytestmark = pytest.mark.gpu


def mm(a, b):
    r = HIP.MatMul(DeviceTensor.from_numpy(a), DeviceTensor.from_numpy(b))
    assert r.Status == OpStatus.Success, r.Message
    return r.Outputs[0].to_numpy()


def wrapped(a, b):
    with np.errstate(over="ignore"):  # numpy's int64 sums wrap modulo 2^64, which keeps them modulo 2^32
        return np.matmul(a.astype(np.int64), b.astype(np.int64)).astype(np.uint64).astype(np.uint32).view(np.int32)


# Small products of K up to 96 on the VALU: one element, less and more than a tile; 32x32 tiles with K dealt out to three to
# eight waves: the first K past the VALU's, a round of 256, K no multiple of 4 (16 bytes at 4-byte alignment), batches,
# the K after which a wave folds its accumulators and past it; then 64x64 tiles (more than 128 of them) likewise, N a
# multiple of 4 (16-byte stores) over several column blocks and not
@pytest.mark.parametrize("batch,m,k,n", [(1, 1, 1, 1), (1, 31, 31, 33), (1, 64, 64, 64), (1, 33, 97, 31), (2, 300, 70, 301),
                                         (1, 3, 257, 130), (6, 96, 384, 96), (1, 2, 131072, 5), (1, 1, 131121, 4),
                                         (130, 1, 1, 1), (33, 65, 68, 65), (44, 63, 130, 129), (33, 65, 100, 68), (6, 384, 384, 384), (130, 2, 16384, 3),
                                         (130, 1, 16449, 4)])
@pytest.mark.parametrize("kind", ["any", "extreme"])
def test_int32_products(hip, batch, m, k, n, kind):
    rng = np.random.default_rng(m * 7 + k + n)
    if kind == "any":
        a, b = (rng.integers(-2**31, 2**31, s, dtype=np.int64).astype(np.int32) for s in ((batch, m, k), (batch, k, n)))
    else:  # every digit -128 or 127, and the type's ends
        v = np.array([0x7F7F7F80, 0x7F7F7F7F, -2**31, 2**31 - 1, -1, 0], np.int64).astype(np.int32)
        a, b = (v[rng.integers(0, 6, s)] for s in ((batch, m, k), (batch, k, n)))
        a[:, 0], b[..., 0] = v[0], v[0]  # the largest digit sums: -128 times -128 throughout
    assert np.array_equal(mm(a, b), wrapped(a, b))


def test_int32_products_of_broadcast_batches_and_unaligned_results(hip):
    """64x64 tiles over broadcast batches, and results at an address that 16-byte stores cannot take."""
    rng = np.random.default_rng(3)
    for sa, sb in [((3, 1, 33, 97), (1, 50, 97, 36)), ((50, 40, 130), (50, 130, 132))]:
        a, b = (rng.integers(-2**31, 2**31, s, dtype=np.int64).astype(np.int32) for s in (sa, sb))
        ref = wrapped(a, b)
        assert np.array_equal(mm(a, b), ref)
        base = DeviceTensor.from_numpy(np.full(ref.size + 2, 7, np.int32))
        out = DeviceTensor.wrap(base.h.data + 4, ref.shape, np.int32, ref.nbytes, keepalive=base)
        r = HIP.MatMul(DeviceTensor.from_numpy(a), DeviceTensor.from_numpy(b), out=out)
        assert r.Status == OpStatus.Success, r.Message
        assert np.array_equal(out.to_numpy(), ref)
        edge = base.to_numpy()
        assert edge[0] == 7 and edge[-1] == 7
