"""Kernels that take whole planes or rows at once, at the sizes where that can go wrong: global pooling around its chunk
and plane-group sizes, 3x3 stride-2 max pooling and 3x3 depthwise convolution across row groups, borders and wavefronts
that end inside a row, batch norm around the plane size it switches at; bit for bit against the oracle."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("shape", [(1, 1, 4, 4), (1, 17, 3, 7), (3, 11, 16, 32), (2, 9, 19, 27), (1, 33, 37, 41), (2, 3, 1, 31), (2, 3, 4, 8), (1, 5, 3, 33),
                                   (1, 3, 24, 24), (2, 9, 34, 32),
                                   (3, 19, 7, 7), (1, 5, 7, 9), (1, 3, 5, 19), (1, 3, 8, 12), (2, 3, 17, 33)])
@pytest.mark.parametrize("kind", ["avg", "max"])
def test_global_pooling(port, shape, kind):
    from tennis_amd import capi
    x = np.random.default_rng(1).standard_normal(shape).astype(np.float32)
    x.ravel()[::11] = -0.0
    x.ravel()[0] = np.nan
    got = capi.global_pooling2d(_dev(x), kind).cpu().numpy()
    assert np.array_equal(bits(got), bits(port.global_pooling2d(x, kind).reshape(got.shape)))


@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 3, 5, 8), (1, 7, 9, 12), (3, 5, 14, 28), (1, 40, 15, 20), (2, 2, 56, 260)])
def test_max_pooling_3x3_stride_2(port, shape):
    from tennis_amd import capi
    x = np.random.default_rng(2).standard_normal(shape).astype(np.float32)
    x.ravel()[::7] = -0.0
    x.ravel()[-3:] = np.nan
    for pads in ((1, 1, 1, 1), (1, 0, 1, 0)):
        got = capi.pooling2d(_dev(x), "max", (3, 3), (2, 2), pads).cpu().numpy()
        exp = port.pooling2d(x, "max", (3, 3), (2, 2), pads)
        assert got.shape == exp.shape and np.array_equal(bits(got), bits(exp)), pads


@pytest.mark.parametrize("shape", [(1, 1, 1, 4), (2, 3, 5, 8), (1, 5, 6, 12), (2, 9, 13, 28), (1, 3, 8, 260)])
@pytest.mark.parametrize("pads", [(1, 1, 1, 1), (0, 2, 1, 1), (2, 0, 1, 1)])
def test_depthwise_3x3(port, shape, pads):
    from tennis_amd import capi
    if shape[2] + pads[0] + pads[1] < 3:
        pytest.skip("no output row")
    rng = np.random.default_rng(3)
    x = rng.standard_normal(shape).astype(np.float32)
    w = rng.standard_normal((1, shape[1], 3, 3)).astype(np.float32)
    bias = rng.standard_normal(shape[1]).astype(np.float32)
    got = capi.depthwise_conv2d(_dev(x), _dev(w), pads, padding_value=0.5, bias=_dev(bias), act="relu").cpu().numpy()
    exp = port.relu(port.add_bias(port.depthwise_conv2d(x, w, pads, padding_value=0.5), bias))
    assert got.shape == exp.shape and np.array_equal(bits(got), bits(exp))


@pytest.mark.parametrize("shape", [(4, 256, 16, 16), (1, 1025, 15, 20), (2, 512, 12, 21), (33, 32, 36, 29), (2, 512, 46, 46), (4, 256, 32, 32), (4, 256, 28, 37)])
def test_plane_batch_norm(port, shape):
    from tennis_amd import capi
    rng = np.random.default_rng(4)
    x = rng.standard_normal(shape).astype(np.float32)
    mean, var, scale, bias = (rng.uniform(0.1, 2, shape[1]).astype(np.float32) for _ in range(4))
    d = [_dev(v) for v in (x, mean, var, scale, bias)]
    for got, exp in ((capi.batch_norm(*d[:3]), port.batch_norm(x, mean, var)), (capi.batch_scale(d[0], d[3], d[4]), port.batch_scale(x, scale, bias)),
                     (capi.fused_batch_norm(*d), port.fused_batch_norm(x, mean, var, scale, bias))):
        assert np.array_equal(bits(got.cpu().numpy()), bits(exp))


@pytest.mark.parametrize("m,k,n", [(1, 256, 16), (32, 256, 1000), (17, 257, 33), (5, 300, 100), (64, 511, 20), (3, 512, 40), (2, 513, 17), (33, 1024, 31),
                                   (4, 1025, 50), (16, 2048, 65)])
@pytest.mark.parametrize("transpose", [False, True])
def test_inner_product_of_few_rows(m, k, n, transpose):
    """Sums of small whole numbers, exact in any order: every K block counted once, whatever the ring holds of them."""
    from tennis_amd import capi
    rng = np.random.default_rng(k)
    a, b = rng.integers(-8, 9, (m, k)).astype(np.float32), rng.integers(-8, 9, (k, n)).astype(np.float32)
    got = capi.inner_prod_f32(_dev(a), _dev(b.T if transpose else b), transpose=transpose).cpu().numpy()
    assert np.array_equal(got, a @ b)
