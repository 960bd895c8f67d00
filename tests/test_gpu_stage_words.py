"""Staging by im2col with a dword per byte (kernels of three and more columns on up to 8 channels): one, two and four output
rows per workgroup, runs of 252 columns that end at and inside a patch row, K that ends inside a dword, dilated rows, strides,
quantized on the way or not; through the convolution, against the CPU oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("case", [
    # n, c, h, w, kh, kw, pads, strides, row dilation
    (1, 3, 20, 248, 3, 3, (1, 1, 1, 1), (1, 1), 1),         # a patch row of 63 lanes
    (1, 3, 9, 252, 3, 3, (1, 1, 4, 4), (1, 1), 1),
    (2, 1, 7, 4, 7, 7, (3, 3, 3, 3), (2, 2), 1),            # K of 49 bytes
    (3, 8, 33, 132, 2, 5, (0, 1, 0, 2), (2, 3), 3),
    (1, 5, 12, 40, 3, 4, (2, 0, 2, 3), (3, 1), 2),
    (1, 3, 9, 61, 3, 3, (1, 1, 1, 1), (1, 1), 1),           # by bytes: the width
    (20, 3, 50, 12, 7, 9, (3, 3, 3, 3), (2, 4), 1),         # two rows per workgroup (of 25)
    (64, 2, 67, 12, 3, 3, (1, 1, 1, 1), (1, 1), 1),         # four; a last group of three rows
])
@pytest.mark.parametrize("quantize", [False, True])
def test_stage_words(port, case, quantize):
    from tennis_amd import capi
    n, c, h, w, kh, kw, pads, st, dil = case
    rng = np.random.default_rng(64)
    wt = rng.integers(-127, 128, (24, c, kh, kw)).astype(np.int8)
    dq = rng.uniform(1e-4, 3e-4, 24).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt), pads, st, (dil, 1), padding_value=-3.0)
    if quantize:
        x, scales = rng.standard_normal((n, c, h, w)).astype(np.float32), rng.uniform(20, 40, n).astype(np.float32)
        xq = port.quantize(x, scales)
        got = conv(dev(x), dq=dev(dq), x_scales=dev(scales))[0]
    else:
        xq = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
        got = conv(dev(xq), dq=dev(dq))[0]
    exp = port.conv2d_quantized(xq, wt, dq, pads, st, (dil, 1), padding_value=-3.0)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), exp.view(np.uint32))
