"""Window-stationary layers of one fragment per wavefront with K in halves (at most 256 workgroups, 24 K-steps, four channel
blocks and more, an even number) and beside the rule's edges, against the oracle: taps, strides, windows of one and of several blocks, every epilogue."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, taps, stride
    (4, 256, 7, 7, 128, 3, 1),       # two blocks each
    (32, 512, 7, 7, 96, 3, 1),       # channels that do not fill the last wavefront
    (2, 448, 9, 8, 130, 3, 1),       # seven blocks: not in halves
    (8, 512, 14, 13, 64, 3, 2),
    (6, 640, 5, 5, 128, 5, 1),
    (30, 2048, 7, 7, 100, 1, 1),     # a window of four blocks
    (9, 1100, 6, 7, 255, 1, 1),      # 18 K-steps: not in halves
    (9, 1536, 6, 7, 255, 1, 1),      # 24
]


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: "-".join(map(str, c)))
def test_conv_i8_k_halves(port, monkeypatch, case):
    from tennis_amd import capi
    for kernel in ("KS", "PX", "FLAT", "RS"):
        monkeypatch.setenv("TSX_CONV_I8_" + kernel, "0")
    n, c, h, w, cout, k, s = case
    rng = np.random.default_rng(13)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, k, k)).astype(np.int8)
    dq = (rng.uniform(1e-5, 3e-5, cout) * 30 / np.sqrt(c) / k).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    pads = (k // 2,) * 4
    conv = capi.Conv2dI8(dev(wt), pads, (s, s))
    st = capi.StagedInput(conv, x.shape)
    conv.stage(dev(x), st)
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq, pads, (s, s), (1, 1)), bias)
    res = rng.standard_normal(plain.shape).astype(np.float32)
    second = capi.Conv2dI8(dev(np.zeros((32, cout, 3, 3), np.int8)), (1, 1, 1, 1))
    y = conv.run_staged(st, dev(dq), dev(bias))[0]
    assert np.array_equal(bits(y.cpu().numpy()), bits(plain))
    for joined in (None, res):
        exp = port.relu(plain if joined is None else (plain + joined).astype(np.float32))
        out = capi.StagedInput(second, plain.shape)
        y = conv.run_staged(st, dev(dq), dev(bias), "relu", residual=dev(joined), q_scales=dev(qs), staged_out=out)[0]
        assert np.array_equal(bits(y.cpu().numpy()), bits(exp))
        assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), port.quantize(exp, qs))
    mish = capi.StagedInput(second, plain.shape)
    y = conv.run_staged(st, dev(dq), dev(bias), "mish", q_scales=dev(qs), staged_out=mish)[0]
    assert np.array_equal(capi.staged_interior(mish, range(n)).cpu().numpy(), port.quantize(y.cpu().numpy(), qs))
