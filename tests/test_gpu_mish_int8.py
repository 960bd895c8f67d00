"""Layers with the exact Mish that hand out nothing but requantized int8 values, at every kind of pre-activation: weights of zero
make it the bias, so the biases are the floats to try -- bit patterns of the whole range, infinities and NaN, arguments whose
product with the scale lies next to a rounding boundary, the ends at which the exact form clamps its argument."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def arguments(port, scales, count):
    rng = np.random.default_rng(411)
    x = [rng.integers(0, 1 << 32, count, dtype=np.uint64).astype(np.uint32).view(np.float32),
         rng.uniform(-25, 45, count).astype(np.float32), (rng.standard_normal(count) * 3).astype(np.float32),
         np.float32([0.0, -0.0, np.inf, -np.inf, np.nan, 3.4e38, -3.4e38, 1e-45, -1e-45, 20, -20, 40, -40, 88.8, -88.8, -1.19, 1e10, -1e10])]
    # mish(x) * s = k + 1/2: x by bisection on the increasing branch, then its neighbours
    for s in scales:
        k = (rng.integers(-int(abs(s) * 0.3), 130, count // 8) + 0.5) / abs(s)
        lo, hi = np.full(k.shape, -1.19), np.full(k.shape, 200.0)
        for _ in range(60):
            mid = (lo + hi) / 2
            above = mid * np.tanh(np.log1p(np.exp(mid))) > k
            lo, hi = np.where(above, lo, mid), np.where(above, mid, hi)
        at = lo.astype(np.float32)
        for step in range(-3, 4):
            x.append((at.view(np.int32) + step).view(np.float32))
    x = np.concatenate(x)
    return x[:len(x) // 32 * 32]


@pytest.mark.parametrize("images", [1, 2])
@pytest.mark.parametrize("side", [4, 20])       # one fragment per wavefront; two
@pytest.mark.parametrize("join", [None, "before", "after"])
def test_every_kind_of_argument(port, monkeypatch, images, side, join):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    scales = np.float32([37.5, -3.0])[:images]
    bias = arguments(port, scales, 2048)
    cout = len(bias)
    rng = np.random.default_rng(5)
    conv = capi.Conv2dI8(dev(np.zeros((cout, 16, 1, 1), np.int8)), (0, 0, 0, 0))
    x = rng.integers(-128, 128, (images, 16, side, side)).astype(np.int8)
    plain = np.broadcast_to(bias[None, :, None, None], (images, cout, side, side)).copy()
    res = None
    if join:
        res = rng.standard_normal(plain.shape).astype(np.float32)
        res[:, ::3] = np.float32([0, 100, -1e9, 3e38, np.inf, np.nan, 1e-30])[rng.integers(0, 7, res[:, ::3].shape)]
    with np.errstate(all="ignore"):
        plain = port.add(plain, np.zeros_like(plain)) if join != "before" else port.add(plain, res)      # 0 * dq + bias
        value = port.mish(plain) if join != "after" else port.add(port.mish(plain), res)
        expected = port.quantize(value, scales)
    staged = capi.StagedInput(conv, x.shape)
    conv.stage(dev(x), staged)
    q = conv.run_staged(staged, dev(np.ones(cout, np.float32)), dev(bias), "mish", 0.0, q_scales=dev(scales), want_f32=False,
                        residual=None if res is None else dev(res), residual_after_act=join == "after")[1]
    assert np.array_equal(q.cpu().numpy(), expected)
