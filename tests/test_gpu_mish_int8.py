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


@pytest.mark.parametrize("act", ["leaky_relu", "mish"])
@pytest.mark.parametrize("case", [
    # n, c, h, w, cout, (kh, kw), stride, pads, forced flat tile: windows that leave no room for the exact Mish's tables in 64 KiB ...
    (15, 70, 47, 47, 17, (5, 5), 2, 2, None), (2, 70, 189, 189, 17, (3, 3), 2, 1, None), (7, 130, 91, 26, 57, (5, 5), 2, 2, None),
    # ... or, all the layer's windows at once, in 160 (two of them do), or not even two
    (7, 300, 5, 10, 70, (3, 3), 1, 1, "33"), (6, 300, 11, 7, 130, (3, 3), 1, 1, "43"), (1, 70, 300, 2, 70, (42, 2), 1, 0, "32"),
], ids=lambda c: "-".join(map(str, c)))
def test_windows_of_the_whole_lds(port, monkeypatch, case, act):
    from tennis_amd import capi
    n, c, h, w, cout, kernel, stride, pad, flat = case
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    monkeypatch.setenv("TSX_CONV_I8_RS", "0")
    monkeypatch.setenv("TSX_CONV_I8_FLAT", "force" + flat if flat else "0")
    rng = np.random.default_rng(17)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c) + kernel).astype(np.int8)
    dq = rng.uniform(1e-5, 3e-5, cout).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt), (pad,) * 4, (stride, stride))
    info = capi.conv2d_i8_plan_info(conv._plan(x.shape)[0])
    assert info["kernel"] == ("flat_tile" if flat else "window_stationary"), info
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq, (pad,) * 4, (stride, stride)), bias)
    res = rng.standard_normal(plain.shape).astype(np.float32)
    value = port.mish(plain) if act == "mish" else port.leaky_relu(plain, 0.1)
    for join, expected in ((None, value), (res, port.add(value, res))):
        out, q, _ = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, slope=0.1, q_scales=dev(qs), residual=None if join is None else dev(join),
                         residual_after_act=join is not None)
        assert np.array_equal(out.cpu().numpy().view(np.int32), expected.view(np.int32))
        assert np.array_equal(q.cpu().numpy(), port.quantize(expected, qs))
