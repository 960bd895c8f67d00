"""What the int8 convolutions' epilogues requantize where products are no finite numbers inside the int8 range, on each kernel, against
the oracle."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


SPECIAL = np.array([0.0, -0.0, 0.5, -0.5, 1.5, 2.5, -2.5, 0.49999997, -0.49999997, 126.5, 127.49999, 127.5, -127.5, -128.5, 1e9, -1e9, 2147483520.0,
                    2147483648.0, -2147483648.0, 4e9, -4e9, 3e38, -3e38, np.inf, -np.inf, np.nan, 1e-42, -1e-42, 8388607.5, 16777217.0, 3.5, -3.5], np.float32)


@pytest.mark.parametrize("images", [1, 3])
@pytest.mark.parametrize("act", ["none", "relu", "leaky_relu"])
@pytest.mark.parametrize("kernel", ["pixel_stream", "window_stationary", "flat_tile", "igemm"])
def test_requantized_special_values(port, monkeypatch, kernel, act, images):
    """Products on ties, beyond int8 and int32, infinite and NaN: the bias alone (the input is zero)."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    if kernel != "pixel_stream":
        monkeypatch.setenv("TSX_CONV_I8_PX", "0")
    if kernel == "flat_tile":
        monkeypatch.setenv("TSX_CONV_I8_FLAT", "force")
    k, st = (1, 2) if kernel == "igemm" else (1, 1) if kernel == "pixel_stream" else (3, 1)
    n, c, h, cout = images, 64, 16, 128
    bias = np.concatenate([SPECIAL, SPECIAL[::-1]] * 2)
    conv = capi.Conv2dI8(dev(np.ones((cout, c, k, k), np.int8)), (k // 2,) * 4, (st, st))
    info = capi.conv2d_i8_plan_info(conv._plan((n, c, h, h))[0])
    assert info["kernel"] == ("window_stationary" if kernel == "pixel_stream" else kernel) and ("pixel_stream" in info) == (kernel == "pixel_stream"), info
    ho = (h - 1) // st + 1
    second = capi.Conv2dI8(dev(np.zeros((32, cout, 1, 1), np.int8)))
    out, staged = capi.StagedInput(second, (n, cout, ho, ho)), capi.StagedInput(conv, (n, c, h, h))
    conv.stage(dev(np.zeros((n, c, h, h), np.int8)), staged)
    qs = np.ones(n, np.float32)
    kw = dict(bias=dev(bias), act=act, slope=0.1, q_scales=dev(qs), staged_out=out)
    f32 = conv.run_staged(staged, dev(np.ones(cout, np.float32)), **kw)[0].cpu().numpy()
    v = np.broadcast_to(bias[None, :, None, None], f32.shape).astype(np.float32)
    v = np.float32(0) * np.float32(1) + v            # the dequantized zero
    exp = {"none": lambda t: t, "relu": port.relu, "leaky_relu": lambda t: port.leaky_relu(t, 0.1)}[act](np.ascontiguousarray(v))
    finite = ~np.isnan(exp)
    assert np.array_equal(np.isnan(f32), ~finite) and np.array_equal(bits(f32)[finite], bits(exp)[finite])
    exp_q = port.quantize(exp, qs)
    assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), exp_q)
    conv.run_staged(staged, dev(np.ones(cout, np.float32)), want_f32=False, **kw)
    assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), exp_q)
