"""What the streaming int8 kernels choose for large outputs, at the sizes where they choose it, bit for bit against the kernels they take
layers from and against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def device(shape, seed, values=None):
    """Values on the device, without a host copy of large tensors: int8 of the whole range, or standard normal floats."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-128, 128, shape, device="cuda", dtype=torch.int8, generator=g) if values is None else torch.randn(shape, device="cuda", generator=g) * values


def layer(n, c, h, w, cout, k=1, stride=1, seed=3):
    """The layer, its scales and biases, and its staged input."""
    from tennis_amd import capi
    conv = capi.Conv2dI8(device((cout, c, k, k), seed), (k // 2,) * 4, (stride, stride))
    staged = capi.StagedInput(conv, (n, c, h, w))
    conv.stage(device((n, c, h, w), seed + 1), staged)
    return conv, device((cout,), seed + 2, 1e-5).abs() * (30 / k) / c ** 0.5 + 1e-6, device((cout,), seed + 3, 1.0), staged


def streams(monkeypatch, conv, shape, name, on):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_" + {"pixel_stream": "PX", "tile_stream": "PT"}[name], "1" if on else "0")
    info = capi.conv2d_i8_plan_info(conv._plan(shape)[0])
    assert (name in info) == on and info["kernel"] != "k_split", info


@pytest.mark.parametrize("c", [64, 100, 256, 512, 1000])
@pytest.mark.parametrize("cout, h, w", [(32, 256, 132), (64, 256, 68), (128, 128, 64), (256, 56, 76), (384, 49, 64)])
def test_streaming_stores(monkeypatch, c, cout, h, w):
    """16 MiB and more of fp32 values, planes of whole half cache lines, the last group of pixels full or not."""
    if cout % (32 if c <= 128 else 64 if c <= 256 else 128):
        pytest.skip("no pixel stream for these channels")
    import torch
    n = 4
    conv, dq, bias, staged = layer(n, c, h, w, cout)
    assert n * cout * h * w * 4 >= 16 << 20 and h * w % 16 == 0
    for act in ("none", "leaky_relu", "mish"):
        got = []
        for on in (False, True):
            streams(monkeypatch, conv, (n, c, h, w), "pixel_stream", on)
            got.append(conv.run_staged(staged, dq, bias, act, 0.1)[0])
        assert torch.equal(got[0].view(torch.int32), got[1].view(torch.int32)), act


def same_outputs(monkeypatch, conv, dq, bias, staged, shape, out_shape, act, f32, requantized, residual=None):
    """Whole output buffers of the layer with and without the pixel stream."""
    import torch
    from tennis_amd import capi
    second = capi.Conv2dI8(torch.zeros((32, out_shape[1], 1, 1), dtype=torch.int8, device="cuda"))
    scales = device((shape[0],), 17, 1.0).abs() * 10 + 20
    got = []
    for on in (False, True):
        streams(monkeypatch, conv, shape, "pixel_stream", on)
        out = capi.StagedInput(second, out_shape) if requantized else None
        y = conv.run_staged(staged, dq, bias, act, 0.1, want_f32=f32, q_scales=scales if requantized else None, staged_out=out, residual=residual)[0]
        got.append((y.view(torch.int32) if f32 else None, out.buf if requantized else None))
    for a, b in zip(*got):
        assert a is None or torch.equal(a, b), act


@pytest.mark.parametrize("n, h, w, cout", [(20, 8, 8, 512), (8, 40, 58, 384), (4, 74, 74, 1024), (3, 67, 59, 128)])     # one turn; four and six, the last ones not full
def test_turns_of_1024_channels(monkeypatch, n, h, w, cout):
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    c = 1000
    conv, dq, bias, staged = layer(n, c, h, w, cout)
    for act, f32, requantized in (("relu", True, False), ("none", False, True), ("mish", True, True)):
        same_outputs(monkeypatch, conv, dq, bias, staged, (n, c, h, w), (n, cout, h, w), act, f32, requantized)


@pytest.mark.parametrize("n, c, h, w, cout", [(12, 64, 41, 43, 2048), (9, 256, 33, 35, 2176), (6, 100, 57, 57, 4096)])
def test_large_outputs_whose_planes_share_lines(monkeypatch, n, c, h, w, cout):
    """Two blocks of channels at a time, or one where their number is odd."""
    conv, dq, bias, staged = layer(n, c, h, w, cout)
    res = device((n, cout, h, w), 23, 1.0)
    for act, f32, requantized, residual in (("relu", True, False, res), ("leaky_relu", True, True, res), ("none", True, False, None), ("mish", True, True, None)):
        same_outputs(monkeypatch, conv, dq, bias, staged, (n, c, h, w), (n, cout, h, w), act, f32, requantized, residual)


TILE_STREAMS_WITH_MISH = [
    # n, c, h, w, cout, taps, strides: a layer for each instantiation of the small-tile kernel that the exact Mish is left on
    (11, 64, 53, 51, 128, (3, 3), (1, 1)), (8, 64, 53, 51, 64, (3, 3), (1, 1)), (9, 50, 120, 110, 32, (3, 3), (1, 1)), (9, 64, 141, 150, 256, (3, 3), (2, 2)),
    (3, 64, 141, 150, 64, (3, 3), (2, 2)), (9, 64, 140, 71, 128, (3, 2), (2, 1)), (3, 64, 70, 81, 64, (2, 3), (1, 1)), (12, 100, 50, 50, 128, (3, 3), (1, 1)),
    (3, 128, 64, 63, 64, (3, 3), (1, 1)),
]


@pytest.mark.parametrize("case", TILE_STREAMS_WITH_MISH, ids=lambda c: "-".join(map(str, c[:5])) + "-k%d%d-s%d%d" % (c[5] + c[6]))
def test_tile_streams_with_the_exact_mish(port, monkeypatch, case):
    """... whole output buffers against the other kernels, and two images of them against the oracle."""
    import torch
    from tennis_amd import capi
    n, c, h, w, cout, (kh, kw), strides = case
    conv = capi.Conv2dI8(device((cout, c, kh, kw), 3), (kh // 2, kh // 2, kw // 2, kw // 2), strides)
    x = device((n, c, h, w), 4)
    staged = capi.StagedInput(conv, x.shape)
    conv.stage(x, staged)
    dq, bias = device((cout,), 5, 1e-5).abs() * 10 / c ** 0.5 + 1e-6, device((cout,), 6, 1.0)
    scales = device((n,), 7, 1.0).abs() * 10 + 20
    ho, wo = (h + 2 * (kh // 2) - kh) // strides[0] + 1, (w + 2 * (kw // 2) - kw) // strides[1] + 1
    second = capi.Conv2dI8(torch.zeros((32, cout, 3, 3), dtype=torch.int8, device="cuda"), (1, 1, 1, 1))
    got = []
    for on in (False, True):
        streams(monkeypatch, conv, x.shape, "tile_stream", on)
        out = capi.StagedInput(second, (n, cout, ho, wo))
        conv.run_staged(staged, dq, bias, "mish", want_f32=False, q_scales=scales, staged_out=out)
        got.append(out)
    assert torch.equal(got[0].buf, got[1].buf)
    two = x[n - 2:].cpu().numpy()       # (one scale each: a single one is rounded half to even)
    weights = device((cout, c, kh, kw), 3).cpu().numpy()
    plain = port.add_bias(port.conv2d_quantized(two, weights, dq.cpu().numpy(), (kh // 2, kh // 2, kw // 2, kw // 2), strides), bias.cpu().numpy())
    assert np.array_equal(capi.staged_interior(got[1], [n - 2, n - 1]).cpu().numpy(), port.quantize(port.mish(plain), scales[n - 2:].cpu().numpy()))
