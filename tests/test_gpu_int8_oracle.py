"""Int8 kernels against the oracle (or, beyond what it can do in time, against each other) where the tests of each kernel by itself compare
it with another form of the same code: wide 1x1 layers without a join, whole fragments that the window-stationary kernel hands
over staged, K in halves with the exact Mish, special values in every requantizing epilogue, tensors beyond 2 GiB."""
import numpy as np
import pytest

from _util import bits
from test_gpu_mish_int8 import arguments
from test_gpu_requantized_values import SPECIAL

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def planned(conv, shape, **words):
    """The plan says these things; None: it does not mention it."""
    from tennis_amd import capi
    info = capi.conv2d_i8_plan_info(conv._plan(shape)[0])
    assert all(info.get(k) == v for k, v in words.items()), info


def layer(n, c, h, w, cout, k, seed, strides=(1, 1)):
    from tennis_amd import capi
    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, k, k)).astype(np.int8)
    dq = (rng.uniform(1e-5, 3e-5, cout) * 30 / np.sqrt(c) / k).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    scales = rng.uniform(20, 30, n).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt), (k // 2,) * 4, strides)
    staged = capi.StagedInput(conv, x.shape)
    conv.stage(dev(x), staged)
    return conv, x, wt, dq, bias, scales, staged


def hand_over(cout, shape):
    """A staged input of a 3x3 consumer, for the layer's outputs."""
    from tennis_amd import capi
    return capi.StagedInput(capi.Conv2dI8(dev(np.zeros((32, cout, 3, 3), np.int8)), (1, 1, 1, 1)), shape)


@pytest.mark.parametrize("c, cout, h, w, n", [(64, 96, 9, 11, 3), (128, 256, 15, 17, 2), (250, 128, 13, 13, 3), (512, 128, 19, 19, 2), (500, 256, 7, 9, 1), (1024, 256, 14, 14, 2), (1000, 384, 9, 8, 3)])
def test_pixel_streams_without_a_join(port, monkeypatch, c, cout, h, w, n):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    conv, x, wt, dq, bias, scales, staged = layer(n, c, h, w, cout, 1, c)
    planned(conv, x.shape, pixel_stream="1")
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq), bias)
    for act, exp in (("none", plain), ("relu", port.relu(plain)), ("leaky_relu", port.leaky_relu(plain, 0.1)), ("mish", port.mish(plain))):
        out = hand_over(cout, plain.shape)
        for f32 in (True, False):
            y = conv.run_staged(staged, dev(dq), dev(bias), act, 0.1, want_f32=f32, q_scales=dev(scales), staged_out=out)[0]
            assert not f32 or np.array_equal(bits(y.cpu().numpy()), bits(exp)), act
            assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), port.quantize(exp, scales)), (act, f32)
            out.buf.zero_()


@pytest.mark.parametrize("stream", ["0", ""])
@pytest.mark.parametrize("n", [1, 3])
@pytest.mark.parametrize("act", ["relu", "leaky_relu", "mish"])
@pytest.mark.parametrize("cout", [32, 96, 128])
def test_whole_fragments_that_are_handed_over_staged(port, monkeypatch, cout, act, n, stream):
    """By the window-stationary kernel (TSX_CONV_I8_PX=0) and by the pixel stream: a residual before and behind the activation, upsampled."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    if stream:
        monkeypatch.setenv("TSX_CONV_I8_PX", stream)
    conv, x, wt, dq, bias, scales, staged = layer(n, 70, 11, 9, cout, 1, cout)
    planned(conv, x.shape, kernel="window_stationary", pixel_stream=None if stream else "1")
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq), bias)
    res = np.random.default_rng(1).standard_normal(plain.shape).astype(np.float32)
    activation = {"relu": port.relu, "leaky_relu": lambda t: port.leaky_relu(t, 0.1), "mish": port.mish}[act]
    for after, exp in ((False, activation(port.add(plain, res))), (True, port.add(activation(plain), res))):
        for up in (1, 2):
            out = hand_over(cout, (n, cout, up * 11, up * 9))
            to = out if up == 1 else capi.StagedSlice(out, 0, cout, upsample=2)
            conv.run_staged(staged, dev(dq), dev(bias), act, 0.1, want_f32=False, q_scales=dev(scales), residual=dev(res), residual_after_act=after, staged_out=to)
            assert np.array_equal(capi.staged_interior(to, range(n)).cpu().numpy(), port.quantize(exp, scales)), (after, up)


@pytest.mark.parametrize("case", [(8, 512, 14, 14, 128, 3, 2), (3, 512, 14, 13, 256, 3, 2), (4, 256, 7, 7, 128, 3, 1), (6, 640, 5, 5, 128, 5, 1), (2, 384, 13, 11, 200, 3, 2), (9, 1536, 6, 7, 255, 1, 1)],
                         ids=lambda c: "-".join(map(str, c)))
def test_k_in_halves(port, monkeypatch, case):
    """... with strides, and with the exact Mish, with and without a join."""
    from tennis_amd import capi
    for kernel in ("KS", "PX", "FLAT", "RS"):
        monkeypatch.setenv("TSX_CONV_I8_" + kernel, "0")
    n, c, h, w, cout, k, s = case
    conv, x, wt, dq, bias, scales, staged = layer(n, c, h, w, cout, k, 13, (s, s))
    planned(conv, x.shape, kernel="window_stationary", k_parts="2")
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq, (k // 2,) * 4, (s, s)), bias)
    assert np.array_equal(bits(conv.run_staged(staged, dev(dq), dev(bias))[0].cpu().numpy()), bits(plain))
    res = np.random.default_rng(2).standard_normal(plain.shape).astype(np.float32)
    for joined in (None, res):
        exp = port.mish(plain if joined is None else port.add(plain, joined))
        out = hand_over(cout, plain.shape)
        for f32 in (True, False):
            y = conv.run_staged(staged, dev(dq), dev(bias), "mish", want_f32=f32, q_scales=dev(scales), residual=dev(joined), staged_out=out)[0]
            assert not f32 or np.array_equal(bits(y.cpu().numpy()), bits(exp))
            assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), port.quantize(exp, scales))
            out.buf.zero_()


def test_k_in_halves_row_major(monkeypatch):
    """The GEMM form, which reaches that kernel where the other two GEMM kernels are switched off or leave it the shape."""
    from tennis_amd import capi
    rng = np.random.default_rng(3)
    for m, n, k in ((96, 300, 2048), (130, 128, 4096), (33, 1000, 1536)):
        monkeypatch.setenv("TSX_GEMM_I8_KSPLIT", "0")
        monkeypatch.setenv("TSX_GEMM_I8_TILE", "0")
        a, b = rng.integers(-128, 128, (m, k)).astype(np.int8), rng.integers(-127, 128, (k, n)).astype(np.int8)
        acc = capi.GemmI8(dev(b))(dev(a), dq=dev(np.ones(n, np.float32)))[0].cpu().numpy()
        assert np.array_equal(acc, (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32)), (m, n, k)


@pytest.mark.parametrize("images", [1, 3])
@pytest.mark.parametrize("act", ["none", "relu", "leaky_relu"])
@pytest.mark.parametrize("kernel, k, c, side", [("tile_stream", 3, 64, 104), ("tile_stream", 3, 128, 104), ("k_split", 3, 64, 9), ("pixel_stream", 1, 1024, 40)])
def test_requantized_special_values(port, monkeypatch, kernel, k, c, side, act, images):
    """Products on ties, beyond int8 and int32, infinite and NaN: the bias alone (the input is zero)."""
    from tennis_amd import capi
    if kernel != "k_split":
        monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    n, cout = images, 256
    bias = np.concatenate([SPECIAL, SPECIAL[::-1]] * 4)
    conv = capi.Conv2dI8(dev(np.ones((cout, c, k, k), np.int8)), (k // 2,) * 4)
    shape = (n, c, side, side)
    info = capi.conv2d_i8_plan_info(conv._plan(shape)[0])
    assert info["kernel"] == kernel if kernel == "k_split" else kernel in info, info
    staged, out = capi.StagedInput(conv, shape), hand_over(cout, (n, cout, side, side))
    conv.stage(dev(np.zeros(shape, np.int8)), staged)
    scales = np.ones(n, np.float32)
    conv.run_staged(staged, dev(np.ones(cout, np.float32)), dev(bias), act, 0.1, want_f32=False, q_scales=dev(scales), staged_out=out)
    v = np.ascontiguousarray(np.broadcast_to(bias[None, :, None, None], (n, cout, side, side))).astype(np.float32)
    v = np.float32(0) * np.float32(1) + v
    exp = {"none": lambda t: t, "relu": port.relu, "leaky_relu": lambda t: port.leaky_relu(t, 0.1)}[act](v)
    assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), port.quantize(exp, scales))


@pytest.mark.parametrize("images", [1, 2])
@pytest.mark.parametrize("kernel, side", [("pixel_stream", 5), ("pixel_stream", 20), ("tile_stream", 16)])
def test_every_kind_of_mish_argument_on_the_streaming_kernels(port, monkeypatch, kernel, side, images):
    """Weights of zero: the biases are the arguments.  The small tiles of so many channels are more than the exact Mish is left from."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    scales = np.float32([37.5, -3.0])[:images]
    bias = arguments(port, scales, 2048)
    bias = bias[:len(bias) // 128 * 128]
    cout, k = len(bias), 1 if kernel == "pixel_stream" else 3
    conv = capi.Conv2dI8(dev(np.zeros((cout, 64, k, k), np.int8)), (k // 2,) * 4)
    shape = (images, 64, side, side)
    assert kernel in capi.conv2d_i8_plan_info(conv._plan(shape)[0]) and -(-images * side * side // 64 // 8) * cout // 128 > 48
    x = np.random.default_rng(5).integers(-128, 128, shape).astype(np.int8)
    staged, out = capi.StagedInput(conv, shape), hand_over(cout, (images, cout, side, side))
    conv.stage(dev(x), staged)
    conv.run_staged(staged, dev(np.ones(cout, np.float32)), dev(bias), "mish", want_f32=False, q_scales=dev(scales), staged_out=out)
    with np.errstate(all="ignore"):
        plain = np.ascontiguousarray(np.broadcast_to(bias[None, :, None, None], (images, cout, side, side)))
        expected = port.quantize(port.mish(port.add(plain, np.zeros_like(plain))), scales)
    assert np.array_equal(capi.staged_interior(out, range(images)).cpu().numpy(), expected)


@pytest.mark.parametrize("kernel, n, c, h, w, cout, channels, f32, join", [
    ("pixel_stream", 9, 64, 491, 489, 256, 0, True, True),              # 2.2 GB of fp32 values, and of a residual's
    ("pixel_stream", 9, 1024, 491, 509, 128, 128, False, False),        # of input
    ("pixel_stream", 9, 256, 391, 351, 512, 2048, False, False),        # of hand-over: a quarter of its channels
    ("tile_stream", 16, 128, 1021, 1031, 64, 64, False, False),
    ("tile_stream", 17, 64, 521, 509, 64, 512, False, False),
])
def test_tensors_beyond_2_gib(monkeypatch, kernel, n, c, h, w, cout, channels, f32, join):
    """The last image's outputs lie beyond 31-bit offsets: whole buffers against the kernel that takes the layer otherwise."""
    import torch
    from tennis_amd import capi
    g = torch.Generator(device="cuda").manual_seed(n)
    k = 1 if kernel == "pixel_stream" else 3
    conv = capi.Conv2dI8(torch.randint(-128, 128, (cout, c, k, k), device="cuda", dtype=torch.int8, generator=g), (k // 2,) * 4)
    shape = (n, c, h, w)
    assert max(n * c * h * w, n * channels * h * w, n * cout * h * w * 4 if f32 else 0) > 1 << 31
    staged = capi.StagedInput(conv, shape)
    staged.buf.random_(-128, 128, generator=g)
    dq, bias = torch.rand(cout, device="cuda", generator=g) * 1e-4 / c ** 0.5, torch.randn(cout, device="cuda", generator=g)
    scales = torch.rand(n, device="cuda", generator=g) * 10 + 20
    residual = torch.randn((n, cout, h, w), device="cuda", generator=g) if join else None
    consumer = capi.Conv2dI8(torch.zeros((16, channels, 1, 1), device="cuda", dtype=torch.int8)) if channels else None
    got = []
    for on in ("0", "1"):
        monkeypatch.setenv("TSX_CONV_I8_" + {"pixel_stream": "PX", "tile_stream": "PT"}[kernel], on)
        assert (kernel in capi.conv2d_i8_plan_info(conv._plan(shape)[0])) == (on == "1")
        whole = capi.StagedInput(consumer, (n, channels, h, w)) if channels else None
        out = None if whole is None else whole if channels == cout else capi.StagedSlice(whole, channels - cout, cout)
        y = conv.run_staged(staged, dq, bias, "relu", want_f32=f32, q_scales=scales if out is not None else None, staged_out=out, residual=residual)[0]
        got.append((y.view(torch.int32) if f32 else None, whole.buf if whole is not None else None))
    for a, b in zip(*got):
        assert a is None or torch.equal(a, b)
    torch.cuda.synchronize()
    del got, staged, residual, y, whole, out
    torch.cuda.empty_cache()
