"""The fp32 convolution on the bf16 matrix cores with its input channels in slices, each a workgroup's, and the tiles of the
largest patches (TSX_CONV_F32_SPLIT = tile / slices): small-integer data, so that any summation order gives equal bits; NaN and
infinities; bias and activation, which the slices' sums get; errors against 64 bits; and replays of a captured call."""
import ctypes

import numpy as np
import pytest

from _util import bits
from test_gpu_conv_f32_split import LAYERS, dev

pytestmark = pytest.mark.gpu

LARGE_PATCHES = [
    (2, 37, 21, 40, 70, 3, (1, 1, 1, 1), (2, 2), 1),       # 9 rows of 65 columns
    (1, 20, 40, 67, 40, 5, (2, 2, 2, 2), (2, 2), 1),       # 11 of 67
    (2, 50, 9, 9, 37, 5, (2, 1, 2, 3), (2, 2), 1),
]
NUMBERS = range(1, 33)           # sixteen tiles, each with column segments and with flat positions


def slices_of(capi, x, w, pads, st, dl):
    """Of the plan under the current switches; 0 without one."""
    geom = capi.make_geom(x.shape, w.shape, pads, st, dl)
    text = ctypes.create_string_buffer(256)
    assert capi.lib().tsx_conv2d_f32_plan_info(ctypes.byref(geom), ctypes.c_void_p(16), text, 256) == 0
    return int(dict(item.split("=", 1) for item in text.value.decode().split()).get("workspace_slices", 0))


@pytest.fixture(autouse=True)
def no_small_kernels(monkeypatch):
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")


@pytest.mark.parametrize("padding_value, finite", [(np.nan, False), (3.0, True), (0.0, True), (0.0, False)])
def test_conv_f32_slices(port, monkeypatch, padding_value, finite):
    from tennis_amd import capi
    rng = np.random.default_rng(79)
    ran = set()
    for case in LAYERS + LARGE_PATCHES:
        n, c, h, w, cout, k, pads, st, dil = case
        dl = (dil, 1)
        x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
        wt = rng.integers(-4, 5, (cout, c, k, k)).astype(np.float32)
        bias = rng.integers(-9, 10, cout).astype(np.float32)
        if not finite:
            x[0, c - 1, h // 2, w // 3] = np.inf           # in the last slice, and in the first
            x[0, 0, 0, w - 1] = -np.inf
            wt[cout - 1, c - 1, 0, 0] = np.inf
            if n > 1:
                x[n - 1, c // 2] = np.nan
        exp = port.add_bias(port.conv2d_f32(x, wt, pads, st, dl, padding_value=padding_value), bias)
        nan = np.isnan(exp)
        x_dev, w_dev, b_dev = dev(x), dev(wt), dev(bias)
        for number in NUMBERS:
            for slices in (1, 2, 5):
                monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}/{slices}")
                used = slices_of(capi, x, wt, pads, st, dl)
                if used == 0 or (used > 1, number, case) in ran and used < slices:
                    continue
                got = capi.conv2d_f32(x_dev, w_dev, pads, st, dl, padding_value=padding_value, bias=b_dev).cpu().numpy()
                assert np.array_equal(np.isnan(got), nan), (case, number, used)
                assert np.array_equal(bits(got[~nan]), bits(exp[~nan])), (case, number, used)
                ran.add((used > 1, number, case))
    # a pointwise patch is the tile's positions: flat only
    for number in set(NUMBERS) - {17, 19}:
        assert any(r[:2] == (True, number) for r in ran) and any(r[:2] == (False, number) for r in ran), number


@pytest.mark.parametrize("act", [None, "relu", "leaky_relu"])
@pytest.mark.parametrize("case", [(3, 40, 7, 5, 33, 3), (1, 50, 6, 6, 67, 3), (2, 40, 8, 9, 5, 5), (1, 200, 5, 7, 65, 1), (2, 200, 4, 4, 64, 1)])
def test_conv_f32_slices_bias_and_activation(port, monkeypatch, case, act):
    """Maps of a multiple of 4 positions and others, numbers of outputs that leave some behind the activation's SIMD body."""
    from tennis_amd import capi
    n, c, h, w, cout, k = case
    rng = np.random.default_rng(80)
    x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
    wt = rng.integers(-4, 5, (cout, c, k, k)).astype(np.float32)
    bias = rng.integers(-9, 10, cout).astype(np.float32)
    x[n - 1, 0, h - 1, w - 1] = np.nan
    pads = (k // 2,) * 4
    plain = port.add_bias(port.conv2d_f32(x, wt, pads, (1, 1), (1, 1)), bias)
    exp = port.relu(plain) if act == "relu" else port.leaky_relu(plain, 0.1) if act else plain
    nan, sliced = np.isnan(exp), 0
    for number in NUMBERS:
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}/3")
        if slices_of(capi, x, wt, pads, (1, 1), (1, 1)) > 1:
            got = capi.conv2d_f32(dev(x), dev(wt), pads, bias=dev(bias), act=act, slope=0.1).cpu().numpy()
            assert np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got[~nan]), bits(exp[~nan])), number
            sliced += 1
    assert sliced > 1


@pytest.mark.parametrize("case", [(2, 233, 19, 6, 98, 3), (1, 256, 14, 14, 64, 3), (2, 64, 12, 12, 32, 5), (2, 512, 7, 7, 128, 1)])
@pytest.mark.parametrize("positive", [False, True])
def test_conv_f32_slices_are_no_less_exact(monkeypatch, case, positive):
    """Than the fp32 MFMA kernel, nor than one slice but for the roundings of the slices' sums: each of them is off by at most 2^-24 of
    a partial sum, which is no larger than the result here, independently of the others.  And a captured call gives the same bits on every
    replay."""
    import torch
    from tennis_amd import capi
    n, c, h, w, cout, k = case
    g = torch.Generator().manual_seed(5)
    x, wt = torch.randn(n, c, h, w, generator=g), torch.randn(cout, c, k, k, generator=g)
    if positive:
        x, wt = x.abs(), wt.abs()
    exact = torch.nn.functional.conv2d(x.double(), wt.double(), padding=k // 2)
    pads, x_dev, w_dev = (k // 2,) * 4, x.cuda(), wt.cuda()
    run = lambda: capi.conv2d_f32(x_dev, w_dev, pads)
    error = lambda got: float((got.cpu().double() - exact).norm() / exact.norm())
    monkeypatch.setenv("TSX_CONV_F32_SPLIT", "0")
    most = error(run())
    for number in NUMBERS:
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}")
        one = error(run())
        for slices in (2, 4, 64):
            monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}/{slices}")
            used = slices_of(capi, x, wt, pads, (1, 1), (1, 1))
            if used > 1:
                assert error(run()) <= min(most, one + used ** 0.5 * 2.0 ** -24), (number, slices)
    monkeypatch.delenv("TSX_CONV_F32_SPLIT")
    eager = run()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        run()
    torch.cuda.current_stream().wait_stream(stream)
    with torch.cuda.graph(graph):
        captured = run()
    for _ in range(3):
        captured.zero_()
        graph.replay()
        assert torch.equal(captured, eager)
        torch.cuda.synchronize()


def test_conv_f32_slices_choice(monkeypatch):
    """Few tiles of many channels are sliced, in a workspace of the split weights and the slices' sums; many tiles are not."""
    from tennis_amd import capi
    shape = lambda *s: np.empty(s, np.float32)
    for x, w, stride, sliced in (((2, 233, 38, 12), (98, 233, 3, 3), 2, True), ((6, 446, 33, 33), (213, 446, 5, 5), 2, True),
                                 ((8, 128, 112, 112), (128, 128, 3, 3), 1, False)):
        pads, st = (w[2] // 2,) * 4, (stride, stride)
        slices = slices_of(capi, shape(*x), shape(*w), pads, st, (1, 1))
        assert (slices > 1) == sliced and slices > 0
        geom = capi.make_geom(x, w, pads, st, (1, 1))
        ho, wo = capi.conv_out_size(geom)
        size = capi.lib().tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(16))
        sums = slices * x[0] * w[0] * ho * wo * 4 if sliced else 0
        assert size - sums >= np.prod(w) * 6 and (size - sums) % 3072 == 0


@pytest.mark.parametrize("case", [(2, 233, 19, 6, 98, 3), (1, 100, 14, 14, 64, 5), (2, 512, 7, 7, 128, 1)])
def test_conv_f32_in_the_workspace_that_there_is(monkeypatch, case):
    """A workspace below what the layer asks for is used as far as it goes: fewer slices down to one in the split weights' bytes, and the
    kernel without a workspace below these."""
    import torch
    from tennis_amd import capi
    n, c, h, w, cout, k = case
    g = torch.Generator().manual_seed(6)
    x, wt = torch.randn(n, c, h, w, generator=g).cuda(), torch.randn(cout, c, k, k, generator=g).cuda()
    pads, lib = (k // 2,) * 4, capi.lib()
    geom = capi.make_geom(tuple(x.shape), tuple(wt.shape), pads)
    pointer = lambda t: ctypes.c_void_p(t.data_ptr())
    asked = lambda: lib.tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), pointer(wt))

    def run(size):
        out, space = torch.full((n, cout, h, w), np.nan, device="cuda"), torch.full((size + 64,), 77, dtype=torch.uint8, device="cuda")
        capi.check(lib.tsx_conv2d_f32_nchw_ws(ctypes.byref(geom), pointer(x), pointer(wt), 0.0, None, 0, 0.0, pointer(out), pointer(space), size,
                                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        assert bool((space[size:] == 77).all())
        return out

    sums = n * cout * h * w * 4
    for number in NUMBERS:
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}")
        if not asked():
            continue
        weights, results = asked(), {}
        for slices in (1, 2, 3):
            monkeypatch.setenv("TSX_CONV_F32_SPLIT", f"{number}/{slices}")
            assert asked() == weights + (slices * sums if slices > 1 else 0)
            results[slices] = run(asked())
        plain = run(weights - 16)
        for size, slices in ((weights + 3 * sums - 16, 2), (weights + 2 * sums, 2), (weights + 2 * sums - 16, 1), (weights, 1)):
            assert torch.equal(run(size), results[slices]), (number, size)
        assert not torch.equal(results[1], results[2]) and not torch.equal(plain, results[1])
    # by itself: where the layer's own choice does not fit it is another choice of the same kernel, not the kernel without a workspace
    monkeypatch.delenv("TSX_CONV_F32_SPLIT")
    if k == 1:      # (stays on that one)
        return
    assert asked() > sums
    best = run(asked())
    less = run(asked() - 16)
    assert not torch.equal(less, plain) and float((less - best).norm() / best.norm()) < 2e-6
