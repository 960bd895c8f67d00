"""The fp32 convolution on the bf16 matrix cores by itself (TSX_CONV_F32_SPLIT puts a layer on one tile and patch form):
every tile with flat positions and with column segments, on layers whose channels, positions and output channels end inside
a chunk or a tile; small-integer data, so that any summation order gives equal bits; NaN and infinities; and errors against
64 bits, which must not exceed those of the fp32 MFMA kernel it stands in for."""
import ctypes

import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, k, pads, strides, row dilation
    (2, 20, 13, 9, 70, 3, (1, 1, 1, 1), (1, 1), 1),        # a last chunk with few channels
    (3, 7, 6, 5, 33, 3, (1, 2, 0, 1), (1, 1), 1),          # less than one chunk; small images: a tile crosses several
    (1, 36, 12, 70, 130, 3, (1, 1, 1, 1), (1, 1), 1),      # wide enough for segments, output channels beside a tile
    (2, 72, 9, 11, 40, 3, (2, 1, 3, 2), (2, 2), 2),
    (2, 40, 9, 8, 40, 5, (2, 2, 2, 2), (1, 1), 1),
    (1, 17, 7, 40, 20, 5, (0, 2, 2, 1), (1, 2), 1),
    (2, 68, 10, 14, 70, 1, (0, 0, 0, 0), (1, 1), 1),
    (3, 5, 12, 13, 31, 1, (1, 0, 0, 1), (2, 2), 1),
    (1, 131, 4, 4, 300, 1, (0, 0, 0, 0), (1, 1), 1),
    # channels in whole eights, which a padding of 0 takes without looking at them one by one, but not in whole chunks
    (3, 8, 7, 6, 33, 3, (1, 1, 1, 1), (1, 1), 1),
    (1, 24, 11, 70, 40, 3, (1, 2, 1, 1), (1, 1), 1),
    (2, 8, 9, 40, 33, 5, (2, 2, 2, 2), (1, 1), 1),
    (2, 24, 9, 13, 130, 1, (0, 0, 0, 0), (1, 1), 1),
    (3, 40, 8, 7, 33, 1, (1, 0, 1, 2), (2, 1), 1),
]
TILES = range(20)                # ten tiles, each with column segments and with flat positions


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def uses_split(capi, x, w, pads, st, dl):
    geom = capi.make_geom(x.shape, w.shape, pads, st, dl)
    return capi.lib().tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(16)) > 0


@pytest.mark.parametrize("padding_value, finite", [(np.nan, False), (np.inf, False), (3.0, True), (0.0, True), (0.0, False)])
def test_conv_f32_split_tiles(port, monkeypatch, padding_value, finite):
    """Finite: everything is a small integer; otherwise NaN and infinities lie in the padding where that can hold them, in the
    last channels, all over the last image and in one weight, and have to stay where the windows that hold them are."""
    from tennis_amd import capi
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")
    rng = np.random.default_rng(77)
    runs = [0] * len(TILES)
    for case in LAYERS:
        n, c, h, w, cout, k, pads, st, dil = case
        dl = (dil, 1)
        x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
        wt = rng.integers(-4, 5, (cout, c, k, k)).astype(np.float32)
        bias = rng.integers(-9, 10, cout).astype(np.float32)
        if not finite:
            x[0, c - 1, h // 2, w // 3] = np.inf
            x[0, 0, 0, w - 1] = -np.inf
            x[0, c // 2, h - 1, 0] = np.nan
            x[0, 1, 1, 1] = np.float32(3.4e38)      # rounds to an infinite bf16
            wt[0, 1] = 0
            if n > 1:
                x[n - 1] = np.nan
            wt[cout - 1, c - 1, 0, 0] = np.inf
        exp = port.add_bias(port.conv2d_f32(x, wt, pads, st, dl, padding_value=padding_value), bias)
        nan = np.isnan(exp)
        x_dev, w_dev, b_dev = dev(x), dev(wt), dev(bias)
        for tile in TILES:
            monkeypatch.setenv("TSX_CONV_F32_SPLIT", str(tile + 1))
            if not uses_split(capi, x, wt, pads, st, dl):
                continue
            got = capi.conv2d_f32(x_dev, w_dev, pads, st, dl, padding_value=padding_value, bias=b_dev).cpu().numpy()
            assert got.shape == exp.shape and np.array_equal(np.isnan(got), nan), (case, tile)
            # the one huge value leaves fp32 integers behind where it is multiplied: there only the magnitude is exact
            huge = np.abs(exp) > 1e30
            ok = ~nan & ~(huge & np.isfinite(exp))
            assert np.array_equal(bits(got[ok]), bits(exp[ok])), (case, tile)
            runs[tile] += 1
    # a pointwise patch is the tile's positions: flat only
    assert all(r > 0 for t, r in enumerate(runs) if t not in (16, 18)), runs


@pytest.mark.parametrize("act", ["relu", "leaky_relu"])
@pytest.mark.parametrize("case", [(3, 24, 7, 5, 33, 3), (1, 17, 5, 41, 67, 3), (1, 40, 7, 9, 33, 5), (1, 72, 5, 7, 65, 1)])
def test_conv_f32_split_activations(port, monkeypatch, case, act):
    """Bias and activation of every tile, on outputs whose number is no multiple of 4: the last ones lie behind the activation's
    SIMD body, which takes a NaN for another value than they do.  With and without a NaN in the last window of every channel."""
    from tennis_amd import capi
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")
    n, c, h, w, cout, k = case
    rng = np.random.default_rng(78)
    x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
    wt = rng.integers(-4, 5, (cout, c, k, k)).astype(np.float32)
    bias = rng.integers(-9, 10, cout).astype(np.float32)
    pads = (k // 2,) * 4
    for last in (x[n - 1, 0, h - 1, w - 1], np.nan):
        x[n - 1, 0, h - 1, w - 1] = last
        plain = port.add_bias(port.conv2d_f32(x, wt, pads, (1, 1), (1, 1)), bias)
        assert plain.size % 4 and np.isnan(plain[n - 1, :, h - 1, w - 1]).all() == np.isnan(last)
        exp = port.relu(plain) if act == "relu" else port.leaky_relu(plain, 0.1)
        nan, runs = np.isnan(exp), 0
        for mode in split_modes(monkeypatch, capi, x, wt, pads):
            got = capi.conv2d_f32(dev(x), dev(wt), pads, bias=dev(bias), act=act, slope=0.1).cpu().numpy()
            assert np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got[~nan]), bits(exp[~nan])), (mode, last)
            runs += 1
        assert runs > 2


@pytest.mark.parametrize("case", [(2, 48, 20, 20, 64, 3), (1, 256, 28, 28, 128, 3), (2, 64, 24, 24, 32, 5), (4, 512, 14, 14, 128, 1)])
@pytest.mark.parametrize("positive", [False, True])
def test_conv_f32_split_is_no_less_exact(monkeypatch, case, positive):
    import torch
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_F32_SMALL", "0")
    monkeypatch.setenv("TSX_GEMM_F32_REGFED", "0")
    n, c, h, w, cout, k = case
    g = torch.Generator().manual_seed(5)
    x, wt = torch.randn(n, c, h, w, generator=g), torch.randn(cout, c, k, k, generator=g)
    if positive:
        x, wt = x.abs(), wt.abs()
    exact = torch.nn.functional.conv2d(x.double(), wt.double(), padding=k // 2)
    pads = (k // 2,) * 4
    err = {}
    for mode in ["0"] + [str(t + 1) for t in TILES]:
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", mode)
        if mode != "0" and not uses_split(capi, x, wt, pads, (1, 1), (1, 1)):
            continue
        got = capi.conv2d_f32(x.cuda(), wt.cuda(), pads).cpu().double()
        err[mode] = float((got - exact).norm() / exact.norm())
    assert len(err) > 2 and all(e <= err["0"] for e in err.values()), err


def test_conv_f32_split_choice(monkeypatch):
    """Large layers take it, small ones and other kernels do not, and it can be switched off."""
    from tennis_amd import capi
    shape = lambda *s: np.empty(s, np.float32)
    big = (shape(8, 256, 28, 28), shape(256, 256, 3, 3), (1, 1, 1, 1), (1, 1))
    assert uses_split(capi, *big, (1, 1))
    assert not uses_split(capi, *big, (1, 2))
    assert not uses_split(capi, shape(1, 64, 56, 56), shape(64, 64, 3, 3), (1, 1, 1, 1), (1, 1), (1, 1))
    monkeypatch.setenv("TSX_CONV_F32_SPLIT", "0")
    assert not uses_split(capi, *big, (1, 1))


def split_modes(monkeypatch, capi, x, wt, pads, strides=(1, 1)):
    """The fp32 MFMA kernel ("0"), then every tile of the split kernel that takes the layer, set one after the other."""
    for mode in ["0"] + [str(t + 1) for t in TILES]:
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", mode)
        if mode == "0" or uses_split(capi, x, wt, pads, strides, (1, 1)):
            yield mode


def one_weight_per_output(rng, cout, c, k, values):
    w = np.zeros((cout, c * k * k), np.float32)
    w[np.arange(cout), rng.integers(0, c * k * k, cout)] = values
    return w.reshape(cout, c, k, k)


@pytest.fixture
def large_kernels(monkeypatch):
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")


SPARSE = [(2, 40, 20, 21, 70, 3), (1, 33, 17, 30, 48, 5), (2, 72, 12, 13, 130, 1)]


@pytest.mark.parametrize("case", SPARSE)
def test_conv_f32_split_one_product_per_output(monkeypatch, large_kernels, case):
    """Kernels with one weight that is not 0: an output is one product, which the fp32 MFMA rounds once.  The split kernel's
    sum of parts is off by 2^-29 of the product at most before that rounding (what is left out is 2^-32, the sum of the small
    parts reaches 2^-6 of the product and is rounded twice at that size)."""
    import torch
    from tennis_amd import capi
    n, c, h, w, cout, k = case
    rng = np.random.default_rng(9)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = one_weight_per_output(rng, cout, c, k, rng.standard_normal(cout))
    wt[0][wt[0] != 0] = np.uint32(0x3f80ff80).view(np.float32)      # the largest middle and low parts there are
    x[0, :, :3] = np.uint32(0x3f80ff80).view(np.float32)
    pads = (k // 2,) * 4
    exact = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(), padding=k // 2).numpy()
    err, seen = {}, exact != 0
    for mode in split_modes(monkeypatch, capi, x, wt, pads):
        got = capi.conv2d_f32(dev(x), dev(wt), pads).cpu().numpy().astype(np.float64)
        assert np.array_equal(got[~seen], exact[~seen])
        rel = np.abs(got[seen] - exact[seen]) / np.abs(exact[seen])
        assert rel.max() <= 2.0 ** -24 + 2.0 ** -29, (mode, rel.max())
        err[mode] = np.sqrt(np.mean(rel ** 2))
    assert len(err) > 2 and all(e <= err["0"] + 2.0 ** -29 for e in err.values()), err


@pytest.mark.parametrize("case", SPARSE)
@pytest.mark.parametrize("side", ["input", "weights"])
@pytest.mark.parametrize("exponents", [(0, 40), (140, 190), (200, 255)])
def test_conv_f32_split_numbers_of_any_size(monkeypatch, large_kernels, case, side, exponents):
    """Numbers from the smallest denormal on, and up to the largest there are, each times one power of two: every product is a
    float, and has to arrive as it is."""
    import torch
    from tennis_amd import capi
    n, c, h, w, cout, k = case
    rng = np.random.default_rng(10)

    def numbers(*shape):
        sign, exponent, mantissa = rng.integers(0, 2, shape), rng.integers(*exponents, shape), rng.integers(0, 1 << 23, shape)
        return (sign << 31 | exponent << 23 | mantissa).astype(np.uint32).view(np.float32)

    powers = lambda shape: (2.0 ** (rng.integers(0, 60, shape) * (1 if exponents[0] < 200 else -1))).astype(np.float32)
    if side == "input":
        x, wt = numbers(n, c, h, w), one_weight_per_output(rng, cout, c, k, powers(cout))
    else:
        wt, x = numbers(cout, c, k, k), np.zeros((n, c, h, w), np.float32)
        x[:, c - 2, ::k, ::k] = powers(x[:, 0, ::k, ::k].shape)      # a window holds one of them
    pads = (k // 2,) * 4
    exact = torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(wt).double(), padding=k // 2).numpy().astype(np.float32)
    runs = 0
    for mode in split_modes(monkeypatch, capi, x, wt, pads):
        got = capi.conv2d_f32(dev(x), dev(wt), pads).cpu().numpy()
        assert np.array_equal(got, exact), (mode, np.abs(got - exact).max())
        runs += 1
    assert runs > 2


@pytest.mark.parametrize("scale", [2.0 ** -61, 2.0 ** -66])
def test_conv_f32_split_tiny_products(monkeypatch, large_kernels, scale):
    """Operands of an ordinary size whose products, or the parts of them, are denormal."""
    import torch
    from tennis_amd import capi
    g = torch.Generator().manual_seed(6)
    x, wt = torch.randn(2, 48, 20, 20, generator=g) * scale, torch.randn(64, 48, 3, 3, generator=g) * scale
    exact = torch.nn.functional.conv2d(x.double(), wt.double(), padding=1)
    err = {}
    for mode in split_modes(monkeypatch, capi, x, wt, (1, 1, 1, 1)):
        err[mode] = float((capi.conv2d_f32(x.cuda(), wt.cuda(), (1, 1, 1, 1)).cpu().double() - exact).norm() / exact.norm())
    assert len(err) > 2 and all(e <= err["0"] for e in err.values()), err


@pytest.mark.parametrize("infinite", ["input", "weights"])
def test_conv_f32_split_infinity_against_tiny(monkeypatch, large_kernels, infinite):
    """An infinity times a denormal is an infinity of the product's sign, times 0 it is NaN."""
    from tennis_amd import capi
    rng = np.random.default_rng(12)
    x, wt = rng.standard_normal((1, 40, 14, 15)).astype(np.float32), rng.standard_normal((70, 40, 3, 3)).astype(np.float32)
    small = np.array([1e-45, -1e-45, 3e-41, -1e-39, 0.0], np.float32)
    if infinite == "input":
        x[0, 7, 5, 6] = -np.inf
        wt[:, 7] = small[np.arange(70) % 5][:, None, None]
        one = wt[:, 7, 1, 1]
    else:
        x[0, 7] = small[rng.integers(0, 5, (14, 15))]
        wt[33, 7] = 0
        wt[33, 7, 1, 1] = -np.inf
        one = x[0, 7]
    expected = np.where(one == 0, np.nan, np.where(one > 0, -np.inf, np.inf))
    runs = 0
    for mode in split_modes(monkeypatch, capi, x, wt, (1, 1, 1, 1)):
        got = capi.conv2d_f32(dev(x), dev(wt), (1, 1, 1, 1)).cpu().numpy()
        got = got[0, :, 5, 6] if infinite == "input" else got[0, 33]
        assert np.array_equal(got, expected, equal_nan=True), mode
        runs += 1
    assert runs > 2
