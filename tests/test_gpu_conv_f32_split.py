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
]
TILES = range(20)                # ten tiles, each with column segments and with flat positions


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def uses_split(capi, x, w, pads, st, dl):
    geom = capi.make_geom(x.shape, w.shape, pads, st, dl)
    return capi.lib().tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(16)) > 0


@pytest.mark.parametrize("padding_value", [np.nan, np.inf, 3.0])
def test_conv_f32_split_tiles(port, monkeypatch, padding_value):
    """With 3.0 everything is a small integer; otherwise NaN and infinities lie in the padding, in the last channels, all over
    the last image and in one weight, and have to stay where the windows that hold them are."""
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
        if not np.isfinite(padding_value):
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
