"""The window kernel of the fp32 convolution by itself (TSX_CONV_F32_TILE puts a layer on one tile and patch form): every
tile with flat positions and with column segments, on layers whose channels, positions and output channels end inside a
chunk or a tile, with strides, dilations and paddings; small-integer data, so that any summation order gives equal
bits and a wrong tap, padding element or channel cannot hide in a tolerance."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, kh, kw, pads, strides, dilations
    (2, 20, 13, 9, 70, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),        # K a multiple of 4, a last chunk with few channels
    (3, 7, 6, 5, 33, 3, 3, (1, 2, 0, 1), (1, 1), (1, 1)),          # K odd; small images: a tile crosses several
    (1, 36, 40, 70, 130, 3, 3, (1, 1, 1, 1), (1, 1), (1, 1)),      # wide enough for segments, output channels beside a tile
    (2, 12, 21, 38, 40, 3, 3, (2, 1, 3, 2), (2, 2), (1, 2)),
    (2, 3, 30, 31, 20, 7, 7, (3, 3, 3, 3), (2, 2), (1, 1)),        # a stem
    (1, 9, 17, 20, 12, 1, 5, (0, 0, 2, 2), (1, 1), (1, 1)),
    (2, 68, 10, 14, 70, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),       # pointwise, positions read 4 at a time
    (2, 66, 9, 11, 65, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),        # ... one at a time
    (3, 5, 12, 13, 31, 1, 1, (1, 0, 0, 1), (2, 2), (1, 1)),        # ... strided and padded
    (1, 131, 4, 4, 8, 1, 1, (0, 0, 0, 0), (1, 1), (1, 1)),
]


@pytest.mark.parametrize("tile", range(10))
def test_conv_f32_window_tiles(port, monkeypatch, tile):
    import torch
    from tennis_amd import capi
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")
    monkeypatch.setenv("TSX_CONV_F32_TILE", str(tile))
    rng = np.random.default_rng(77)
    ran = 0
    for case in LAYERS:
        n, c, h, w, cout, kh, kw, pads, st, dl = case
        if kh * kw == 1 and tile % 2 == 0:
            continue                                   # a pointwise patch is the tile's positions: one form
        x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
        wt = rng.integers(-4, 5, (cout, c, kh, kw)).astype(np.float32)
        bias = rng.integers(-9, 10, cout).astype(np.float32)
        try:
            got = capi.conv2d_f32(dev(x), dev(wt), pads, st, dl, padding_value=3.0, bias=dev(bias), act="relu").cpu().numpy()
        except capi.TsxError as e:
            assert "does not suit" in str(e), case     # a patch beyond this tile's LDS
            continue
        exp = port.relu(port.add_bias(port.conv2d_f32(x, wt, pads, st, dl, padding_value=3.0), bias))
        assert got.shape == exp.shape and np.array_equal(bits(got), bits(exp)), case
        ran += 1
    assert ran >= 3


@pytest.mark.parametrize("padding_value", [np.nan, np.inf, 3.0])
@pytest.mark.parametrize("tile", range(10))
def test_conv_f32_window_tiles_not_finite(port, monkeypatch, tile, padding_value):
    """NaN and infinities stay where the windows that hold them are: in the padding, in the last channels (a chunk that is not
    full reads other data behind them), and all over the last image, whose elements lie next to those of the one before.
    Sums of them do not depend on the order; all else is small integers."""
    import torch
    from tennis_amd import capi
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    for env in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.setenv(env, "0")
    monkeypatch.setenv("TSX_CONV_F32_TILE", str(tile))
    rng = np.random.default_rng(78)
    ran = 0
    for case in LAYERS:
        n, c, h, w, cout, kh, kw, pads, st, dl = case
        if kh * kw == 1 and tile % 2 == 0:
            continue
        x = rng.integers(-8, 9, (n, c, h, w)).astype(np.float32)
        x[0, c - 1, h // 2, w // 3] = np.inf
        x[0, 0, 0, w - 1] = -np.inf
        x[0, c // 2, h - 1, 0] = np.nan
        if n > 1:
            x[n - 1] = np.nan
        wt = rng.integers(-4, 5, (cout, c, kh, kw)).astype(np.float32)
        wt[cout - 1, c - 1, 0, 0] = np.inf
        try:
            got = capi.conv2d_f32(dev(x), dev(wt), pads, st, dl, padding_value=padding_value).cpu().numpy()
        except capi.TsxError as e:
            assert "does not suit" in str(e), case
            continue
        exp = port.conv2d_f32(x, wt, pads, st, dl, padding_value=padding_value)
        nan = np.isnan(exp)
        assert np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got[~nan]), bits(exp[~nan])), case
        assert not nan.all(), case
        ran += 1
    assert ran >= 3
