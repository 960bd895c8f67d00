"""The tile kernel of the int8 GEMM by itself (TSX_GEMM_I8_TILE=1..3 gives it every GEMM of more than 32 rows that no
K-split kernel takes), bit for bit against the oracle: rows and columns that end inside a tile, an odd number of K-steps (half
a last chunk), one K-step, columns that are no multiple of 4 or 16 (elements behind the activation's SIMD body, single-byte
stores), packed int8 output, and more tiles than one group of four rows of tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def bits(x):
    return np.ascontiguousarray(x).view(np.int32)


@pytest.mark.parametrize("m,k,n", [(33, 64, 128), (129, 100, 131), (257, 192, 400), (300, 321, 30), (1300, 128, 272), (128, 640, 513)])
@pytest.mark.parametrize("tile", ["1", "2", "3"])
def test_gemm_i8_tile_kernel(port, monkeypatch, m, k, n, tile):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_GEMM_I8_TILE", tile)
    monkeypatch.setenv("TSX_GEMM_I8_KSPLIT", "0")
    rng = np.random.default_rng(340 + m + n)
    a = rng.integers(-128, 128, (m, k)).astype(np.int8)
    b = rng.integers(-128, 128, (k, n)).astype(np.int8)
    dqw = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    dqa = rng.uniform(0.5, 2.0, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    qs = rng.uniform(5, 20, m).astype(np.float32)
    g = capi.GemmI8(_dev(b))
    for row_scale, with_bias, act in ((dqa, True, "relu"), (None, False, None), (dqa, True, "leaky_relu")):
        kw = dict(dq=_dev(dqw), row_scale=None if row_scale is None else _dev(row_scale), bias=_dev(bias) if with_bias else None, act=act, slope=0.1)
        exp, exp_acc = port.gemm_i8_dequant(a, b, dqw, row_scale, bias if with_bias else None, return_acc=True)
        exp = port.relu(exp) if act == "relu" else port.leaky_relu(exp, 0.1) if act else exp
        out, _, _ = g(_dev(a), **kw)
        assert np.array_equal(bits(out.cpu().numpy()), bits(exp)), act
        _, q, _ = g(_dev(a), q_scales=_dev(qs), want_f32=False, **kw)
        assert np.array_equal(q.cpu().numpy(), port.quantize(exp, qs)), act
        out, q, acc = g(_dev(a), q_scales=_dev(qs), want_acc=True, **kw)
        assert np.array_equal(acc.cpu().numpy(), exp_acc)
        assert np.array_equal(bits(out.cpu().numpy()), bits(exp)) and np.array_equal(q.cpu().numpy(), port.quantize(exp, qs)), act


@pytest.mark.parametrize("m,k,n", [(1, 7, 5), (1, 17, 64), (2, 8, 33), (32, 100, 33), (31, 1500, 96), (33, 1, 40), (129, 3, 33), (192, 5, 144), (130, 77, 64),
                                   (197, 1500, 77), (65, 2049, 66), (64, 2500, 72), (130, 1985, 48), (70, 2048, 64)])
@pytest.mark.parametrize("kernel", ["chosen", "window_stationary", "tile_1", "tile_2", "tile_3", "k_split"])
def test_gemm_i8_rows_of_any_length(port, monkeypatch, m, k, n, kernel):
    """Rows that are no multiple of a K-step, from a pointer that is no multiple of anything, read where they are: the
    last row's last pieces, rows shorter than a piece, a matrix shorter than one; above 32 rows on the kernel of few tiles, which the sizes
    give them, and on each of the others."""
    import torch
    from tennis_amd import capi
    if kernel != "chosen":
        monkeypatch.setenv("TSX_GEMM_I8_KSPLIT", "force" if kernel == "k_split" else "0")
        monkeypatch.setenv("TSX_GEMM_I8_TILE", kernel[-1] if kernel.startswith("tile") else "0")
    rng = np.random.default_rng(350 + m + n)
    a = rng.integers(-128, 128, (m, k)).astype(np.int8)
    b = rng.integers(-128, 128, (k, n)).astype(np.int8)
    dqw = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    dqa = rng.uniform(0.5, 2.0, m).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    qs = rng.uniform(5, 20, m).astype(np.float32)
    exp, exp_acc = port.gemm_i8_dequant(a, b, dqw, dqa, bias, return_acc=True)
    exp = port.relu(exp)
    kw = dict(dq=_dev(dqw), row_scale=_dev(dqa), bias=_dev(bias), act="relu")
    g = capi.GemmI8(_dev(b))
    flat = torch.from_numpy(a).reshape(-1)
    for x in (_dev(a), torch.cat([flat[:1], flat]).cuda()[1:].view(m, k)):
        out, _, acc = g(x, want_acc=True, **kw)
        assert np.array_equal(acc.cpu().numpy(), exp_acc)
        assert np.array_equal(bits(out.cpu().numpy()), bits(exp))
        _, q, _ = g(x, q_scales=_dev(qs), want_f32=False, **kw)
        assert np.array_equal(q.cpu().numpy(), port.quantize(exp, qs))


@pytest.mark.parametrize("m", [65, 130, 131, 259])
@pytest.mark.parametrize("n", [1, 2, 3, 5])
@pytest.mark.parametrize("tile", ["1", "2", "3", "0", "force"])
def test_gemm_i8_tile_kernel_few_columns(port, monkeypatch, tile, n, m):
    """The up to three elements behind the activation's SIMD body are the last of the tensor: with one output column they
    are several rows.  Body and tail differ in what they make of NaN and of -0, which fill the last rows here.  The other
    GEMM kernels besides: "0" the window-stationary kernel's GEMM form, "force" the K-split kernel."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_GEMM_I8_TILE", tile if tile != "force" else "0")
    monkeypatch.setenv("TSX_GEMM_I8_KSPLIT", "force" if tile == "force" else "0")
    rng = np.random.default_rng(345 + m + n)
    k = 70
    a = rng.integers(-128, 128, (m, k)).astype(np.int8)
    b = rng.integers(-128, 128, (k, n)).astype(np.int8)
    dqw = rng.uniform(1e-4, 1e-3, n).astype(np.float32)
    qs = rng.uniform(5, 20, m).astype(np.float32)
    g = capi.GemmI8(_dev(b))
    for row_value in (np.nan, -0.0):
        dqa = rng.uniform(0.5, 2.0, m).astype(np.float32)
        dqa[m - 5:] = row_value
        for act in ("relu", "leaky_relu"):
            exp = port.gemm_i8_dequant(a, b, dqw, dqa, None)
            exp = port.relu(exp) if act == "relu" else port.leaky_relu(exp, 0.1)
            kw = dict(dq=_dev(dqw), row_scale=_dev(dqa), act=act, slope=0.1)
            out = g(_dev(a), **kw)[0].cpu().numpy()
            assert np.array_equal(np.isnan(out), np.isnan(exp))
            assert np.array_equal(bits(np.nan_to_num(out)), bits(np.nan_to_num(exp))), (row_value, act)
            q = g(_dev(a), q_scales=_dev(qs), want_f32=False, **kw)[1].cpu().numpy()
            assert np.array_equal(q, port.quantize(exp, qs)), (row_value, act)
