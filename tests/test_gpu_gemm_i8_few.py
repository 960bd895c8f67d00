"""The int8 GEMM of few tiles of 32 x 32 and more than 32 rows: rows and columns that end inside a tile, K of less than a step,
of whole rounds of the eight wavefronts' requests and one step more, aligned rows and rows at any address, bit for bit
against the oracle; and the K-split kernel, which has larger ones, on the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def bits(a):
    return np.ascontiguousarray(a).view(np.int32)


@pytest.mark.parametrize("kernel", ["few", "ksplit"])
@pytest.mark.parametrize("m,k,n", [(33, 64, 32), (64, 65, 31), (65, 2049, 33), (40, 2048, 95), (200, 15, 100), (34, 16, 4), (1000, 63, 40), (160, 2112, 132),
                                   (35, 4100, 5), (256, 512, 1024), (500, 300, 1024),
                                   # rows at odd addresses, which this kernel takes up to a K of 7000, or two tiles a CU up to a shorter one
                                   (33, 6931, 96), (33, 7001, 96), (300, 1061, 928), (300, 1301, 928)])
def test_few_tiles(port, monkeypatch, m, k, n, kernel):
    import torch
    from tennis_amd import capi
    if kernel == "ksplit":
        monkeypatch.setenv("TSX_GEMM_I8_KSPLIT", "force")
    rng = np.random.default_rng(m + k + n)
    a, b = rng.integers(-128, 128, (m, k)).astype(np.int8), rng.integers(-128, 128, (k, n)).astype(np.int8)
    dqw, dqa = rng.uniform(1e-4, 1e-3, n).astype(np.float32), rng.uniform(0.5, 2.0, m).astype(np.float32)
    bias, qs = rng.standard_normal(n).astype(np.float32), rng.uniform(5, 20, m).astype(np.float32)
    plain, exp_acc = port.gemm_i8_dequant(a, b, dqw, dqa, bias, return_acc=True)
    g = capi.GemmI8(dev(b))
    flat = torch.from_numpy(a).reshape(-1)
    for x in (dev(a), torch.cat([flat[:1], flat]).cuda()[1:].view(m, k)):
        for act in ("relu", "leaky_relu", "mish"):
            exp = port.relu(plain) if act == "relu" else port.leaky_relu(plain, 0.1) if act == "leaky_relu" else port.mish(plain)
            kw = dict(dq=dev(dqw), row_scale=dev(dqa), bias=dev(bias), act=act, slope=0.1)
            out, q, acc = g(x, q_scales=dev(qs), want_acc=True, **kw)
            assert np.array_equal(acc.cpu().numpy(), exp_acc)
            assert np.array_equal(bits(out.cpu().numpy()), bits(exp)) and np.array_equal(q.cpu().numpy(), port.quantize(exp, qs)), act
            assert np.array_equal(bits(g(x, **kw)[0].cpu().numpy()), bits(exp)), act
            assert np.array_equal(g(x, q_scales=dev(qs), want_f32=False, **kw)[1].cpu().numpy(), port.quantize(exp, qs)), act
