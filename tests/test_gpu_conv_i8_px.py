"""The pixel-stream kernel of 1x1 int8 layers against the kernels it takes layers from (TSX_CONV_I8_PX=0), bit for bit over whole
output buffers: every number of K-steps and of fragments side by side, strides, buffers with a halo, last groups that are not
full, several turns per wavefront, one image (rounding half to even) and several, every epilogue that it writes; and against the
oracle."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, strides, halo of the buffer that is read
    (2, 64, 9, 11, 32, (1, 1), 0),            # four fragments side by side, one of them not full, one without a pixel
    (1, 20, 16, 16, 96, (1, 1), 0),           # one image; three fragments of channels
    (3, 64, 10, 7, 64, (1, 1), 1),
    (4, 64, 131, 127, 256, (1, 1), 0),        # three turns, the last ones not full
    (2, 128, 15, 17, 32, (2, 1), 0),
    (2, 100, 12, 20, 192, (1, 1), 2),
    (5, 128, 33, 31, 128, (2, 2), 0),
    (2, 256, 13, 13, 64, (1, 1), 0),
    (3, 256, 28, 30, 128, (2, 2), 1),
    (1, 250, 4, 8, 512, (1, 1), 0),           # one group in all
    (2, 512, 19, 19, 128, (1, 1), 1),
    (3, 1000, 14, 14, 256, (2, 2), 0),
    (40, 1024, 14, 14, 256, (1, 1), 0),       # two turns
]


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: "-".join(map(str, c[:5])) + "-s%d%d-halo%d" % (c[5] + c[6:]))
def test_conv_i8_px(port, monkeypatch, case):
    import torch
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    n, c, h, w, cout, strides, halo = case
    rng = np.random.default_rng(7)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, 1, 1)).astype(np.int8)
    dq = (rng.uniform(1e-5, 3e-5, cout) * 30 / np.sqrt(c)).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    ho, wo = (h - 1) // strides[0] + 1, (w - 1) // strides[1] + 1
    res = rng.standard_normal((n, cout, ho, wo)).astype(np.float32)

    def run(px, **kw):
        monkeypatch.setenv("TSX_CONV_I8_PX", px)
        conv = capi.Conv2dI8(dev(wt), (0,) * 4, strides)
        info = capi.conv2d_i8_plan_info(conv._plan(x.shape)[0])
        assert (info.get("pixel_stream") == "1") == (px == "1"), info
        # the input inside a buffer that is `halo` pixels larger all around, filled with other values there
        wide = capi.Conv2dI8(dev(wt), (halo,) * 4)
        whole = capi.StagedInput(wide, x.shape)
        wide.stage(dev(x), whole)
        st = capi.StagedView(whole, 0, 0) if halo else capi.StagedInput(conv, x.shape)
        if not halo:
            conv.stage(dev(x), st)
        return conv, st, kw

    second = capi.Conv2dI8(dev(np.zeros((32, cout, 3, 3), np.int8)), (1, 1, 1, 1))
    for act in ("none", "relu", "leaky_relu", "mish", "mish_fast"):
        for residual, after in ((None, False), (res, False), (res, True)):
            for f32, staged, up in ((True, False, 1), (True, True, 1), (False, True, 1), (False, True, 2)):
                if up == 2 and (act != "relu" or residual is not None):
                    continue
                got = []
                for px in ("0", "1"):
                    conv, st, _ = run(px)
                    out = capi.StagedInput(second, (n, cout, up * ho, up * wo)) if staged else None
                    kw = dict(bias=dev(bias), act=act, slope=0.1, want_f32=f32, residual=dev(residual), residual_after_act=after)
                    if staged:
                        kw.update(q_scales=dev(qs), staged_out=capi.StagedSlice(out, 0, cout, upsample=2) if up == 2 else out)
                    y = conv.run_staged(st, dev(dq), **kw)[0]
                    got.append((None if y is None else y.view(torch.int32), out.buf if staged else None))
                for a, b in zip(*got):
                    assert a is None or torch.equal(a, b), (act, residual is not None, after, f32, staged, up)
    # the oracle: fp32 values and requantized ones of a join
    plain = port.conv2d_quantized(x, wt, dq, (0,) * 4, strides, (1, 1))
    exp = port.relu((port.add_bias(plain, bias) + res).astype(np.float32))
    conv, st, _ = run("1")
    out = capi.StagedInput(second, (n, cout, ho, wo))
    y = conv.run_staged(st, dev(dq), dev(bias), "relu", residual=dev(res), q_scales=dev(qs), staged_out=out)[0]
    assert np.array_equal(bits(y.cpu().numpy()), bits(exp))
    assert np.array_equal(capi.staged_interior(out, range(n)).cpu().numpy(), port.quantize(exp, qs))
