"""The small-tile kernel of int8 layers of several taps on few channels against the kernels it takes layers from
(TSX_CONV_I8_PT=0), bit for bit over whole output buffers: both numbers of K-steps, of taps and of window chunks, one to four
fragments of channels side by side, taps in other shapes, strides, dilations, buffers with a halo, tiles wider than the map and
across images, several turns per workgroup, one image (rounding half to even) and several; and against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, taps, strides, dilations, halo of the buffer that is read
    (4, 64, 53, 51, 64, (3, 3), (1, 1), (1, 1), 0),
    (1, 20, 120, 96, 64, (3, 3), (1, 1), (1, 1), 0),          # one image
    (64, 64, 13, 13, 96, (3, 3), (1, 1), (1, 1), 1),          # three fragments of channels, tiles across images
    (4, 64, 31, 45, 512, (3, 3), (1, 1), (1, 1), 0),
    (6, 32, 120, 110, 32, (3, 3), (1, 1), (1, 1), 0),         # four fragments of positions
    (3, 64, 141, 150, 64, (3, 3), (2, 2), (1, 1), 0),         # five chunks of the window per thread
    (5, 64, 67, 90, 256, (3, 3), (2, 1), (1, 1), 1),
    (300, 64, 41, 3, 64, (3, 3), (1, 1), (1, 1), 0),          # a map of three columns
    (2, 64, 80, 90, 128, (3, 3), (1, 1), (2, 2), 0),
    (5, 48, 90, 80, 128, (3, 3), (1, 2), (1, 3), 0),
    (2, 64, 90, 80, 128, (1, 9), (1, 1), (1, 1), 0),
    (3, 64, 70, 81, 64, (2, 3), (1, 1), (1, 1), 0),
    (3, 64, 140, 71, 128, (3, 2), (2, 1), (1, 1), 1),
    (4, 64, 70, 71, 64, (6, 1), (1, 1), (1, 1), 0),
    (3, 128, 64, 63, 64, (3, 3), (1, 1), (1, 1), 1),
    (2, 100, 62, 62, 384, (3, 3), (1, 1), (1, 1), 0),
    (40, 64, 60, 60, 64, (3, 3), (1, 1), (1, 1), 0),          # several turns, the last ones not full
    (40, 128, 30, 33, 256, (3, 3), (1, 1), (1, 1), 0),
]


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("case", LAYERS, ids=lambda c: "-".join(map(str, c[:5])) + "-k%d%d-s%d%d-d%d%d-halo%d" % (c[5] + c[6] + c[7] + c[8:]))
def test_conv_i8_pt(port, monkeypatch, case):
    import torch
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    n, c, h, w, cout, taps, strides, dilations, halo = case
    reach = [(k - 1) * d for k, d in zip(taps, dilations)]
    pads = (reach[0] // 2, reach[0] - reach[0] // 2, reach[1] // 2, reach[1] - reach[1] // 2)
    ho, wo = (h - 1) // strides[0] + 1, (w - 1) // strides[1] + 1
    rng = np.random.default_rng(11)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c) + taps).astype(np.int8)
    dq = (rng.uniform(1e-5, 3e-5, cout) * 10 / np.sqrt(c)).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    second = capi.Conv2dI8(dev(np.zeros((32, cout, 3, 3), np.int8)), (1, 1, 1, 1))
    # the input inside a buffer that is `halo` pixels larger all around, filled with other values there
    conv = capi.Conv2dI8(dev(wt), pads, strides, dilations)
    wide = capi.Conv2dI8(dev(wt), tuple(p + halo for p in pads), strides=(1, 1), dilations=dilations)
    whole = capi.StagedInput(wide, x.shape)
    wide.stage(dev(x), whole)
    st = capi.StagedView(whole, pads[0], pads[2]) if halo else capi.StagedInput(conv, x.shape)
    if not halo:
        conv.stage(dev(x), st)

    def run(pt, act, biased=True, up=1):
        monkeypatch.setenv("TSX_CONV_I8_PT", pt)
        info = capi.conv2d_i8_plan_info(conv._plan(x.shape)[0])
        assert ("tile_stream" in info) == (pt == "1"), info
        out = capi.StagedInput(second, (n, cout, up * ho, up * wo))
        conv.run_staged(st, dev(dq), bias=dev(bias) if biased else None, act=act, slope=0.1, want_f32=False, q_scales=dev(qs),
                        staged_out=capi.StagedSlice(out, 0, cout, upsample=2) if up == 2 else out)
        return out

    for act in ("none", "relu", "leaky_relu", "mish", "mish_fast"):
        assert torch.equal(run("0", act).buf, run("1", act).buf), act
    for kw in (dict(biased=False), dict(up=2)):
        assert torch.equal(run("0", "relu", **kw).buf, run("1", "relu", **kw).buf), kw
    if n * c * h * w * cout > 2e8:      # (the oracle's time)
        return
    exp = port.relu(port.add_bias(port.conv2d_quantized(x, wt, dq, pads, strides, dilations), bias))
    assert np.array_equal(capi.staged_interior(run("1", "relu"), range(n)).cpu().numpy(), port.quantize(exp, qs))
