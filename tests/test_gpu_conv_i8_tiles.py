"""The window-stationary int8 kernel on tiles narrower than the map: last column tiles that end outside it, tiles that span two
images, strides, and runs of one image's end and the next one's start on different workgroups, against the CPU oracle bit for bit."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("act", ["leaky_relu", "mish"])
@pytest.mark.parametrize("case", [
    # n, c, h, w, cout, k, stride
    (8, 64, 38, 37, 96, 3, 1), (9, 70, 19, 19, 130, 3, 1), (4, 33, 77, 75, 64, 3, 2), (3, 64, 43, 100, 40, 3, 1), (2, 20, 61, 130, 20, 5, 1),
    (16, 16, 11, 301, 64, 3, 1), (5, 40, 57, 113, 65, 1, 1),
], ids=lambda c: "-".join(map(str, c)))
def test_conv_i8_tiles(port, monkeypatch, case, act):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    monkeypatch.setenv("TSX_CONV_I8_FLAT", "0")
    n, c, h, w, cout, k, s = case
    rng = np.random.default_rng(63)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, k, k)).astype(np.int8)
    dq = rng.uniform(1e-5, 3e-5, cout).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt), (k // 2,) * 4, (s, s))
    info = capi.conv2d_i8_plan_info(conv._plan(x.shape)[0])
    assert info["kernel"] == "window_stationary" and info["fragments_per_wavefront"] in "1234", info
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq, (k // 2,) * 4, (s, s)), bias)
    exp = port.leaky_relu(plain, 0.1) if act == "leaky_relu" else port.mish(plain)
    exp_q = port.quantize(exp, qs)
    out, q, _ = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, slope=0.1, q_scales=dev(qs))
    assert np.array_equal(bits(out.cpu().numpy()), bits(exp)) and np.array_equal(q.cpu().numpy(), exp_q)
    # ... into the next layer's staged input, behind a residual join
    second = capi.Conv2dI8(dev(rng.integers(-127, 128, (8, cout, 3, 3)).astype(np.int8)), (1, 1, 1, 1))
    dq2 = rng.uniform(1e-4, 3e-4, 8).astype(np.float32)
    staged, to = capi.StagedInput(conv, x.shape), capi.StagedInput(second, exp.shape)
    conv.stage(dev(x), staged)
    res = rng.standard_normal(exp.shape).astype(np.float32)
    out = conv.run_staged(staged, dev(dq), dev(bias), act, 0.1, q_scales=dev(qs), residual=dev(res), residual_after_act=True, staged_out=to)[0]
    joined = port.add(exp, res)
    assert np.array_equal(bits(out.cpu().numpy()), bits(joined))
    got = second.run_staged(to, dev(dq2))[0].cpu().numpy()
    assert np.array_equal(bits(got), bits(port.conv2d_quantized(port.quantize(joined, qs), second.w.cpu().numpy(), dq2, (1, 1, 1, 1))))


@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("act", ["mish", "mish_fast", "relu"])
@pytest.mark.parametrize("cout", [9, 18, 33, 47, 63, 65, 32, 96])
def test_channels_of_partial_fragments(port, monkeypatch, cout, act, n):
    """Fragments whose 32 channels do not all exist, and those that do where a kernel has nothing else (a wavefront of the last block
    may have no channel at all there; with raw sums they take the other epilogue), with a join: raw sums, fp32, NCHW int8 (one image: half to even up to the last
    whole eight; two: a scale each) and staged int8, by itself and upsampled."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    c, h, w = 70, 11, 9
    rng = np.random.default_rng(cout)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, 1, 1)).astype(np.int8)
    dq = rng.uniform(1e-4, 3e-4, cout).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt))
    plain = port.add_bias(port.conv2d_quantized(x, wt, dq), bias)
    res = rng.standard_normal(plain.shape).astype(np.float32)
    activated = port.relu(plain) if act == "relu" else port.mish(plain)
    if act == "mish_fast":       # the short form's values, by a layer whose epilogue has no join
        short = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act)[0].cpu().numpy()
        assert np.all(np.abs(short - activated) <= 6 * 2.0 ** -24 * np.abs(plain))
        activated = short
    joined = port.add(activated, res)
    expected = port.quantize(joined, qs)
    out, q, acc = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, q_scales=dev(qs), residual=dev(res), residual_after_act=True, want_acc=True)
    assert np.array_equal(acc.cpu().numpy(), np.einsum("nchw,oc->nohw", x.astype(np.int32), wt[:, :, 0, 0].astype(np.int32)))
    assert np.array_equal(bits(out.cpu().numpy()), bits(joined)) and np.array_equal(q.cpu().numpy(), expected)
    out, q, _ = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, q_scales=dev(qs), residual=dev(res), residual_after_act=True)
    assert np.array_equal(bits(out.cpu().numpy()), bits(joined)) and np.array_equal(q.cpu().numpy(), expected)
    q = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, q_scales=dev(qs), residual=dev(res), residual_after_act=True, want_f32=False)[1]
    assert np.array_equal(q.cpu().numpy(), expected)
    staged = capi.StagedInput(conv, x.shape)
    conv.stage(dev(x), staged)
    for up in (1, 2):
        to = capi.StagedInput(capi.Conv2dI8(dev(np.zeros((8, cout, 3, 3), np.int8)), (1, 1, 1, 1)), (n, cout, up * h, up * w))
        to = to if up == 1 else capi.StagedSlice(to, 0, cout, upsample=2)
        conv.run_staged(staged, dev(dq), dev(bias), act, 0.0, q_scales=dev(qs), want_f32=False, residual=dev(res), residual_after_act=True, staged_out=to)
        assert np.array_equal(capi.staged_interior(to, range(n)).cpu().numpy(), port.quantize(joined, qs))
