"""The K-split int8 convolution kernel on each of its tiles, and the kernels it stands in for (TSX_CONV_I8_KS = tile, or 0),
against the CPU oracle bit for bit: channels, positions and output channels that end inside a
block or a tile, more wavefronts than K-steps, several rounds of the operand ring, tiles that span images, a buffer wider
than the layer needs, and every epilogue term."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

LAYERS = [
    # n, c, h, w, cout, k, pads, strides, dilations
    (1, 100, 13, 13, 150, 3, (1, 1, 1, 1), (2, 2), (1, 1)),
    (3, 64, 7, 7, 32, 1, (0, 0, 0, 0), (1, 1), (1, 1)),           # one K-step for four wavefronts
    (2, 130, 9, 11, 37, 1, (0, 0, 0, 0), (2, 2), (1, 1)),         # the generic kernel's weights
    (5, 70, 3, 2, 65, 1, (1, 0, 0, 1), (2, 3), (1, 1)),           # ... several images per tile, with a halo
    (2, 64, 40, 33, 129, 1, (0, 0, 0, 0), (2, 1), (1, 1)),
    (7, 200, 1, 1, 30, 1, (0, 0, 0, 0), (1, 1), (1, 1)),          # a position per image
    (2, 512, 7, 7, 48, 3, (1, 1, 1, 1), (1, 1), (1, 1)),          # 72 K-steps: more than a round of every ring
    (1, 300, 8, 9, 17, 5, (2, 1, 2, 3), (1, 2), (2, 1)),
    (1, 3, 6, 5, 1, 2, (0, 1, 1, 0), (1, 1), (1, 1)),             # packed by im2col; one output channel
]


def dev(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("tile", ["0", "1", "2", "3"])
@pytest.mark.parametrize("case", LAYERS, ids=lambda c: "-".join(map(str, c[:6])))
def test_conv_i8_ks(port, monkeypatch, tile, case):
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", tile)
    n, c, h, w, cout, k, pads, st, dl = case
    rng = np.random.default_rng(61)
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    wt = rng.integers(-127, 128, (cout, c, k, k)).astype(np.int8)
    dq = rng.uniform(1e-5, 3e-5, cout).astype(np.float32)
    bias = rng.standard_normal(cout).astype(np.float32)
    qs = rng.uniform(20, 30, n).astype(np.float32)
    conv = capi.Conv2dI8(dev(wt), pads, st, dl)
    info = capi.conv2d_i8_plan_info(conv._plan(x.shape)[0])
    assert (info["kernel"] == "k_split") == (tile != "0") and info.get("tile", "0") == tile, info
    plain, exp_acc = port.conv2d_quantized(x, wt, dq, pads, st, dl, return_acc=True)
    for act in ("none", "relu", "leaky_relu", "mish"):
        activated = {"none": lambda t: t, "relu": port.relu, "leaky_relu": lambda t: port.leaky_relu(t, 0.1), "mish": port.mish}[act]
        exp = activated(port.add_bias(plain, bias))
        exp_q = port.quantize(exp, qs)
        out, q, acc = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, slope=0.1, q_scales=dev(qs), want_acc=True)
        assert np.array_equal(acc.cpu().numpy(), exp_acc)
        assert np.array_equal(bits(out.cpu().numpy()), bits(exp)) and np.array_equal(q.cpu().numpy(), exp_q)
        out, q, _ = conv(dev(x), dq=dev(dq), bias=dev(bias), act=act, slope=0.1)
        assert q is None and np.array_equal(bits(out.cpu().numpy()), bits(exp))
    if c <= 8:
        return                             # a layer that stages by im2col has no buffer that a producer could write
    # residual join in front of and behind the activation, into the next layer's staged input (checked by that layer)
    res = rng.standard_normal(plain.shape).astype(np.float32)
    second = capi.Conv2dI8(dev(rng.integers(-127, 128, (40, cout, 3, 3)).astype(np.int8)), (1, 1, 1, 1))
    dq2 = rng.uniform(1e-4, 3e-4, 40).astype(np.float32)
    staged = capi.StagedInput(conv, x.shape)
    conv.stage(dev(x), staged)
    for after in (False, True):
        joined = port.add(port.relu(port.add_bias(plain, bias)), res) if after else port.relu(port.add(port.add_bias(plain, bias), res))
        to = capi.StagedInput(second, plain.shape)
        out = conv.run_staged(staged, dev(dq), dev(bias), "relu", q_scales=dev(qs), residual=dev(res), residual_after_act=after, staged_out=to)[0]
        assert np.array_equal(bits(out.cpu().numpy()), bits(joined))
        got = second.run_staged(to, dev(dq2))[0].cpu().numpy()
        exp2 = port.conv2d_quantized(port.quantize(joined, qs), second.w.cpu().numpy(), dq2, (1, 1, 1, 1))
        assert np.array_equal(bits(got), bits(exp2)), after


@pytest.mark.parametrize("tile", ["0", "1", "2", "3"])
def test_conv_i8_ks_reads_a_wider_buffer(port, monkeypatch, tile):
    """A 1x1 layer with and without a stride on the staged input of a padded 3x3 one."""
    from tennis_amd import capi
    monkeypatch.setenv("TSX_CONV_I8_KS", tile)
    rng = np.random.default_rng(62)
    n, c, h, w, cout = 3, 70, 11, 13, 36
    x = rng.integers(-128, 128, (n, c, h, w)).astype(np.int8)
    owner = capi.Conv2dI8(dev(np.zeros((8, c, 3, 3), np.int8)), (1, 1, 1, 1))
    staged = capi.StagedInput(owner, x.shape)
    owner.stage(dev(x), staged)
    wt = rng.integers(-127, 128, (cout, c, 1, 1)).astype(np.int8)
    dq = rng.uniform(1e-4, 3e-4, cout).astype(np.float32)
    for st in (1, 2):
        conv = capi.Conv2dI8(dev(wt), (1, 1, 1, 1), (st, st))
        got = conv.run_staged(staged, dev(dq))[0].cpu().numpy()
        assert np.array_equal(bits(got), bits(port.conv2d_quantized(x, wt, dq, (1, 1, 1, 1), (st, st))))
