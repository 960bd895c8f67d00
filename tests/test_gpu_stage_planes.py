"""The staging of an int8 convolution's input, [n][c][h][w] -> [n][hs][ws][cp] with halo, byte for byte against the
quantize oracle and a numpy layout: runs of four pixels and their overlapping last one, channel counts around the
chunks of 16 and blocks of 64, several workgroups along a plane, maps cut off by a stride, odd alignments."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# n, c, h, w, kernel, stride, pads (t, b, l, r)
CASES = [
    (1, 1, 2, 2, 1, 1, (0, 0, 0, 0)),          # one lane
    (2, 15, 1, 5, 1, 1, (0, 0, 0, 0)),         # the last lane overlaps the first
    (3, 17, 13, 13, 3, 2, (1, 1, 1, 1)),
    (1, 64, 7, 9, 3, 1, (1, 1, 1, 1)),         # one scale: half to even up to the last element but 0..7
    (2, 65, 16, 16, 5, 1, (2, 2, 2, 2)),       # 64 lanes exactly
    (1, 129, 5, 205, 3, 1, (0, 1, 2, 0)),      # five workgroups of 52 lanes along the plane
    (5, 30, 31, 33, 3, 3, (0, 0, 0, 0)),       # rows and columns behind the last window are not staged
    (2, 9, 3, 2, 3, 1, (4, 4, 3, 3)),          # a map smaller than its halo
]


@pytest.mark.parametrize("quantized", [True, False])
@pytest.mark.parametrize("case", CASES, ids=str)
def test_staged_bytes(port, case, quantized):
    import ctypes
    import torch
    from tennis_amd import capi
    n, c, h, w, k, stride, pads = case
    rng = np.random.default_rng(7)
    src = (rng.standard_normal((n, c, h, w)) * 40).astype(np.float32)
    src.ravel()[::3] = np.round(src.ravel()[::3]) + 0.5
    scales = np.ones(n, np.float32) if n == 1 else rng.uniform(0.5, 1.5, n).astype(np.float32)
    q = port.quantize(src, scales)
    # one element into an allocation: the smallest alignment a tensor can have
    flat = torch.from_numpy(src if quantized else q).reshape(-1)
    x = torch.cat([flat[:1], flat]).cuda()[1:].view(n, c, h, w)
    conv = capi.Conv2dI8(torch.ones((4, c, k, k), dtype=torch.int8, device="cuda"), pads, (stride, stride), padding_value=-3)
    g = conv._plan((n, c, h, w))[0]
    hs, ws, cp = (ctypes.c_int32() for _ in range(3))
    capi.check(capi.lib().tsx_conv2d_i8_staged_dims(ctypes.byref(g), ctypes.byref(hs), ctypes.byref(ws), ctypes.byref(cp)))
    hs, ws, cp = hs.value, ws.value, cp.value
    staged = torch.full((n, hs, ws, cp), 99, dtype=torch.int8, device="cuda")
    s = torch.from_numpy(scales).cuda()
    capi.check(capi.lib().tsx_conv2d_i8_stage(ctypes.byref(g), x.data_ptr(), int(quantized), s.data_ptr() if quantized else None, n if quantized else 0,
                                              -3.0, staged.data_ptr(), staged.numel(), torch.cuda.current_stream().cuda_stream))
    want = np.zeros((n, hs, ws, cp), np.int8)
    want[..., :c] = -3
    t, l = pads[0], pads[2]
    rows, cols = max(0, min(h, hs - t)), max(0, min(w, ws - l))
    want[:, t:t + rows, l:l + cols, :c] = q.transpose(0, 2, 3, 1)[:, :rows, :cols]
    assert np.array_equal(staged.cpu().numpy(), want)
