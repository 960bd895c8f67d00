"""The Winograd GEMMs on the matrix cores at the sizes where their tiling can go wrong, bit for bit against the oracle:
channel counts that leave a part of a group of 8 (and a remainder behind the four interleaved chains), output channels
beside a fragment of 32 and a block of 8, tile counts with and without tail columns, one and two column fragments per
wavefront."""
import numpy as np
import pytest

from _util import bits

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, cout
    (1, 1, 3, 3, 1),           # one channel, one tile: everything is padding
    (2, 4, 17, 17, 31),        # nine tiles of F(6,3): one chain block and one tail column per image
    (3, 12, 16, 15, 33),       # a channel group half filled, a fragment of rows with one row
    (2, 13, 48, 24, 40),       # 32 tiles of F(6,3), no tail; remainder channel
    (1, 23, 30, 31, 72),       # 30 tiles: 24 chained, 6 in the tail; three remainder channels
    (5, 34, 28, 28, 65),       # columns of several images in one fragment
    (4, 64, 62, 40, 128),      # enough wavefronts for two fragments each, an odd number of fragments
]


@pytest.mark.parametrize("mode", ["f63", "f23"])
@pytest.mark.parametrize("case", CASES)
def test_winograd_gemm_edges(port, case, mode):
    import torch
    from tennis_amd import capi
    n, c, h, w, cout = case
    rng = np.random.default_rng(c)
    x = rng.uniform(-1, 1, (n, c, h, w)).astype(np.float32)
    wt = (rng.standard_normal((cout, c, 3, 3)) * np.sqrt(2.0 / (c * 9))).astype(np.float32)
    op = capi.Winograd(torch.from_numpy(wt).cuda(), (1, 1, 1, 1), padding_value=0.25, mode=mode)
    got = op(torch.from_numpy(x).cuda()).cpu().numpy()
    exp = getattr(port, "winograd_" + mode)(x, wt, (1, 1, 1, 1), padding_value=0.25)
    assert np.array_equal(bits(got), bits(exp)), (bits(got) != bits(exp)).mean()
