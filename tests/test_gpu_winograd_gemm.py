"""The Winograd GEMMs on the matrix cores at the sizes where their tiling can go wrong, bit for bit against the oracle:
channel counts that leave a part of a group of 8 (and a remainder behind the four interleaved chains), output channels
beside a fragment of 32 and a block of 8, tile counts with and without tail columns, one and four column fragments per
wavefront, and a workgroup's wavefronts along rows, along columns and along both."""
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
    (4, 64, 62, 40, 128),      # tail fragments computed with the column blocks
    (6, 20, 6, 42, 33),        # seven tiles of F(6,3) an image, all in the tail: three fragments of 16, an odd number of channel groups
    (8, 131, 18, 110, 128),    # F(6,3): four column fragments per wavefront, the last block of two, and a tail fragment with them
    # wavefronts of a workgroup along the columns, the last of whose groups has one block: two rows of them by two, or four in a row
    (2, 20, 78, 66, 40), (2, 20, 78, 66, 31),      # F(6,3): nine column fragments, a tail fragment with them
    (3, 20, 41, 37, 40), (3, 20, 41, 37, 31),      # F(2,3): 37, two tail fragments with them, or by themselves
    (3, 21, 65, 67, 29),                           # F(2,3): 105 in fours, one with them; remainder channel
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


@pytest.mark.parametrize("entry", ["f63", "f63_fast", "f23"])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_winograd_operands_at_any_float_address(port, entry, offset):
    """Workspace and transformed kernel one to three floats behind a 16-byte boundary: both are float arrays, no more."""
    import ctypes
    import torch
    from tennis_amd import capi
    n, c, h, w, cout = 2, 13, 28, 30, 40
    rng = np.random.default_rng(offset)
    x = rng.uniform(-1, 1, (n, c, h, w)).astype(np.float32)
    wt = rng.standard_normal((cout, c, 3, 3)).astype(np.float32)
    L, mode = capi.lib(), entry[:3]
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(wt).cuda()
    geom = capi.make_geom(x.shape, wt.shape, (1, 1, 1, 1))
    need = getattr(L, "tsx_winograd_%s_workspace_bytes" % entry)(ctypes.byref(geom))
    u = torch.zeros(getattr(L, "tsx_winograd_%s_kernel_bytes" % mode)(cout, c) // 4 + 8, device="cuda")
    workspace = torch.full((need // 4 + 8,), float("nan"), device="cuda")
    out = torch.empty((n, cout, h, w), device="cuda")
    at = ctypes.c_void_p(u.data_ptr() + 4 * offset)
    capi.check(getattr(L, "tsx_winograd_%s_transform_kernel" % mode)(cout, c, capi._ptr(wd), at, capi._stream()))
    capi.check(getattr(L, "tsx_conv2d_winograd_%s_nchw" % entry)(ctypes.byref(geom), capi._ptr(xd), at, 0.0, None, 0, 0.0, capi._ptr(out),
                                                                 ctypes.c_void_p(workspace.data_ptr() + 4 * offset), need, capi._stream()))
    exp = getattr(port, "winograd_" + mode)(x, wt, (1, 1, 1, 1))
    assert np.array_equal(bits(out.cpu().numpy()), bits(exp))
    # and nothing beside the two ranges was written
    assert torch.isnan(workspace[:offset]).all() and torch.isnan(workspace[need // 4 + offset:]).all()
    assert (u[:offset] == 0).all() and (u[u.numel() - 8 + offset:] == 0).all()


def test_winograd_products_in_several_launches(port):
    """More blocks of columns than one launch holds (8.4 million images of 12 tiles, 8 of them chains and 4 tail columns):
    the same bits as the images in parts that take one launch each."""
    import torch
    from tennis_amd import capi
    n, h, w = (1 << 23) + 4097, 6, 8
    if torch.cuda.mem_get_info()[0] < 96 << 30:
        pytest.skip("needs 64 GiB of device memory")
    wt = torch.randn((1, 1, 3, 3), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    x = torch.randn((n, 1, h, w), device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))
    op = capi.Winograd(wt, (1, 1, 1, 1), mode="f23")
    whole = op(x)
    part = (1 << 20) + 33
    for first in range(0, n, part):
        assert torch.equal(whole[first:first + part], op(x[first:first + part])), first
    some = x[-5:].cpu().numpy()
    assert np.array_equal(bits(whole[-5:].cpu().numpy()), bits(port.winograd_f23(some, wt.cpu().numpy(), (1, 1, 1, 1))))
