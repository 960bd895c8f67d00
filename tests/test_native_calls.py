"""What tennis_amd.capi's calls keep to although a native extension does their host work: errors of the type torch raises,
layers that can be copied and stored, other Python threads that run while a launch waits, workspaces that are given back."""
import copy
import ctypes
import pickle
import subprocess
import threading
import time

import numpy as np
import pytest


@pytest.fixture
def capi():
    from tennis_amd import capi as c
    c.lib()
    return c


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _layer(capi, c=40, cout=48, k=3, seed=5):
    rng = np.random.default_rng(seed)
    conv = capi.Conv2dI8(_dev(rng.integers(-127, 128, (cout, c, k, k)).astype(np.int8)), (k // 2,) * 4)
    return conv, _dev(rng.uniform(1e-4, 1e-3, cout).astype(np.float32))


def _input(n, c, h, w, seed=6):
    return _dev(np.random.default_rng(seed).integers(-128, 128, (n, c, h, w)).astype(np.int8))


# ---------------------------------------------------------------- errors

@pytest.mark.gpu
def test_out_of_memory_is_torch_out_of_memory(capi):
    """A program that halves its batch when an output does not fit catches torch.OutOfMemoryError."""
    import torch
    side = 1 << 17                                    # 64 GiB of fp32 products
    column = torch.zeros((side, 1), device="cuda")
    row = torch.zeros((1, side), device="cuda")
    gemm = capi.GemmI8(torch.zeros((64, side), dtype=torch.int8, device="cuda"))
    lhs, dq = torch.zeros((side, 64), dtype=torch.int8, device="cuda"), torch.zeros(side, device="cuda")
    conv = capi.Conv2dI8(torch.zeros((4096, 64, 1, 1), dtype=torch.int8, device="cuda"))
    x, conv_dq = torch.zeros((1, 64, 1024, 1024), dtype=torch.int8, device="cuda"), torch.zeros(4096, device="cuda")
    image, filters = torch.zeros((1, 1, 1024, 1024), device="cuda"), torch.zeros((4096, 1, 1, 1), device="cuda")
    torch.cuda.empty_cache()
    total = torch.cuda.mem_get_info()[1]
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 30)) / total)    # the allocator refuses by itself
    try:
        for call in (lambda: capi.inner_prod_f32(column, row), lambda: gemm(lhs, dq=dq), lambda: conv(x, dq=conv_dq),
                     lambda: capi.conv2d_f32(image, filters)):
            with pytest.raises(torch.OutOfMemoryError):
                call()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
