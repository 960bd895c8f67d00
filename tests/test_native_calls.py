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


# ---------------------------------------------------------------- copies and stored layers

def _on_host(capi, monkeypatch):
    monkeypatch.setattr(capi, "_dev", lambda t, dtype: t)


@pytest.mark.parametrize("how", ["deepcopy", "copy", "pickle"])
def test_a_layer_can_be_copied_and_stored(capi, monkeypatch, how):
    import torch
    _on_host(capi, monkeypatch)
    conv = capi.Conv2dI8(torch.arange(2 * 3 * 9, dtype=torch.int8).view(2, 3, 3, 3), (1, 0, 1, 0), (2, 1), (1, 2), padding_value=-3)
    other = {"deepcopy": copy.deepcopy, "copy": copy.copy, "pickle": lambda c: pickle.loads(pickle.dumps(c))}[how](conv)
    assert torch.equal(other.w, conv.w) and (other.w is conv.w) == (how == "copy")
    assert (other.pads, other.strides, other.dilations, other.padding_value) == ((1, 0, 1, 0), (2, 1), (1, 2), -3.0)
    assert other._state is not conv._state and type(other._state) is type(conv._state)


def test_a_layer_stored_without_its_native_state_loads(capi, monkeypatch):
    """What a layer's pickle held before there was a native state."""
    import torch
    _on_host(capi, monkeypatch)
    conv = object.__new__(capi.Conv2dI8)
    conv.__setstate__(dict(w=torch.zeros((2, 3, 1, 1), dtype=torch.int8), pads=(0,) * 4, strides=(1, 1), dilations=(1, 1), padding_value=0.0,
                           _packed={}, _workspace=None))
    assert type(conv._state).__name__ == "ConvState"


def test_a_stored_layer_is_called_in_a_process_that_made_none(capi, monkeypatch):
    """The library is loaded by the first call that needs it, also where that is a call of a layer read from a file."""
    import torch
    gemm = object.__new__(capi.GemmI8)
    gemm.__dict__.update(w=torch.zeros((64, 8), dtype=torch.int8), transpose=False, n=8, k=64, packed=torch.zeros(8192, dtype=torch.uint8), _workspace=None)
    conv = object.__new__(capi.Conv2dI8)
    conv.__setstate__(dict(w=torch.zeros((2, 3, 1, 1), dtype=torch.int8), pads=(0,) * 4, strides=(1, 1), dilations=(1, 1), padding_value=0.0,
                           _packed={}, _workspace=None))
    for call in (lambda: gemm(torch.zeros((2, 64), dtype=torch.int8)), lambda: conv(torch.zeros((1, 3, 4, 4), dtype=torch.int8))):
        monkeypatch.setattr(capi, "_native_module", capi._NotLoaded())
        monkeypatch.setattr(capi, "_lib", None)
        with pytest.raises(capi.TsxError, match="device tensor"):
            call()


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["deepcopy", "pickle"])
def test_copied_layers_and_networks_compute_the_same(capi, how):
    import torch
    from tennis_amd import resnet50
    twin = copy.deepcopy if how == "deepcopy" else lambda c: pickle.loads(pickle.dumps(c))
    conv, dq = _layer(capi)
    x = _input(2, 40, 9, 11)
    first = conv(x, dq=dq)[0]                         # a state that holds a plan
    assert torch.equal(first, twin(conv)(x, dq=dq)[0])
    net = resnet50.ResNet50Int8(*resnet50.make_parameters(width=0.25, blocks=[1, 1, 1, 1], classes=10))
    image = torch.randn((1, 3, 64, 64), device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    net.calibrate(image)
    assert torch.equal(net.forward(image), twin(net).forward(image))


@pytest.mark.gpu
def test_a_layer_follows_its_attributes(capi):
    """Padding and its value set after calls: the layer computes what one made with them computes."""
    import torch
    conv, dq = _layer(capi)
    x = _input(2, 40, 9, 11)
    conv(x, dq=dq)
    for change in ({"padding_value": -7.0}, {"pads": (0, 1, 2, 0)}, {"pads": (1, 1, 1, 1), "padding_value": 3.0}):
        for name, value in change.items():
            setattr(conv, name, value)
        made = capi.Conv2dI8(conv.w, conv.pads, padding_value=conv.padding_value)
        assert torch.equal(conv(x, dq=dq)[0], made(x, dq=dq)[0]), change


# ---------------------------------------------------------------- threads and re-entry

SLOW = "#include <unistd.h>\nint slow(const void *x, long long n, void *out, void *stream) { usleep(400000); return 0; }\n"


@pytest.mark.gpu
def test_other_threads_run_while_a_launch_waits(capi, tmp_path):
    """An entry point that blocks, as a launch into a full queue does, stands in for tsx_relu_f32."""
    import torch
    source, so = tmp_path / "slow.c", tmp_path / "libslow.so"
    source.write_text(SLOW)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(source)])
    slow = ctypes.CDLL(str(so)).slow
    real = {name: ctypes.cast(getattr(capi.lib(), name), ctypes.c_void_p).value for name in capi.SIGNATURES}
    x = torch.zeros(16, device="cuda")
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.005)

    thread = threading.Thread(target=tick)
    capi._native().bind(dict(real, tsx_relu_f32=ctypes.cast(slow, ctypes.c_void_p).value), capi.TsxError)
    try:
        thread.start()
        began = time.perf_counter()
        capi.relu(x)
        ended = time.perf_counter()
    finally:
        stop.set()
        thread.join()
        capi._native().bind(real, capi.TsxError)
    assert ended - began > 0.39
    assert sum(began < t < ended for t in ticks) >= 10
    assert torch.equal(capi.relu(x), x)


@pytest.mark.gpu
def test_threads_share_a_layer(capi):
    """Four threads call one layer with more shapes than it keeps plans for, on one stream: staging and convolution of a
    call are enqueued together although the calls share a workspace, and a plan outlives its place among the kept ones."""
    import torch
    conv, dq = _layer(capi)
    inputs = [_input(1 + i % 3, 40, 5 + i, 7 + 2 * i, seed=i) for i in range(12)]
    want = [conv(x, dq=dq)[0] for x in inputs]
    torch.cuda.synchronize()
    wrong = []

    def work(k):
        for turn in range(40):
            i = (5 * turn + 3 * k) % len(inputs)
            got = conv(inputs[i], dq=dq)[0]
            if not torch.equal(got, want[i]):
                wrong.append((k, turn, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.gpu
def test_a_call_made_while_another_reads_its_arguments(capi):
    """A staged output whose attribute runs the layer on other shapes: the outer call's plan stays what it is."""
    import torch
    conv, dq = _layer(capi)
    x = _input(2, 40, 12, 13)
    consumer = capi.Conv2dI8(_dev(np.ones((8, 48, 1, 1), np.int8)))
    qs = torch.full((2,), 5.0, device="cuda")
    plain = capi.StagedInput(consumer, (2, 48, 12, 13))
    kw = dict(dq=dq, act="relu", q_scales=qs)
    want = conv(x, staged_out=plain, **kw)[0]

    class Busy(capi.StagedInput):
        @property
        def hs(self):
            for i in range(20):
                conv(_input(1, 40, 4 + i, 6), dq=dq)
            return self._hs

        @hs.setter
        def hs(self, v):
            self._hs = v

    busy = Busy(consumer, (2, 48, 12, 13))
    got = conv(x, staged_out=busy, **kw)[0]
    assert torch.equal(got, want) and torch.equal(busy.buf, plain.buf)


# ---------------------------------------------------------------- workspaces

@pytest.mark.gpu
def test_a_larger_shape_gives_the_smaller_workspace_back(capi):
    import torch
    conv, dq = _layer(capi, c=64)
    shapes = [(1, 64, 180 + 40 * i, 256) for i in range(6)]
    small = _input(*shapes[0])
    conv(small, dq=dq)                                # weights packed
    del small
    conv._workspace = None
    before = torch.cuda.memory_allocated()
    first = None
    for shape in shapes:
        out = conv(_input(*shape), dq=dq)[0]
        first = out.cpu() if first is None else first
        del out
    kept = torch.cuda.memory_allocated() - before
    assert kept <= conv._workspace.numel() + 4096, (kept, conv._workspace.numel())
    assert torch.equal(conv(_input(*shapes[0]), dq=dq)[0].cpu(), first)


@pytest.mark.gpu
def test_a_captured_layer_outlives_its_workspace(capi):
    """A larger shape replaces the layer's workspace; a graph captured before goes on with the one it was captured with."""
    import torch
    conv, dq = _layer(capi)
    x = _input(2, 40, 14, 15)
    want = conv(x, dq=dq)[0]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = conv(x, dq=dq)[0]
    large = _input(4, 40, 60, 62)
    for turn in range(3):
        conv(large, dq=dq)
        small = torch.full((conv._workspace.numel(),), 77, dtype=torch.int8, device="cuda")    # where a freed workspace would lie
        out.zero_()
        graph.replay()
        assert torch.equal(out, want) and (small == 77).all(), turn
        large = torch.cat([large, large])
    assert len(conv._graph_workspaces) == 1 and copy.deepcopy(conv)._graph_workspaces == []
