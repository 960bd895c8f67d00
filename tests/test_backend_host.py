"""CPU-side checks of the boundary: the C-ABI library exports every symbol include/tsx_hip.h
declares, the C++ operator layer registers the hot-path operators for device "hip", and its
host logic (parameter checking, error behaviour) follows the reference.  No compute calls."""
import ctypes
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_c_abi_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "tsx_hip.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(tsx_[a-z0-9_]+)\s*\(", header))
    assert len(declared) >= 25
    lib = ctypes.CDLL(os.path.join(ROOT, "tennis_amd", "lib", "libtsx_hip.so"))
    missing = [name for name in sorted(declared) if not hasattr(lib, name)]
    assert not missing, missing
    from tennis_amd import capi
    assert declared == set(capi.SIGNATURES), declared ^ set(capi.SIGNATURES)


def test_argument_errors_need_no_device():
    from tennis_amd import capi
    L = capi.lib()
    assert L.tsx_version() == 100
    g = capi.ConvGeom(1, 8, 2, 2, 4, 3, 3, 0, 0, 0, 0, 1, 1, 1, 1)          # 3x3 on 2x2 without padding
    assert L.tsx_conv2d_i8_workspace_bytes(ctypes.byref(g)) == 0
    assert b"empty output" in L.tsx_last_error()
    g = capi.ConvGeom(1, 8, 5, 5, 4, 3, 3, 1, 1, 1, 1, 0, 1, 1, 1)          # zero stride
    assert L.tsx_conv2d_i8_packed_weight_bytes(ctypes.byref(g)) == 0
    g = capi.ConvGeom(1, 8, 9, 9, 4, 5, 5, 1, 1, 1, 1, 1, 1, 1, 1)          # Winograd needs 3x3
    assert L.tsx_winograd_f63_workspace_bytes(ctypes.byref(g)) == 0
    assert L.tsx_quantize_f32_i8(None, -1, None, 1, None, None) == -1
    # geometry bookkeeping of config 2
    g = capi.ConvGeom(32, 256, 28, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    assert L.tsx_conv2d_i8_workspace_bytes(ctypes.byref(g)) == 32 * 30 * 30 * 256
    assert L.tsx_conv2d_i8_packed_weight_bytes(ctypes.byref(g)) == 256 * 256 * 9
    ho, wo = capi.conv_out_size(g)
    assert (ho, wo) == (28, 28)


def test_kernel_choices_need_no_device(monkeypatch):
    """Which kernel a layer takes is decided on the host from the geometry (and the weights' alignment) alone, and the
    plan-info entry points report it: config 2 on the weight-stationary int8 kernel, config 1 on the small-layer fp32
    kernel, and the environment switches that tests use to put small layers on a given kernel."""
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_I8_FLAT", "TSX_CONV_I8_RS", "TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED"):
        monkeypatch.delenv(name, raising=False)

    def i8(geom):
        buf = ctypes.create_string_buffer(256)
        assert L.tsx_conv2d_i8_plan_info(ctypes.byref(geom), buf, len(buf)) == 0
        return dict(word.split("=", 1) for word in buf.value.decode().split())

    def f32(geom, weights_address=4096):
        buf = ctypes.create_string_buffer(256)
        assert L.tsx_conv2d_f32_plan_info(ctypes.byref(geom), ctypes.c_void_p(weights_address), buf, len(buf)) == 0
        return dict(word.split("=", 1) for word in buf.value.decode().split())

    c2 = capi.ConvGeom(32, 256, 28, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    assert i8(c2)["fp32_kernel"] == "weight_stationary"
    monkeypatch.setenv("TSX_CONV_I8_RS", "0")
    assert i8(c2)["fp32_kernel"] != "weight_stationary"
    c1 = capi.ConvGeom(1, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    assert f32(c1) == {"kernel": "small_3x3", "tiles": "196"}
    assert f32(c1, weights_address=4100)["kernel"] == "staged_32x32_ksplit"       # rows of A not 16-byte aligned
    big = capi.ConvGeom(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    assert f32(big)["kernel"] == "staged_64x64"
    monkeypatch.setenv("TSX_CONV_F32_SMALL", "force")
    assert f32(big)["kernel"] == "small_3x3"
    monkeypatch.setenv("TSX_CONV_F32_SMALL", "0")
    assert f32(c1)["kernel"] == "register_fed"
    assert L.tsx_conv2d_f32_plan_info(ctypes.byref(c1), None, None, 0) == -1


def test_fp32_plan_info_names_the_kernel_of_a_call_with_workspace(monkeypatch):
    """A layer has use for a workspace exactly where the plan names a kernel of its own for that call."""
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT"):
        monkeypatch.delenv(name, raising=False)

    def plan(geom):
        buf = ctypes.create_string_buffer(256)
        assert L.tsx_conv2d_f32_plan_info(ctypes.byref(geom), ctypes.c_void_p(4096), buf, len(buf)) == 0
        info = dict(word.split("=", 1) for word in buf.value.decode().split())
        assert ("workspace_kernel" in info) == (L.tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(4096)) > 0)
        return info

    large = capi.ConvGeom(8, 256, 28, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
    info = plan(large)
    assert info["workspace_kernel"] == "bf16_split" and info["kernel"] == "staged_64x64"
    rows, positions = map(int, info["workspace_tile"].split("x"))
    assert rows % 32 == 0 and positions % 32 == 0 and info["workspace_window"] in ("flat", "segments")
    monkeypatch.setenv("TSX_CONV_F32_SPLIT", "0")
    assert "workspace_kernel" not in plan(large)
    monkeypatch.delenv("TSX_CONV_F32_SPLIT")
    assert "workspace_kernel" not in plan(capi.ConvGeom(1, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1))
    assert "workspace_kernel" not in plan(capi.ConvGeom(1, 128, 28, 28, 128, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1))


@pytest.mark.parametrize("layer, takes", [
    # us without a workspace / with one: 59 / 31, 27 / 18, 35 / 32, 88 / 36 ...
    ((10, 78, 20, 20, 971, 3, 2, 1), True), ((1, 85, 42, 42, 84, 3, 2, 1), True), ((2, 179, 81, 81, 292, 1, 1, 0), True), ((4, 90, 121, 138, 32, 3, 2, 1), True),
    # ... and 62 / 88, 40 / 46, 44 / 49, 20 / 25, 89 / 98
    ((3, 124, 261, 261, 32, 3, 2, 1), False), ((25, 32, 11, 179, 432, 1, 1, 0), False), ((2, 31, 103, 201, 541, 1, 1, 0), False),
    ((1, 32, 68, 173, 747, 1, 1, 0), False), ((8, 32, 216, 216, 31, 5, 2, 2), False),
])
def test_fp32_layers_use_a_workspace_where_that_is_faster(monkeypatch, layer, takes):
    from tennis_amd import capi
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT", "TSX_CONV_F32_TILE"):
        monkeypatch.delenv(name, raising=False)
    n, c, h, w, cout, k, stride, pad = layer
    geom = capi.ConvGeom(n, c, h, w, cout, k, k, pad, pad, pad, pad, stride, stride, 1, 1)
    assert (capi.lib().tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(4096)) > 0) == takes


def test_every_tile_of_the_bf16_split_kernel_is_reached(monkeypatch):
    """Each tile that TSX_CONV_F32_SPLIT can name takes some layer, is no twin of another one, and is what the planner
    chooses for some layer by itself."""
    import random
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT"):
        monkeypatch.delenv(name, raising=False)
    rng = random.Random(1)
    between = lambda lo, hi: int(round(lo * (hi / lo) ** rng.random()))
    layers = []
    for _ in range(12000):
        k = rng.choice([1, 3, 5])
        pad, stride = rng.choice([0, k // 2, k // 2]), rng.choice([1, 1, 2])
        layers.append(capi.ConvGeom(between(1, 32), between(3, 1024), between(5, 304), between(5, 304), between(16, 1024), k, k, pad, pad, pad, pad,
                                    stride, stride, 1, 1))

    def tile(geom):
        buf = ctypes.create_string_buffer(256)
        assert L.tsx_conv2d_f32_plan_info(ctypes.byref(geom), ctypes.c_void_p(4096), buf, len(buf)) == 0
        info = dict(word.split("=", 1) for word in buf.value.decode().split())
        return (geom.kh, info["workspace_tile"], info["workspace_patch"]) if "workspace_kernel" in info else None

    chosen = {tile(geom) for geom in layers} - {None}
    named = {}
    for number in range(1, 65):
        monkeypatch.setenv("TSX_CONV_F32_SPLIT", str(number))
        found = next((t for t in map(tile, layers[:3000]) if t is not None), None)
        if found is not None:
            named.setdefault((number - 1) // 2, set()).add(found)
    assert sorted(named) == list(range(len(named))), "tiles that take no layer"
    names = [t for tiles in named.values() for t in tiles]
    assert len(names) == len(set(names)) == len(named) and set(names) == chosen, set(names) ^ chosen


def test_other_kernels_switches_keep_layers_off_the_k_split_kernel_where_they_have_a_value(monkeypatch):
    from tennis_amd import capi
    L = capi.lib()
    layer = capi.ConvGeom(1, 256, 14, 14, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)

    def kernel(**switches):
        buf = ctypes.create_string_buffer(256)
        with monkeypatch.context() as m:
            for name in ("FLAT", "RS", "KS"):
                m.delenv("TSX_CONV_I8_" + name, raising=False)
            for name, value in switches.items():
                m.setenv("TSX_CONV_I8_" + name, value)
            assert L.tsx_conv2d_i8_plan_info(ctypes.byref(layer), buf, len(buf)) == 0
        return dict(word.split("=", 1) for word in buf.value.decode().split())["kernel"]

    assert kernel() == "k_split"
    for name in ("FLAT", "RS"):
        assert kernel(**{name: ""}) == "k_split", name
        for value in ("0", "1", "force"):
            assert kernel(**{name: value}) != "k_split", (name, value)
        assert kernel(**{name: "force", "KS": "1"}) == "k_split"
        assert kernel(**{name: "0", "KS": "0"}) == "window_stationary"


@pytest.mark.parametrize("layer, fragments, tiles", [
    ((10, 287, 139, 59, 162, 3, 2, 1), 3, 512), ((28, 330, 130, 134, 23, 5, 2, 2), 1, 1820), ((31, 54, 50, 50, 28, 5, 1, 2), 2, 310),
])
def test_int8_windows_may_fill_64_kib(monkeypatch, layer, fragments, tiles):
    """The largest tile whose two windows fit: what only some activations need in LDS beside them is no other layer's loss."""
    from tennis_amd import capi
    for name in ("FLAT", "RS", "KS"):
        monkeypatch.delenv("TSX_CONV_I8_" + name, raising=False)
    n, c, h, w, cout, k, stride, pad = layer
    geom = capi.ConvGeom(n, c, h, w, cout, k, k, pad, pad, pad, pad, stride, stride, 1, 1)
    buf = ctypes.create_string_buffer(256)
    assert capi.lib().tsx_conv2d_i8_plan_info(ctypes.byref(geom), buf, len(buf)) == 0
    info = dict(word.split("=", 1) for word in buf.value.decode().split())
    assert info["kernel"] == "window_stationary" and (int(info["fragments_per_wavefront"]), int(info["tiles"])) == (fragments, tiles)


@pytest.mark.parametrize("layer, fragments", [
    # two where fragments are whole and planes are whole cache lines ...
    ((32, 256, 56, 56, 64, 1, 1, 0), "2"), ((32, 128, 28, 28, 512, 1, 1, 0), "2"),
    # ... the model's one where they are not
    ((13, 29, 226, 74, 52, 1, 1, 0), "1"), ((24, 6, 91, 91, 47, 1, 1, 0), "1"), ((13, 8, 29, 29, 776, 3, 1, 0), "1"),
    ((3, 96, 122, 27, 801, 1, 1, 0), "1"), ((7, 168, 166, 176, 32, 1, 1, 0), "1"),
])
def test_int8_layers_of_one_tap_take_two_fragments_where_that_pays(monkeypatch, layer, fragments):
    from tennis_amd import capi
    for name in ("FLAT", "RS"):
        monkeypatch.delenv("TSX_CONV_I8_" + name, raising=False)
    monkeypatch.setenv("TSX_CONV_I8_KS", "0")
    n, c, h, w, cout, k, stride, pad = layer
    geom = capi.ConvGeom(n, c, h, w, cout, k, k, pad, pad, pad, pad, stride, stride, 1, 1)
    buf = ctypes.create_string_buffer(256)
    assert capi.lib().tsx_conv2d_i8_plan_info(ctypes.byref(geom), buf, len(buf)) == 0
    info = dict(word.split("=", 1) for word in buf.value.decode().split())
    assert (info["kernel"], info["fragments_per_wavefront"]) == ("window_stationary", fragments)


def test_kept_fp32_plans_follow_what_they_depend_on(monkeypatch):
    """A thread keeps its plans: with every switch, weights' alignment and geometry in turn they are what a thread that has
    planned nothing yet answers."""
    import threading
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT", "TSX_CONV_F32_TILE"):
        monkeypatch.delenv(name, raising=False)

    def plan(geom, address):
        buf = ctypes.create_string_buffer(256)
        assert L.tsx_conv2d_f32_plan_info(ctypes.byref(geom), ctypes.c_void_p(address), buf, len(buf)) == 0
        return buf.value, L.tsx_conv2d_f32_workspace_bytes(ctypes.byref(geom), ctypes.c_void_p(address))

    def in_a_new_thread(*args):
        answer = []
        thread = threading.Thread(target=lambda: answer.append(plan(*args)))
        thread.start()
        thread.join()
        return answer[0]

    layers = [capi.ConvGeom(8, 256, 28, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1), capi.ConvGeom(8, 256, 28, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 2, 1),
              capi.ConvGeom(8, 256, 28, 28, 256, 3, 3, 1, 0, 1, 1, 1, 1, 1, 1), capi.ConvGeom(1, 128, 28, 28, 128, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1),
              capi.ConvGeom(4, 100, 33, 41, 150, 5, 5, 2, 2, 2, 2, 1, 1, 1, 1)]
    answers = set()
    for switch in ({}, {"TSX_CONV_F32_SPLIT": "0"}, {"TSX_CONV_F32_SPLIT": "3"}, {"TSX_CONV_F32_TILE": "1"}, {"TSX_GEMM_F32_REGFED": "0"}, {}):
        with monkeypatch.context() as m:
            for name, value in switch.items():
                m.setenv(name, value)
            for geom in layers:
                for address in (4096, 4100):
                    first = plan(geom, address)
                    assert plan(geom, address) == first == in_a_new_thread(geom, address), (switch, address)
                    answers.add(first)
    assert len(answers) > 10


def test_hot_path_operators_are_registered_for_hip():
    from tennis_amd import operators as ops
    for name in ops.SYMBOLS:
        assert hasattr(ops.lib(), name)
    for op in ("quantize", "conv2d_quantized", "conv2d", "conv2d_winograd", "inner_prod", "add_bias", "relu", "leaky_relu",
               "pooling2d", "global_pooling2d", "add", "depthwise_conv2d", "conv2d_v2", "conv2d_winograd_v2",
               "depthwise_conv2d_v2", "pooling2d_v2", "concat", "_resize2d", "mul", "softplus", "tanh",
               "conv2d_quantized_fused"):
        assert ops.is_registered("hip", op), op
    assert not ops.is_registered("hip", "softmax")
    assert not ops.is_registered("cpu", "conv2d")            # this library ships no host operators
    with pytest.raises(ops.OperatorNotFound):
        ops.check_params("softmax", {})                       # strict: no silent fallback


def test_parameter_checking_follows_the_reference():
    from tennis_amd import operators as ops
    good = ops.conv_params((1, 1, 1, 1))
    good["dequantize_scales"] = np.ones(4, np.float32)
    ops.check_params("conv2d_quantized", good)
    # required field missing (src/runtime/operator.cpp:174-193)
    missing = dict(good)
    del missing["dequantize_scales"]
    with pytest.raises(ops.OperatorError, match="dequantize_scales"):
        ops.check_params("conv2d_quantized", missing)
    # unknown parameter names are rejected in strict mode (operator.cpp:26-38)
    with pytest.raises(ops.OperatorError, match="Unidentified param"):
        ops.check_params("conv2d_quantized", dict(good, quantize_scale=np.ones(1, np.float32)))
    # the typo'd spelling of dilation is accepted, none at all is not (base_conv2d.cpp:51-60)
    typo = dict(good)
    typo["dialations"] = typo.pop("dilation")
    ops.check_params("conv2d_quantized", typo)
    none = dict(good)
    del none["dilation"]
    with pytest.raises(ops.OperatorError, match="must set dilation or dialations"):
        ops.check_params("conv2d_quantized", none)
    # padding / stride on batch or channel are refused
    bad = dict(good, padding=np.array([[1, 0], [0, 0], [1, 1], [1, 1]], np.int32))
    with pytest.raises(ops.OperatorError, match="do not support padding"):
        ops.check_params("conv2d", {k: v for k, v in bad.items() if k != "dequantize_scales"})
    bad = dict(good, stride=np.array([1, 2, 1, 1], np.int32))
    with pytest.raises(ops.OperatorError, match="do not support stride"):
        ops.check_params("conv2d_quantized", bad)
    with pytest.raises(ops.OperatorError, match="do not support format"):
        ops.check_params("conv2d_quantized", dict(good, format="NCDHW"))
    with pytest.raises(ops.OperatorError):
        ops.check_params("add_bias", {})                      # needs format or dim
    ops.check_params("add_bias", {"dim": np.array([1], np.int32)})
    ops.check_params("quantize", {"quantize_scale": np.ones(3, np.float32)})
    with pytest.raises(ops.OperatorError, match="quantize_scale"):
        ops.check_params("quantize", {})
    with pytest.raises(ops.OperatorError, match="scale"):
        ops.check_params("leaky_relu", {})
    # pooling2d: ksize / stride / padding on the two image axes only (base_pooling2d.cpp:66-98)
    pool = {"format": "NCHW", "type": np.array([0], np.int32), "padding": np.zeros((4, 2), np.int32),
            "ksize": np.array([1, 1, 3, 3], np.int32), "stride": np.array([1, 1, 2, 2], np.int32)}
    ops.check_params("pooling2d", pool)                       # padding_type is optional (BLACK)
    with pytest.raises(ops.OperatorError, match="do not support ksize"):
        ops.check_params("pooling2d", dict(pool, ksize=np.array([1, 2, 3, 3], np.int32)))
    with pytest.raises(ops.OperatorError, match="do not support padding"):
        ops.check_params("pooling2d", dict(pool, padding=np.array([[0, 0], [0, 1], [0, 0], [0, 0]], np.int32)))
    with pytest.raises(ops.OperatorError, match="type"):
        ops.check_params("global_pooling2d", {"format": "NCHW"})
    ops.check_params("add", {})
    ops.check_params("depthwise_conv2d", {k: v for k, v in good.items() if k != "dequantize_scales"})


def seconds_per_call(calls):
    import time
    best = 1e9
    for _ in range(7):
        start = time.perf_counter()
        for call in calls:
            call()
        best = min(best, (time.perf_counter() - start) / len(calls))
    return best


def test_plans_of_many_channels_cost_no_more(monkeypatch):
    """Planning a layer of 2048 channels weighs as many tiles as one of 64, and only those numbers of slices that can win."""
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT", "TSX_CONV_F32_TILE"):
        monkeypatch.delenv(name, raising=False)

    def plans(channels):      # more layers than a thread keeps: each call plans
        geoms = [capi.ConvGeom(8, channels, 28 + i, 28, 256, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1) for i in range(1500)]
        return seconds_per_call([lambda g=g: L.tsx_conv2d_f32_workspace_bytes(ctypes.byref(g), ctypes.c_void_p(4096)) for g in geoms])

    assert any(plans(2048) < 1.6 * plans(64) for _ in range(3))      # (another process may take the CPU meanwhile)


def test_the_layers_of_a_network_are_planned_once(monkeypatch):
    """Sixty layers in turn take the time of one again and again: none displaces another's plan."""
    import random
    from tennis_amd import capi
    L = capi.lib()
    for name in ("TSX_CONV_F32_SMALL", "TSX_GEMM_F32_REGFED", "TSX_CONV_F32_SPLIT", "TSX_CONV_F32_TILE"):
        monkeypatch.delenv(name, raising=False)
    rng = random.Random(2)
    geoms = [capi.ConvGeom(rng.choice([1, 8, 32]), 64 * rng.randint(1, 32), size, size, 64 * rng.randint(1, 32), k, k, k // 2, k // 2, k // 2, k // 2, 1, 1, 1, 1)
             for k, size in zip([1, 3] * 30, [7, 14, 28, 56] * 15)]
    call = lambda g: L.tsx_conv2d_f32_workspace_bytes(ctypes.byref(g), ctypes.c_void_p(4096))
    in_turn = lambda: seconds_per_call([lambda g=g: call(g) for g in geoms * 20])
    alone = lambda: max(seconds_per_call([lambda g=g: call(g)] * 200) for g in geoms[::6])
    assert any(in_turn() < 1.5 * alone() for _ in range(3))
