"""The kernels that int8 calls launch, by name and grid: a plan names the kernels a layer may take, a call's epilogue decides among them.
The library is loaded in a process where the runtime's launch calls are recorded and not carried out: no device and no
memory are needed."""
import json
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RECORDER = r"""
#include <stdint.h>
#include <stdio.h>
#include <string.h>
typedef struct { uint32_t x, y, z; } dims;
static dims grid, block;
static size_t dynamic;
static struct { const void *host; char name[240]; } kernels[8192];
static int count;
char launched[4096];
void **__hipRegisterFatBinary(const void *data) { static void *handle; return &handle; }
void __hipUnregisterFatBinary(void **modules) {}
void __hipRegisterVar() {}
void __hipRegisterManagedVar() {}
void __hipRegisterFunction(void **modules, const void *host, char *device_name, const char *name, unsigned limit, void *a, void *b, void *c, void *d, int *e) {
    if (count < 8192) {
        kernels[count].host = host;
        strncpy(kernels[count++].name, name, 239);
    }
}
unsigned __hipPushCallConfiguration(dims g, dims b, size_t shared, void *stream) { grid = g; block = b; dynamic = shared; return 0; }
unsigned __hipPopCallConfiguration(dims *g, dims *b, size_t *shared, void **stream) { *g = grid; *b = block; *shared = dynamic; *stream = 0; return 0; }
int hipLaunchKernel(const void *f, dims g, dims b, void **args, size_t shared, void *stream) {
    for (int i = 0; i < count; ++i)
        if (kernels[i].host == f) sprintf(launched + strlen(launched), "%s %u %u;", kernels[i].name, g.x * g.y, b.x);
    return 0;
}
int hipGetLastError(void) { return 0; }
int hipGetDevice(int *device) { *device = 0; return 0; }
int hipFuncSetAttribute(const void *f, int what, int value) { return 0; }
"""

CALLS = r"""
import ctypes, json, sys
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
L = ctypes.CDLL(sys.argv[2])
sys.path.insert(0, sys.argv[4])
from tennis_amd.capi import ConvGeom, Epilogue, SIGNATURES, _ACT
L.tsx_conv2d_i8_staged.argtypes = SIGNATURES["tsx_conv2d_i8_staged"][1]
L.tsx_conv2d_i8_plan_info.argtypes = SIGNATURES["tsx_conv2d_i8_plan_info"][1]
L.tsx_last_error.restype = ctypes.c_char_p
launched = (ctypes.c_char * 4096).in_dll(recorder, "launched")
at = 1 << 20                      # an address that nothing reads
out = []
for n, c, h, w, cout, k, s, act, outputs in json.loads(sys.argv[3]):
    kh, kw = k if isinstance(k, list) else (k, k)
    sh, sw = s if isinstance(s, list) else (s, s)
    geom = ConvGeom(n, c, h, w, cout, kh, kw, kh // 2, kh // 2, kw // 2, kw // 2, sh, sw, 1, 1)
    ho, wo = (h + 2 * (kh // 2) - kh) // sh + 1, (w + 2 * (kw // 2) - kw) // sw + 1
    ep = Epilogue(dq_dev=at, bias_dev=at, act=_ACT[act], slope=0.1)
    if "i8" in outputs or "staged" in outputs:
        ep.q_scales_dev, ep.n_qscales = at, n
    if "staged" in outputs:
        ep.staged_out_dev, ep.staged_hs, ep.staged_ws, ep.staged_cp = at, ho, wo, (cout + 63) // 64 * 64
    if "join" in outputs:
        ep.residual_dev = at
    launched.value = b""
    rc = L.tsx_conv2d_i8_staged(ctypes.byref(geom), at, at, ctypes.byref(ep), at if "f32" in outputs else None, at if "i8" in outputs else None, None, None)
    info = ctypes.create_string_buffer(512)
    assert L.tsx_conv2d_i8_plan_info(ctypes.byref(geom), info, 512) == 0
    out.append([rc, launched.value.decode(), info.value.decode()] if rc == 0 else [rc, L.tsx_last_error().decode(), ""])
print(json.dumps(out))
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    """Calls (n, c, h, w, cout, k, stride, activation, outputs) -> for each the kernel's name with its template arguments, its
    workgroups, the plan's text."""
    from tennis_amd.build import LIB_PATH
    where = tmp_path_factory.mktemp("recorder")
    source, so = where / "recorder.c", where / "librecorder.so"
    source.write_text(RECORDER)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(source)])
    env = {k: v for k, v in os.environ.items() if not k.startswith("TSX_")}

    def routes(calls, **switches):
        run = subprocess.run([sys.executable, "-c", CALLS, str(so), LIB_PATH, json.dumps(calls), ROOT], capture_output=True, text=True, cwd=ROOT,
                             env=dict(env, **{"TSX_CONV_I8_" + k: v for k, v in switches.items()}))
        assert run.returncode == 0, run.stderr
        out = []
        for call, (rc, launched, info) in zip(calls, json.loads(run.stdout)):
            assert rc == 0 and launched.count(";") == 1, (call, rc, launched)
            out.append(launched.rstrip(";").split(" ")[:2] + [dict(word.split("=", 1) for word in info.split())])
        names = subprocess.run(["c++filt"], input="\n".join(name for name, _, _ in out), capture_output=True, text=True, check=True).stdout.splitlines()
        return [("%s<%s>" % re.search(r"(\w+)<([^<>]*)>", name).groups(), int(workgroups), info) for name, (_, workgroups, info) in zip(names, out)]
    return routes


def test_large_plain_fp32_outputs_of_whole_half_lines_are_streamed(route):
    calls = [([32, 256, 56, 56, 512, 1, 2, "none", "f32"], True), ([7, 1024, 32, 32, 2048, 1, 1, "relu", "f32"], True), ([8, 64, 304, 304, 64, 1, 1, "mish", "f32"], True),
             ([4, 64, 128, 128, 64, 1, 1, "none", "f32"], True),                                    # 16 MiB
             ([4, 64, 124, 128, 64, 1, 1, "none", "f32"], False),                                   # less
             ([4, 64, 130, 130, 64, 1, 1, "none", "f32"], False),                                   # planes of 16900 values
             ([32, 64, 56, 56, 256, 1, 1, "relu", "f32 join"], False), ([32, 64, 56, 56, 256, 1, 1, "relu", "f32 staged"], False)]
    for (call, streams), (kernel, _, _) in zip(calls, route([call for call, _ in calls])):
        arguments = kernel[:-1].split("<")[1].split(", ")
        assert kernel.startswith("conv_i8_px_kernel<") and arguments[6] == ("true" if streams else "false"), (call, kernel)


def test_pixel_streams_of_1024_channels_fill_rounds_of_two_workgroups_per_cu(route):
    """Turns by what the busiest CU of an XCD takes: its groups of 32 pixels over 32 CUs, two at a time."""
    calls = [([8, 1024, 40, 58, 384, 1, 1, "mish", "f32 staged"], 73, 3, 4), ([2, 1024, 182, 21, 1024, 1, 1, "mish", "f32 staged"], 30, 8, 4),
             ([20, 1024, 14, 14, 256, 1, 1, "relu", "staged"], 16, 2, 1), ([4, 1024, 74, 74, 1024, 1, 1, "relu", "f32"], 86, 8, 6)]
    for (call, per_xcd, blocks, turns), (kernel, workgroups, _) in zip(calls, route([c[0] for c in calls])):
        assert kernel.startswith("conv_i8_px_kernel<16, 1, ") and workgroups == 8 * blocks * -(-per_xcd // turns), (call, kernel, workgroups)


def test_pixel_streams_whose_planes_share_lines_take_two_blocks_of_channels_at_a_time(route):
    calls = [([10, 64, 54, 54, 2048, 1, 1, "relu", "f32 join"], True), ([32, 256, 19, 19, 4096, 1, 1, "mish", "f32 staged join"], True), ([16, 1024, 37, 37, 2048, 1, 1, "relu", "f32"], True),
             ([9, 256, 33, 35, 2176, 1, 1, "relu", "f32 join"], True),                             # 17 blocks: one at a time
             ([10, 64, 56, 56, 2048, 1, 1, "relu", "f32 join"], False), ([10, 64, 54, 54, 1024, 1, 1, "relu", "f32 join"], False),        # whole lines; 8 blocks
             ([2, 64, 41, 43, 2048, 1, 1, "relu", "f32 join"], False), ([3, 64, 41, 43, 2048, 1, 1, "mish", "f32 join"], False),          # below 32 MiB; 64
             ([10, 64, 54, 54, 2048, 1, 1, "relu", "staged"], False), ([10, 64, 52, 52, 2048, 1, 1, "relu", "f32"], False)]               # no fp32 output; a streamed one
    for (call, panels), (kernel, workgroups, _) in zip(calls, route([c for c, _ in calls])):
        assert kernel.startswith("conv_i8_px_kernel<") and (kernel[:-1].split(", ")[-1] == "true") == panels, (call, kernel)
        assert workgroups % (8 * call[4] // 128) == 0


def test_small_tiles_keep_the_layers_that_gain(route):
    """Little more than a round of two workgroups per CU, few tiles with the exact Mish and tiles that are mostly empty stay on the other kernels."""
    tiles = [([32, 64, 56, 56, 64, 3, 1, "relu", "staged"], "1, 9, 2, 3, false"), ([32, 128, 28, 28, 128, 3, 1, "relu", "staged"], "2, 9, 1, 4, false"),
             ([8, 128, 76, 76, 256, 3, 1, "leaky_relu", "staged"], "2, 9, 1, 4, false"), ([8, 128, 76, 76, 256, 3, 1, "mish", "staged"], "2, 9, 1, 4, true"),
             ([8, 64, 304, 304, 128, 3, 2, "mish", "staged"], "1, 9, 1, 5, true"), ([8, 64, 608, 304, 64, [3, 2], [2, 1], "mish", "staged"], "1, 6, 2, 3, true"),
             ([3, 128, 64, 63, 64, 3, 1, "relu", "staged"], "2, 9, 2, 4, false"),
             ([26, 100, 36, 36, 128, 3, 1, "mish", "staged"], "2, 9, 1, 4, true")]               # (the other kernel: flat tiles)
    for (call, arguments), (kernel, _, _) in zip(tiles, route([c for c, _ in tiles])):
        assert kernel == "conv_i8_pt_kernel<" + arguments + ">", (call, kernel)
    others = [[1, 128, 151, 151, 256, 3, 1, "none", "staged"], [9, 128, 70, 70, 128, 3, 1, "mish", "staged"], [16, 64, 29, 29, 128, 3, 1, "mish", "staged"],
              [20, 128, 12, 251, 256, 3, 2, "mish", "staged"], [8, 128, 7, 167, 512, 3, 2, "none", "staged"]]
    for call, (kernel, _, _) in zip(others, route(others)):
        assert not kernel.startswith("conv_i8_pt_kernel<"), (call, kernel)


def test_the_exact_mish_on_small_tiles_is_compared(route):
    from test_gpu_conv_i8_streams import TILE_STREAMS_WITH_MISH
    calls = [[n, c, h, w, cout, list(taps), list(strides), "mish", "staged"] for n, c, h, w, cout, taps, strides in TILE_STREAMS_WITH_MISH]
    kernels = [kernel for kernel, _, _ in route(calls)]
    assert sorted(kernels) == sorted("conv_i8_pt_kernel<%s, true>" % a for a in
                                     ("1, 9, 1, 3", "1, 9, 2, 3", "1, 9, 4, 3", "1, 9, 1, 5", "1, 9, 2, 5", "1, 6, 1, 3", "1, 6, 2, 3", "2, 9, 1, 4", "2, 9, 2, 4")), kernels


def test_small_tiles_take_one_turn_where_the_compiled_kernels_hold_all_workgroups(route):
    """Three workgroups with five window chunks a thread to a CU, four with six taps: 96 and 128 to an XCD."""
    calls = [([14, 64, 73, 73, 256, 3, 2, "none", "staged"], "1, 9, 1, 5, false", 2, True), ([18, 64, 73, 73, 256, 3, 2, "none", "staged"], "1, 9, 1, 5, false", 2, False),
             ([8, 64, 100, 71, 64, [3, 2], 1, "relu", "staged"], "1, 6, 2, 3, false", 1, True), ([10, 64, 100, 71, 64, [3, 2], 1, "relu", "staged"], "1, 6, 2, 3, false", 1, False),
             ([9, 64, 73, 73, 256, 3, 2, "mish", "staged"], "1, 9, 1, 5, true", 2, True)]
    for (call, arguments, blocks, one), (kernel, workgroups, info) in zip(calls, route([c[0] for c in calls])):
        assert kernel == "conv_i8_pt_kernel<" + arguments + ">", (call, kernel)
        n, _, h, w, _, k, s = call[:7]
        kh, kw = k if isinstance(k, list) else (k, k)
        th, tw = (int(v) for v in info["tile_stream"].split("x"))
        rows, columns = n * ((h + 2 * (kh // 2) - kh) // s + 1), (w + 2 * (kw // 2) - kw) // s + 1
        per_xcd = -(-(-(-rows // th) * -(-columns // tw)) // 8)
        assert (workgroups == 8 * blocks * per_xcd) == one, (call, workgroups, per_xcd)


def test_plans_say_which_pixel_streams_take_joins(route):
    calls = [[40, c, 14, 14, 256, 1, 1, "relu", outputs] for c in (64, 250, 512, 1000) for outputs in ("f32", "f32 join", "staged", "staged join")]
    for call, (kernel, _, info) in zip(calls, route(calls, KS="0")):
        joins = call[1] <= 256
        assert info["pixel_stream"] == "1" and info["pixel_stream_joins"] == str(int(joins)), info
        assert kernel.startswith("conv_i8_px_kernel<") == (joins or "join" not in call[-1]), (call, kernel)


def test_plans_say_which_layers_have_k_in_halves(route):
    layers = [((4, 256, 7, 7, 128, 3, 1), 2), ((32, 512, 7, 7, 96, 3, 1), 2), ((2, 448, 9, 8, 130, 3, 1), 1), ((8, 512, 14, 13, 64, 3, 2), 1), ((8, 512, 14, 14, 128, 3, 2), 2),
              ((6, 640, 5, 5, 128, 5, 1), 2), ((30, 2048, 7, 7, 100, 1, 1), 2), ((9, 1100, 6, 7, 255, 1, 1), 1), ((9, 1536, 6, 7, 255, 1, 1), 2)]
    calls = [(list(layer) + [act, outputs], parts) for layer, parts in layers for outputs in ("f32", "f32 staged", "staged join") for act in ("relu", "mish")]
    for (call, parts), (kernel, _, info) in zip(calls, route([c for c, _ in calls], KS="0", PX="0", FLAT="0", RS="0")):
        assert kernel.startswith("conv_i8_ws_kernel<1, ") and info["k_parts"] == str(parts), (call, kernel, info)
        assert (kernel.split(", ")[6] == "2") == (parts == 2), (call, kernel)


def test_layers_with_special_values_run_on_the_small_tiles(route):
    calls = [[n, c, 104, 104, 256, 3, 1, act, "staged"] for n in (1, 3) for c in (64, 128) for act in ("none", "relu", "leaky_relu")]
    calls += [[n, 64, 16, 16, 8192, 3, 1, "mish", "staged"] for n in (1, 2)]
    for call, (kernel, _, _) in zip(calls, route(calls, KS="0")):
        assert kernel.startswith("conv_i8_pt_kernel<"), (call, kernel)
