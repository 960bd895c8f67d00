"""The grids of kernels whose launches grow with the batch, at extents no test allocates: a launch holds fewer than 2^32 work
items along an axis, so beyond that a kernel with capped or smaller grids, or several launches, have to do.  The library is
loaded in a process where the runtime's launch calls are recorded and not carried out: no device and no memory are needed."""
import json
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RECORDER = r"""
#include <stddef.h>
#include <stdint.h>
typedef struct { uint32_t x, y, z; } dims;
static dims grid, block;
uint32_t recorded[64][6];
int launches;
unsigned __hipPushCallConfiguration(dims g, dims b, size_t shared, void *stream) { grid = g; block = b; return 0; }
unsigned __hipPopCallConfiguration(dims *g, dims *b, size_t *shared, void **stream) { *g = grid; *b = block; *shared = 0; *stream = 0; return 0; }
int hipLaunchKernel(const void *f, dims g, dims b, void **args, size_t shared, void *stream) {
    uint32_t *at = recorded[launches++ % 64];
    at[0] = g.x, at[1] = g.y, at[2] = g.z, at[3] = b.x, at[4] = b.y, at[5] = b.z;
    return 0;
}
int hipGetLastError(void) { return 0; }
"""

CALLS = r"""
import ctypes, json, sys
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
L = ctypes.CDLL(sys.argv[2])
i32, i64, f32, p, sz = ctypes.c_int32, ctypes.c_int64, ctypes.c_float, ctypes.c_void_p, ctypes.c_size_t
L.tsx_batch_norm_f32.argtypes = [p, i64, i32, i64, p, p, f32, p, p]
L.tsx_batch_scale_f32.argtypes = [p, i64, i32, i64, p, p, p, p]
L.tsx_fused_batch_norm_f32.argtypes = [p, i64, i32, i64, p, p, p, p, f32, p, p]
L.tsx_pooling2d_f32.argtypes = [p, i64] + [i32] * 10 + [p, i32, i32, p]
for mode in ("f23", "f63"):
    getattr(L, "tsx_winograd_%s_workspace_bytes" % mode).restype = sz
    getattr(L, "tsx_conv2d_winograd_%s_nchw" % mode).argtypes = [p, p, p, f32, p, i32, f32, p, p, sz, p]
recorded = (ctypes.c_uint32 * 6 * 64).in_dll(recorder, "recorded")
launches = ctypes.c_int.in_dll(recorder, "launches")
at = 1 << 20                      # an address that nothing reads
out = []
for what, *extents in json.loads(sys.argv[3]):
    launches.value = 0
    if what in ("f23", "f63"):
        n, c, h, w, cout = extents
        geom = (i32 * 15)(n, c, h, w, cout, 3, 3, 1, 1, 1, 1, 1, 1, 1, 1)
        need = getattr(L, "tsx_winograd_%s_workspace_bytes" % what)(geom)
        rc = getattr(L, "tsx_conv2d_winograd_%s_nchw" % what)(geom, at, at, 0.0, None, 0, 0.0, at, at, need, None)
    else:
        planes, extent = extents
        if what == "batch_norm":
            rc = L.tsx_batch_norm_f32(at, planes, 1, extent, at, at, 1e-5, at, None)
        elif what == "batch_scale":
            rc = L.tsx_batch_scale_f32(at, planes, 1, extent, at, at, at, None)
        elif what == "fused_batch_norm":
            rc = L.tsx_fused_batch_norm_f32(at, planes, 1, extent, at, at, at, at, 1e-5, at, None)
        else:
            rc = L.tsx_pooling2d_f32(at, planes, extent, 4, what == "avg", 0, 0, extent, 4, 1, 1, 0, at, 1, 1, None)
    out.append([rc, [list(r) for r in recorded[:launches.value]]])
print(json.dumps(out))
"""

CASES = ([[what, planes, extent] for what in ("batch_norm", "batch_scale", "fused_batch_norm") for extent in (256, 1024)
          for planes in (1024, (1 << 26) - 4, (1 << 26) - 3, 1 << 26, (1 << 26) + 1, (1 << 28) + 5, (1 << 31) + 7)] +
         [[what, planes, extent] for what in ("max", "avg") for extent in (4, 56)
          for planes in (1, (1 << 28) - 16, (1 << 28) - 15, 1 << 28, (1 << 28) + 1, (1 << 32) - 256)] +
         [["f23", 1891, 3, 2175, 85, 1], ["f23", 4367, 4, 815, 151, 4], ["f23", 22285, 33, 55, 231, 2], ["f23", 8, 256, 28, 28, 256],
          ["f63", 57961, 3, 10, 1309, 5], ["f63", 30000, 1, 100, 100, 1], ["f63", 8, 256, 28, 28, 256]])


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    from tennis_amd.build import LIB_PATH
    where = tmp_path_factory.mktemp("recorder")
    source, so = where / "recorder.c", where / "librecorder.so"
    source.write_text(RECORDER)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(so), str(source)])
    run = subprocess.run([sys.executable, "-c", CALLS, str(so), LIB_PATH, json.dumps(CASES)], capture_output=True, text=True, cwd=ROOT)
    assert run.returncode == 0, run.stderr
    return json.loads(run.stdout)


@pytest.mark.parametrize("i", range(len(CASES)), ids=lambda i: "-".join(map(str, CASES[i])))
def test_launches_hold_their_work_items(recorded, i):
    rc, launches = recorded[i]
    assert rc == 0 and launches
    for gx, gy, gz, bx, by, bz in launches:
        assert gx * bx < 1 << 32 and gy * by < 1 << 32 and gz * bz < 1 << 32, (gx, bx)
    assert CASES[i][0] not in ("f23", "f63") or CASES[i][1] > 8 or len(launches) == 3       # transform, products, transform
