"""Error paths of the entry points on a stand-in HIP runtime (host_hip.cpp,
no GPU): an allocation or a kernel launch fails, and the call reports it,
waits for the copies it has queued from memory that goes away with it, and
leaves nothing half made for the next call.  And which kernels the transforms
of a shape launch."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
hip = C.CDLL({so!r}, mode=C.RTLD_GLOBAL)
hip.host_hip_calls.restype = C.c_char_p
sys.path[:0] = [{root!r}, {here!r}]
import numpy as np
import haagenti_amd as H
ctx = H.HipContext(0)
def calls():
    return hip.host_hip_calls().decode().split("\\n")[:-1]
def launches(name):
    return [c for c in calls() if name in c]
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libhost_hip.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "host_hip.cpp")], check=True)

    def run(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE.format(so=so, root=os.path.dirname(HERE), here=HERE) + code],
                           capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stderr[-3000:]
    return run


@pytest.mark.parametrize("rows,cols,route,kernel", [
    (8, 12, "auto", "lines_tables_kernel"),
    (64, 17920, "auto", "fft_tables_kernel"),
    (64, 24, "dense", "basis"),
])
def test_tables_of_a_failed_launch_are_not_kept(host, rows, cols, route, kernel):
    host(f"""
x = np.zeros(2 * {rows * cols} + 4, np.float32)
at = (x.ctypes.data + 15) & ~15
to = at + 4 * {rows * cols}
for n in (1, 2):                        # the tables of the first and of the second side fail
    ctx = H.HipContext(0)
    ctx.set_dct_route({route!r})
    hip.host_hip_fail({kernel!r}.encode(), n)
    rc = H._lib.hh_dct_2d(ctx.handle, at, {rows}, {cols}, to, None)
    assert rc != H.OK and launches({kernel!r})[n - 1:] == launches("failed"), calls()
    hip.host_hip_fail(b"", 0)
    rc = H._lib.hh_dct_2d(ctx.handle, at, {rows}, {cols}, to, None)
    assert rc == H.OK and len(launches({kernel!r})) == 3 - n, calls()
""")


@pytest.mark.parametrize("rows,cols,route,fail", [
    (64, 48, "auto", "row_counts_kernel"),      # the fragments read by the row pass
    (64, 48, "auto", "lines_tables_kernel"),
    (512, 1024, "dense", "amax_f16_kernel"),    # the even / odd split of the bases
    (64, 24, "dense", "basis"),                 # the dense products
    (64, 24, "coefficients", "scatter"),        # no transform
])
def test_a_failed_decode_waits_for_its_copies(host, rows, cols, route, fail):
    host(f"""
from test_oracle_hct3 import container, random_fragment
data = container([random_fragment(np.random.default_rng(1), {rows * cols}, 0.3)])
out = np.zeros({rows * cols} + 4, np.float32)
at = (out.ctypes.data + 15) & ~15
hip.host_hip_fail({fail!r}.encode(), 1)
if {route!r} == "coefficients":
    rc = H._lib.hh_hct3_coefficients(ctx.handle, data, len(data), {rows * cols}, at, None)
else:
    ctx.set_dct_route({route!r})
    arr, rank = H._shape_arr([{rows}, {cols}])
    rc = H._lib.hh_hct3_decompress(ctx.handle, data, len(data), arr, rank, H.F32, at, None)
c = calls()
assert rc != H.OK and launches("failed"), c
assert "copy" in c and "synchronize" in c[len(c) - c[::-1].index("copy"):], c
""")


def test_routes_of_the_transforms(host):
    # the two passes up to 16384, rows and transposes above, the dense
    # products for the lengths neither takes
    host("""
from test_gpu_dct_lines import test_transforms_vs_f64 as lines
from test_gpu_dct_long import FRAGMENTS, SHAPES
two, rows, dense = "12lines_kernel", "dct_fft_rows_kernel", "dct_gemm"
shapes = [(s, two) for m in lines.pytestmark if m.name == "parametrize" for s in m.args[1]]
shapes += [(s, rows) for s in SHAPES + FRAGMENTS] + [((64, 131), dense), ((17000, 64), dense)]
for (r, c), kernel in shapes:
    hip.host_hip_fail(b"", 0)
    assert H._lib.hh_dct_2d(ctx.handle, 16, r, c, 32, None) == H.OK
    assert H._lib.hh_idct_2d(ctx.handle, 16, r, c, H.F32, 32, None) == H.OK
    got = {k for k in (two, rows, dense) if launches(k)}
    assert got == {kernel}, (r, c, calls())
from test_oracle_hct3 import container, random_fragment
for (r, c), scatter in zip(FRAGMENTS, (False, False, True, True)):
    data = container([random_fragment(np.random.default_rng(1), r * c, 0.01)])
    out = np.zeros(r * c + 4, np.float32)
    arr, rank = H._shape_arr([r, c])
    hip.host_hip_fail(b"", 0)
    assert H._lib.hh_hct3_decompress(ctx.handle, data, len(data), arr, rank, H.F32, (out.ctypes.data + 15) & ~15,
                                     None) == H.OK
    assert launches(rows) and bool(launches("hct3_scatter_kernel")) == scatter, (r, c, calls())
""")
