"""A boundary-system call that ends in an error leaves no inverse behind that a
later call would take for its own: rocblas_set_stream, which stands between the
new system and its factors, reports an error once (a host function of its name
is found before the library's), and the next call has to solve the new system."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
int fail_next = 0;
int (*real)(void*, void*) = 0;
int rocblas_set_stream(void* handle, void* stream) {
    if (fail_next) {
        fail_next = 0;
        return 6;   /* rocblas_status_internal_error */
    }
    return real(handle, stream);
}
"""

RUN = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import vvflow_amd as V
V.lib()
path = [q.split()[-1] for q in open("/proc/self/maps") if "/librocblas.so" in q][0]
real = ctypes.CDLL(path).rocblas_set_stream
ctypes.c_void_p.in_dll(shim, "real").value = ctypes.cast(real, ctypes.c_void_p).value

r = np.random.default_rng(3)
v = np.zeros((300, 6))
v[:, 0], v[:, 1] = r.uniform(-1, 1, 300), np.where(r.random(300) < 0.5, 1, -1) * r.uniform(0.5, 1.0, 300)
v[:, 2] = r.normal(size=300) * 1e-3


def solve(ctx, height):
    print("case slae error ellipse", height, flush=True)
    segs = np.ascontiguousarray(V.segments_from_corners(V.gen_cylinder(0.4, 40) * [1.0, height]), dtype=V.SEG_DTYPE)
    b = np.zeros(1, dtype=V.BODY_DTYPE)
    b["nseg"] = 40
    ctx.set_params(re=600.0, dt=0.005, time=0.5)
    ctx.upload_bodies(segs, b)
    ctx.upload(v)
    ctx.tree_build(8, 0.05, 10.0)
    ctx.epsilon(False)
    ctx.calc_circulation((1.0, 0.2))
    return ctx.download_bodies()[0]["g"].copy()


ctx, new = V.Context(0), V.Context(0)
solve(ctx, 1.0)
ctypes.c_int.in_dll(shim, "fail_next").value = 1
try:
    solve(ctx, 0.5)
    sys.exit("the call did not report the error")
except V.VVHDError as e:
    print(e, flush=True)
got, want = solve(ctx, 0.5), solve(new, 0.5)
# the same factors or inverse of one 40 x 40 system of condition number ~100
err = np.linalg.norm(got - want) / np.linalg.norm(want)
print("difference", err, flush=True)
sys.exit(0 if err < 1e-12 else "solved with the inverse of another system")
"""


def test_no_inverse_after_an_error(tmp_path):
    src, lib = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src)], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-u", "-c", RUN, str(lib)], cwd=root, capture_output=True, text=True,
                       timeout=100)
    print(p.stdout, p.stderr, flush=True)
    assert p.returncode == 0, p.stderr
