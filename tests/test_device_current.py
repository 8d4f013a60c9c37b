"""Buffers that a context allocates after its creation (bins, lists, frames) land on the context's own
device, whichever is current, and the caller's current device stays.  Runs the host code on a runtime of two
host-memory devices (cpp/hip_host_stub.c) in a process of its own."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import ctypes
hip = ctypes.CDLL("libamdhip64.so.7")
from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import HipMD

def current():
    d = ctypes.c_int(-1)
    hip.hipGetDevice(ctypes.byref(d))
    return d.value

p, box, col = configs.bulk_3d_mixed(n=4000, seed=5)
hip.hipSetDevice(1)
md = HipMD(p, box, [2 * sp["capacity"] for sp in col.species])
assert hip.stub_allocs(0) == 0 and hip.stub_allocs(1) > 0
hip.hipSetDevice(0)
md.upload(col)
for what, call in (("more bins", lambda: md.set_tuning(4, 256)),
                   ("lists", lambda: md.set_neighbour_list(True, 0.4, 64, inner_skin=0.1)),
                   ("longer lists", lambda: md.set_neighbour_list(True, 0.4, 256, inner_skin=0.1)),
                   ("frame", lambda: md.download(col.copy()))):
    before = hip.stub_allocs(1)
    call()
    assert hip.stub_allocs(0) == 0, what
    assert hip.stub_allocs(1) > before, what
    assert current() == 0, what
md.close()
print("two devices ok")
"""


def test_late_buffers_land_on_the_contexts_device(tmp_path):
    lib = tmp_path / "libamdhip64.so.7"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-Wl,-soname,libamdhip64.so.7", "-o", str(lib),
                    os.path.join(ROOT, "tests", "cpp", "hip_host_stub.c")], check=True)
    env = dict(os.environ, LD_LIBRARY_PATH=str(tmp_path), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "two devices ok" in r.stdout, r.stdout + r.stderr
