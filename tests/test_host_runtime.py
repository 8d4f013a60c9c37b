"""What the host code asks of the runtime, on a stub of two host-memory devices (cpp/hip_host_stub.c) in a
process of its own: buffers that a context allocates after its creation (bins, lists, frames) land on the
context's own device, whichever is current, and the caller's current device stays; a batch's calls launch as
many kernels for many colonies as for few."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DEVICES = """
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
print("ok")
"""

LAUNCHES = """
import ctypes
hip = ctypes.CDLL("libamdhip64.so.7")
from cil_cuda_amd import abi, configs
from cil_cuda_amd.colony import HipBatch, HipMD

def launches(n):
    mds = []
    for k in range(n):
        p, box, col = configs.binary_2d_fene(n_cells=30, seed=k)
        assert p.noise == abi.NOISE_CELL_WIENER
        md = HipMD(p, box, [sp["capacity"] for sp in col.species])
        md.upload(col)
        md.forces(want=False)
        mds.append(md)
    batch = HipBatch(mds)
    ts = batch.step(1, [0] * n)  # the members' own passes drew their noise in place: stored once
    before = hip.stub_launches()
    batch.step(1, ts)
    count = hip.stub_launches() - before
    mds[0].forces(want=False)  # a pass of its own: stored again for this member
    before = hip.stub_launches()
    batch.step(1, [t + 1 for t in ts])
    assert hip.stub_launches() - before == count + 1
    batch.close()
    return count

assert launches(2) == launches(9)
print("ok")
"""


def _run(program, tmp_path):
    lib = tmp_path / "libamdhip64.so.7"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-Wl,-soname,libamdhip64.so.7", "-o", str(lib),
                    os.path.join(ROOT, "tests", "cpp", "hip_host_stub.c")], check=True)
    env = dict(os.environ, LD_LIBRARY_PATH=str(tmp_path), PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", program], cwd=ROOT, env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr


def test_late_buffers_land_on_the_contexts_device(tmp_path):
    _run(DEVICES, tmp_path)


def test_batch_calls_launch_the_same_for_any_number_of_colonies(tmp_path):
    _run(LAUNCHES, tmp_path)
