"""Contexts on two devices used from threads whose current device is the other
one: everything a context makes at its first evaluation belongs to its own
device, and the thread's current device stays what it was.  Runs on the CPU over
a stand-in for the HIP runtime (tests/cpp/two_devices.cpp), which checks every
copy, memset and event against the device of its stream."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import ctypes as C, sys
hip = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
import threading
import numpy as np
import a2c_amd as A

n = 10000  # of each species: a state of several transfer parts
rng = np.random.default_rng(0)
X = rng.uniform(0.0, 100.0, (2 * n, 4))
X[:, 3] = 0.1
X, x = X.reshape(-1), rng.uniform(0.0, 0.6, n)
box = (100.0, 100.0, 100.0)


def current():
    d = C.c_int(-1)
    hip.hipGetDevice(C.byref(d))
    return d.value


def on(device, fn):
    err = []

    def body():
        try:
            hip.hipSetDevice(device)
            fn()
            assert current() == device
        except BaseException as e:
            err.append(e)

    t = threading.Thread(target=body)
    t.start()
    t.join()
    if err:
        raise err[0]


def callback(fe):
    fe.formFunctionAndGradient(X)


for precision in ("fp64", "mixed"):
    ctx = []
    for device in (0, 1):
        fe = A.FreeEntropy(n, n, box, (0, 0, 0), T=400.0, precision=precision, device=device)
        fe.set_occupancy(x)
        fe.findNeighbors(X)
        ctx.append(fe)
    for device in (0, 1):
        on(1 - device, lambda: callback(ctx[device]))
        on(device, lambda: callback(ctx[device]))
b = A.Batch(precision="fp64", max_lattices=1, device=1)
slot = b.add(X, x, n, n, box, (0, 0, 0), T=400.0)
on(0, lambda: (b.eval([slot]), b.get_state(slot)))
bad = hip.two_devices_violations()
print("violations", bad)
sys.stdout.flush()
import os
os._exit(1 if bad else 0)
"""


def test_first_evaluation_from_another_current_device(tmp_path):
    shim = str(tmp_path / "two_devices.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "two_devices.cpp"), "-o", shim], check=True)
    r = subprocess.run([sys.executable, "-c", PROGRAM, shim], cwd=ROOT, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
