"""libt0mi's host side on a machine without a GPU: fake_hip.cpp in the HIP runtime's place, in a process of
its own (the real runtime may be loaded in this one)."""
import json
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIP_INCLUDE = "/opt/rocm/include"

_PRELUDE = """
import ctypes, json, sys
sys.modules["torch"] = None  # its own HIP runtime stays out of this process
hip = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)
hip.fake_launches.restype = ctypes.c_char_p
hip.fake_set_malloc_limit.argtypes = [ctypes.c_size_t]
hip.fake_allocated.restype = ctypes.c_size_t
sys.path[:0] = [{root!r}, {pkg!r}]
import t0mi
rt = t0mi.Runtime(0)
hip.fake_launches()
X, B, Y, BIAS = 1 << 40, 2 << 40, 3 << 40, 4 << 40  # operands far from each other

def launches():
    "The launches since the last call: [kernel name, grid x, y, z, block], oldest first."
    return [[f if i == 0 else int(f) for i, f in enumerate(l.split(" "))]
            for l in hip.fake_launches().decode().splitlines()]

def names(f, *args, **kw):
    "The kernels that one call launches, without their template arguments."
    hip.fake_launches()
    f(*args, **kw)
    return [l[0].split("<")[0] for l in launches()]

def done(value):
    print(json.dumps(value))
"""


@pytest.fixture(scope="session")
def host(tmp_path_factory):
    """host(code): runs `code` with the prelude's names and returns what it passed to done()."""
    if shutil.which("g++") is None or not os.path.isdir(HIP_INCLUDE):
        pytest.skip("needs g++ and the HIP headers")
    if not os.path.exists(os.path.join(ROOT, "rust-gpu_amd", "t0mi", "libt0mi.so")):
        import __graft_entry__
        __graft_entry__.build()
    so = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-Wno-unused-result", "-shared", "-fPIC",
                    "-D__HIP_PLATFORM_AMD__", "-isystem", HIP_INCLUDE, "-o", so, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)

    def run(code):
        prelude = _PRELUDE.format(so=so, root=ROOT, pkg=os.path.join(ROOT, "rust-gpu_amd"))
        r = subprocess.run([sys.executable, "-c", prelude + code], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, r.stderr[-4000:]
        return json.loads(r.stdout.strip().splitlines()[-1])

    return run
