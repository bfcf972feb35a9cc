"""Programs of tests/host: the library's sources compiled for the host only,
linked with host memory in the place of the GPU runtime (tests/host/hip_host.h)."""

import functools
import os
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

import helpers as H

HERE = os.path.join(H.REPO, "tests", "host")
CSRC = os.path.join(H.REPO, "rast-3dmhd_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "--offload-host-only", "-fuse-cuid=none", "-O1", "-std=c++17", "-fPIC", "-pthread"]


def _run(cmd, stdin=None):
    r = subprocess.run(cmd, input=stdin, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, " ".join(cmd) + "\n" + r.stdout + r.stderr
    return r.stdout


@functools.lru_cache(None)
def _objects():
    """(directory, object files) of the library, compiled once a session."""
    tmp = tempfile.TemporaryDirectory(prefix="rast3dmhd_host_")
    src = sorted(f for f in os.listdir(CSRC) if f.startswith("mhd_") and f.endswith(".hip"))
    obj = [os.path.join(tmp.name, f[:-4] + ".o") for f in src]
    with ThreadPoolExecutor(4) as ex:
        list(ex.map(lambda so: _run([HIPCC, *FLAGS, "-c", os.path.join(CSRC, so[0]), "-o", so[1]]), zip(src, obj)))
    return tmp, obj


@functools.lru_cache(None)
def _program(name):
    tmp, obj = _objects()
    main, exe = os.path.join(tmp.name, name + "_main.o"), os.path.join(tmp.name, name)
    _run([HIPCC, *FLAGS, "-x", "hip", "-c", os.path.join(HERE, name + ".cpp"), "-o", main])
    # (every object holds the same empty module id)
    _run(["g++", "-pthread", "-rdynamic", "-Wl,-z,muldefs", main, *obj, "-ldl", "-o", exe])
    return exe


def run(name, *args, stdin=None):
    """Builds tests/host/<name>.cpp and runs it; its output, or the test fails with it."""
    return _run([_program(name), *args], stdin)
