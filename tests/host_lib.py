"""Builds a host-only library from tests/host/<name>.hip: the device sources' host code, with no device
code and no GPU."""
import ctypes
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def build(name, folder):
    obj, so = os.path.join(folder, name + ".o"), os.path.join(folder, name + ".so")
    host = os.path.join(ROOT, "sparse-operator-graph-lu_amd", "build", "libsogl_host.so")
    rocm = os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "lib")
    for cmd in ([HIPCC, "-std=c++17", "-O1", "-fPIC", "--offload-arch=gfx950", "--offload-host-only", "-fuse-cuid=none",
                 "-I", os.path.join(ROOT, "include"), "-c", os.path.join(ROOT, "tests", "host", name + ".hip"), "-o", obj],
                ["g++", "-shared", "-Wl,-Bsymbolic", "-o", so, obj, host, f"-L{rocm}", "-lamdhip64", f"-Wl,-rpath,{rocm}",
                 f"-Wl,-rpath,{os.path.dirname(host)}"]):
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
    return ctypes.CDLL(so)
