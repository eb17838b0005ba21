"""Runs a function of a test module in a process of its own in which libmeshstage.so works on hip_host/hip_host.cpp: memory of a
stated size on the host, launches that are noted and not run."""
import ctypes
import functools
import importlib
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "hip_host", "hip_host.cpp")


@functools.lru_cache(None)
def _library():
    d = tempfile.TemporaryDirectory()
    lib = os.path.join(d.name, "libhip_host.so")
    cmd = [os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-Wall", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", SRC, "-o", lib]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hip_host build failed:\n%s\n%s" % (" ".join(cmd), r.stderr))
    return lib, d


def call(fn, **kw):
    """fn(host, **kw) in a child process; its result, through JSON."""
    lib, _ = _library()
    r = subprocess.run([sys.executable, os.path.abspath(__file__), lib, fn.__module__, fn.__name__, json.dumps(kw)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-3000:]
    return json.loads(r.stdout.splitlines()[-1])


class Host:
    def __init__(self, lib):
        self.lib = ctypes.CDLL(lib, mode=ctypes.RTLD_GLOBAL)
        self.lib.host_launches.restype = ctypes.c_char_p
        self.lib.host_used.restype = ctypes.c_size_t

    def memory(self, total):
        self.lib.host_memory(ctypes.c_size_t(total))

    def others(self, n):
        self.lib.host_others(ctypes.c_longlong(n))

    def take_after_info(self, n):
        self.lib.host_take_after_info(ctypes.c_longlong(n))

    @property
    def used(self):
        return self.lib.host_used()

    def launches(self):
        """[(name, (grid x, y, z), threads)] since the last call; name as in gemm_f16_kernel<1,4,3> (types left out)."""
        out = []
        for line in self.lib.host_launches().decode().splitlines():
            name, *dims = line.split()
            x, y, z, n = map(int, dims)
            out.append((kernel_name(name), (x, y, z), n))
        return out


def kernel_name(mangled):
    """_ZN4mesh15gemm_f16_kernelILNS_7TileOutE1ELi4ELi3EEEv... -> gemm_f16_kernel<1,4,3>"""
    import re
    m = re.match(r"_ZN4mesh(?:12_GLOBAL__N_1|5f16sk)?(\d+)", mangled)
    if not m:
        return mangled
    n = int(m.group(1))
    name, rest = mangled[m.end():m.end() + n], mangled[m.end() + n:]
    if not rest.startswith("I"):
        return name
    args = re.match(r"I((?:L(?:NS_\d+\w+?E|[a-z])\d+E)*)", rest).group(1)
    return "%s<%s>" % (name, ",".join(re.findall(r"L(?:NS_\d+\w+?E|[a-z])(\d+)E", args)))


if __name__ == "__main__":
    sys.path.insert(0, HERE)
    host = Host(sys.argv[1])                # (before anything loads libmeshstage.so)
    fn = getattr(importlib.import_module(sys.argv[2]), sys.argv[3])
    print(json.dumps(fn(host, **json.loads(sys.argv[4]))), flush=True)
