"""Runs library calls on the stand-in for the HIP runtime (cpp/host_hip.cpp), in a process of
their own: no GPU, kernels recorded and not run.  Freed memory is overwritten there
(MALLOC_PERTURB_), so that a copy whose host source did not live until the stream's wait shows."""
import ctypes as C
import json
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SRC = os.path.join(HERE, "cpp", "host_hip.cpp")
OUT = os.path.join(HERE, "cpp", "_build", "libhost_hip.so")


def build():
    if not os.path.exists(OUT) or os.path.getmtime(OUT) < os.path.getmtime(SRC):
        os.makedirs(os.path.dirname(OUT), exist_ok=True)
        tmp = f"{OUT}.{os.getpid()}"
        subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", SRC, "-o", tmp], check=True)
        os.replace(tmp, OUT)
    return OUT


def run(code, timeout=300):
    """The JSON value that `code` leaves in `result`; it has rt (Runtime), capi and numpy as np."""
    build()
    head = "from tests.host_hip import Runtime\nrt = Runtime()\nimport numpy as np\nfrom dmftpack_amd import capi\n"
    tail = "\nimport json\nprint('RESULT ' + json.dumps(result))\n"
    env = dict(os.environ, MALLOC_PERTURB_="165", PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(code) + tail], cwd=ROOT, env=env, capture_output=True,
                       text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return json.loads([x for x in r.stdout.splitlines() if x.startswith("RESULT ")][-1][7:])


class Runtime:
    def __init__(self):
        self.hip = C.CDLL(OUT, mode=C.RTLD_GLOBAL)  # before libdmftgpu.so, whose calls resolve here
        self.hip.host_hip_events.restype = C.c_char_p
        self.hip.host_hip_peak.restype = C.c_size_t
        self.hip.host_hip_alloc.restype = C.c_void_p
        self.hip.host_hip_alloc.argtypes = [C.c_size_t]
        from dmftpack_amd import capi
        self.lib, self.capi = capi.lib(), capi

    def reset(self):
        self.hip.host_hip_reset()

    def stale(self):
        return self.hip.host_hip_stale()

    def peak(self):
        return self.hip.host_hip_peak()

    def dev(self, array_or_bytes):
        """device buffer: a copy of an array, or zeros"""
        import numpy as np
        if isinstance(array_or_bytes, int):
            return C.c_void_p(self.hip.host_hip_alloc(array_or_bytes))
        a = np.ascontiguousarray(array_or_bytes)
        p = self.hip.host_hip_alloc(a.nbytes)
        C.memmove(p, a.ctypes.data, a.nbytes)
        return C.c_void_p(p)

    def handle(self, stream=None):
        h = C.c_void_p()
        assert self.lib.dmftgpu_create(C.byref(h), stream) == 0
        return h

    def check(self, h, rc):
        assert rc == 0, (rc, self.lib.dmftgpu_last_error(h))

    def events(self):
        return self.hip.host_hip_events().decode().splitlines()

    def launches(self):
        """[(kernel, grid, block)]"""
        out = []
        for e in self.events():
            if e.startswith("launch "):
                name, grid, block, _, _ = e[7:].rsplit(" | ", 4)
                out.append((name, tuple(map(int, grid.split())), tuple(map(int, block.split()))))
        return out

    def prepare(self, h, n, nc, nk, n_freq, beta=40.0, high_freq=2, moments=None):
        """binds a lattice of zeros (the kernels do not run); the buffers live on"""
        import numpy as np
        lat = self.capi.Lattice(n, nc, 1, nk, nk, n_freq, high_freq, beta)
        mom = np.zeros((4, nc, nc), np.complex128) if moments is None else moments
        self.check(h, self.lib.dmftgpu_prepare(h, C.byref(lat), self.dev(16 * nk * n * n), self.dev(mom)))
        return lat
