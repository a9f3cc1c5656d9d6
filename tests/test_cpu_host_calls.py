"""Host side of the library's calls, on the stand-in for the HIP runtime (host_hip.py): which
kernels a call launches with which grids, how much scratch it asks for, and that the host
source of every asynchronous copy lives until the stream is waited for."""
import pytest

from tests import host_hip

FT = """
import ctypes as C
h = rt.handle()
d, nf, nt = 4, 40, 64
f, g = rt.dev(16 * nf * d * d), rt.dev(16 * (nt + 1) * d * d)
mom = rt.dev(np.stack([np.zeros((d, d)), np.eye(d), 0.1 * np.eye(d), np.eye(d)]).astype(np.complex128))
"""


@pytest.mark.parametrize("call", [
    "rt.lib.dmftgpu_ft_w2tau(h, d, nf, nt, 20.0, f, mom, g, None)",
    "rt.lib.dmftgpu_ft_w2tau_points(h, d, nf, 20.0, f, mom, 3, (C.c_double * 3)(0.1, 0.2, 0.3), g)",
])
def test_tail_copy_source_outlives_the_copy(call):
    assert host_hip.run(FT + f"rt.reset()\nrt.check(h, {call})\nresult = rt.stale()") == 0
