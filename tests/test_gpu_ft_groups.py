"""Transforms whose partial sums do not all fit at once (d = 32, eight input tiles in four
groups), against an FFT (tau -> iw) and the oracle (iw -> tau) on a few entries; 1e-12 of the
largest entry as in test_gpu_ft_grid."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_ft_grid import propagator, rel

D = 32


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


@pytest.mark.gpu
def test_tau2w_groups(G):
    import torch
    nf, nt, beta = 8192, 16384, 20.0
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    g = torch.randn((nt + 1, D, D, 2), generator=gen, device="cuda", dtype=torch.float64)
    g = torch.view_as_complex(g).contiguous()
    fw = torch.empty((nf, D, D), dtype=torch.complex128, device="cuda")
    h = G.Handle()
    h.check(h.lib.dmftgpu_ft_tau2w(h.h, D, nf, nt, beta, C.c_void_p(g.data_ptr()), C.c_void_p(fw.data_ptr()), None))
    pick = [0, 1, 31, 500, 1023]
    x = g.reshape(nt + 1, -1)[:, pick].cpu().numpy()
    got = fw.reshape(nf, -1)[:, pick].cpu().numpy()
    t = np.arange(nt)
    th = (2 * np.arange(nf) + 1) * np.pi / nt
    s = nt * np.fft.ifft(np.where(t[:, None] > 0, x[:-1], 0) * np.exp(1j * np.pi * t / nt)[:, None], axis=0)[:nf]
    # int_0^1 (1-u) e^{i th u} du by 64-point Gauss-Legendre (th < pi)
    u, w = np.polynomial.legendre.leggauss(64)
    u, w = 0.5 * (u + 1), 0.5 * w
    al = (np.exp(1j * th[:, None] * u) * (1 - u) * w).sum(1)[:, None]
    ref = (beta / nt) * ((np.sinc(th / (2 * np.pi)) ** 2)[:, None] * s + al * x[0] - al.conj() * x[-1])
    assert rel(got, ref) <= 1e-12
    h.close()


@pytest.mark.gpu
def test_w2tau_groups(G):
    nf, nt, beta = 16384, 8192, 20.0
    f, mom = propagator(D, nf, beta, 11)
    h = G.Handle()
    gt, patched = h.fourier_transform(f, mom, beta, nt)
    assert not patched
    for j in (2731, nt):
        assert rel(gt[j], O.ft_tau(f, mom, beta, j * beta / nt)) <= 1e-12
    h.close()
