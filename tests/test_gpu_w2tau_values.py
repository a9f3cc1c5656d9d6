"""iw -> tau, the whole grid against the oracle with its causality patch, in cases that must not be
skipped where the patch acts: grid sizes around the chirp-z tiles, one-point grids, and matrices up to
d = 32; 1e-12 of the largest entry as in test_gpu_ft, the patch flag equal."""
import os

import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_ft_grid import SIZES, propagator, rel

THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


@pytest.mark.gpu
@pytest.mark.parametrize("d,nf,nt", [(1, *s) for s in SIZES] + [(5, *s) for s in SIZES] +
                         [(9, 40, 33), (16, 33, 20), (17, 30, 21), (32, 24, 16)])
def test_whole_grid(G, d, nf, nt):
    beta = 20.0
    f, mom = propagator(d, nf, beta, 100 * nf + nt)
    h = G.Handle()
    gt, patched = h.fourier_transform(f, mom, beta, nt)
    ref, rp = O.ft_w2tau(f, mom, beta, nt, nthreads=THREADS)
    print(f"d={d} nf={nf} nt={nt}: patched {patched}", flush=True)
    assert patched == rp
    assert rel(gt, ref) <= 1e-12
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("d", [1, 4, 9, 16, 17, 32])
def test_patch_acts(G, d):
    """a spike at one frequency adds 40/beta cos(w tau) I, which at some tau outweighs -G (at most I):
    every eigenvalue is positive there and the patch acts on both sides"""
    nf, nt, beta = 24, 40, 20.0
    f, mom = propagator(d, nf, beta, 5)
    f = f.copy()
    f[3] += 20.0 * np.eye(d)
    h = G.Handle()
    gt, patched = h.fourier_transform(f, mom, beta, nt)
    ref, rp = O.ft_w2tau(f, mom, beta, nt, nthreads=THREADS)
    assert patched == rp == 1
    assert rel(gt, ref) <= 1e-12
    h.close()
