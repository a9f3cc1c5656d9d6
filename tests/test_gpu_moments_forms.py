"""Tail moments on both sides of the line between one moment and all moments a thread
(40960 window and pair fits), against the oracle: both sum in its order, so the windows are
equal and the moments agree to 1e-12 as in test_gpu_ft."""
import numpy as np
import pytest

from oracle import oracle as O
from tests.test_gpu_ft import rel, three_pole_g


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


@pytest.mark.gpu
@pytest.mark.parametrize("d,nf", [(13, 449), (13, 451), (16, 302), (32, 100)])
@pytest.mark.parametrize("green", [False, True])
def test_moments(G, d, nf, green):
    fw = three_pole_g(d, nf, 20.0, 7 * d + nf)
    if not green:
        fw = 0.8 * fw + 0.3 * np.eye(d)
    h = G.Handle()
    got, win = h.get_asymto_moments(fw, 20.0, green, return_windows=True)
    ref, rwin = O.asymto_moments(fw, 20.0, green, return_windows=True)
    assert list(win) == list(rwin)
    assert rel(got, ref) <= 1e-12
    h.close()
