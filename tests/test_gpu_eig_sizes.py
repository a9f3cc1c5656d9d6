"""Batched Hermitian eigensolver around the switch between its LDS and 32-lane forms (m = 26):
eigenvalues against numpy, orthogonality and reconstruction, degenerate and diagonal spectra.
Bounds: Jacobi stops at off-diagonal norm 1e-17 |A| after at most ~10 sweeps of m - 1 rounds, each
a few roundings: 1e-13 |A| covers m = 32 on all of them (the bound of the smaller sizes)."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def matrices(n, kind):
    rng = np.random.default_rng(n)
    if kind == "random":
        X = rng.normal(size=(5, n, n)) + 1j * rng.normal(size=(5, n, n))
        return 0.5 * (X + X.conj().transpose(0, 2, 1))
    if kind == "degenerate":
        q, _ = np.linalg.qr(rng.normal(size=(5, n, n)) + 1j * rng.normal(size=(5, n, n)))
        return (q * np.repeat(np.arange(4.0), n)[:n * 4:4][None, None, :]) @ q.conj().transpose(0, 2, 1)
    return np.stack([np.diag(rng.normal(size=n)).astype(complex) for _ in range(5)])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [17, 25, 26, 27, 31, 32])
@pytest.mark.parametrize("kind", ["random", "degenerate", "diagonal"])
def test_static_eig_sizes(G, n, kind):
    Hk = matrices(n, kind)
    Hk = 0.5 * (Hk + Hk.conj().transpose(0, 2, 1))
    sig, mom = L.pole_sigma(2, 4, 10.0, n)
    mom[0] = np.array([[0.3, 0.1 - 0.2j], [0.1 + 0.2j, -0.4]])
    lat = G.LatticeGF(Hk, 2, 4, 10.0, mom)
    ev, U = lat.static_eig()
    lat.close()
    H = Hk.copy()
    H[:, :2, :2] += mom[0]
    scale = np.linalg.norm(H, axis=(1, 2)).max()
    assert np.abs(ev - np.linalg.eigvalsh(H)).max() <= 1e-13 * scale
    assert np.abs(U.conj().transpose(0, 2, 1) @ U - np.eye(n)).max() <= 1e-13
    assert np.abs(U * ev[:, None, :] @ U.conj().transpose(0, 2, 1) - H).max() <= 1e-13 * scale


@pytest.mark.gpu
@pytest.mark.parametrize("n,nk", [(26, 2000), (27, 1600), (28, 1025), (29, 1300)])
def test_many_matrices(G, n, nk):
    """counts at which these sizes take the 32-lane slots"""
    rng = np.random.default_rng(n)
    X = rng.normal(size=(nk, n, n)) + 1j * rng.normal(size=(nk, n, n))
    H = 0.5 * (X + X.conj().transpose(0, 2, 1))
    sig, mom = L.pole_sigma(2, 4, 10.0, n)
    mom[0] = 0.0
    lat = G.LatticeGF(H, 2, 4, 10.0, mom)
    ev, U = lat.static_eig()
    lat.close()
    scale = np.linalg.norm(H, axis=(1, 2)).max()
    assert np.abs(ev - np.linalg.eigvalsh(H)).max() <= 1e-13 * scale
    assert np.abs(U * ev[:, None, :] @ U.conj().transpose(0, 2, 1) - H).max() <= 1e-13 * scale
