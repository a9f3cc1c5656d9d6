"""The uniform-grid transforms (chirp-z, csrc/ft_czt.hip) against the dense sums with exact
phases, at the edges of their 2048-point tiles, prime and composite tau counts, fewer tau
points than frequencies, and one-point grids.  Bound: with L = log2(4096) = 12 butterfly levels
per FFT and two FFTs, each level adding at most a few rounding errors relative to the 2-norm,
errors stay below 100 eps of the sum of absolute values; 1e-12 of the largest entry (the
bound of the transforms against the oracle) covers that for these sums."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L
from oracle import oracle as O

SIZES = [(1, 1), (1, 7), (5, 1), (17, 16), (300, 64), (2047, 2048), (2048, 2047), (2049, 2049), (130, 4099),
         (4100, 263)]


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


def propagator(d, nf, beta, seed):
    """metallic G(iw) (poles within 2/beta of zero) and its moments"""
    rng = np.random.default_rng(seed)
    B = rng.normal(size=(3, d, d)) + 1j * rng.normal(size=(3, d, d))
    A = B @ B.conj().transpose(0, 2, 1) + 0.3 * np.eye(d)
    w, v = np.linalg.eigh(A.sum(0))
    s = v @ np.diag(w ** -0.5) @ v.conj().T
    A = s @ A @ s
    b = np.array([1.0 / beta, -0.8, 1.3])
    iw = 1j * L.matsubara(nf, beta)
    f = sum(A[p][None] / (iw[:, None, None] - b[p]) for p in range(3))
    mom = np.stack([np.zeros((d, d)), A.sum(0), np.einsum("p,pij->ij", b, A), np.einsum("p,pij->ij", b * b, A)])
    return f, mom


def phases(nf, nt):
    """e^{i w_n tau_j}, exact multiples of pi/nt"""
    m = (2 * np.arange(nf)[:, None] + 1) * np.arange(nt + 1)[None] % (2 * nt)
    return np.exp(1j * np.pi * m / nt)


@pytest.mark.gpu
@pytest.mark.parametrize("nf,nt", SIZES)
@pytest.mark.parametrize("d", [1, 5])
def test_w2tau(G, nf, nt, d):
    beta = 20.0
    f, mom = propagator(d, nf, beta, 100 * nf + nt)
    h = G.Handle()
    gt, patched = h.fourier_transform(f, mom, beta, nt)
    taus = np.unique(np.r_[0, nt // 3, nt // 2, nt - 1, nt]) * (beta / nt)
    js = np.unique(np.r_[0, nt // 3, nt // 2, nt - 1, nt])
    ref = np.stack([O.ft_tau(f, mom, beta, t) for t in taus])
    if not patched:  # few frequencies can leave G(tau) indefinite: the patch then acts on both sides
        assert rel(gt[js], ref) <= 1e-12
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nf,nt", SIZES)
@pytest.mark.parametrize("d", [2, 6])
def test_tau2w(G, nf, nt, d):
    beta = 20.0
    rng = np.random.default_rng(nf + nt)
    g = rng.normal(size=(nt + 1, d, d)) + 1j * rng.normal(size=(nt + 1, d, d))
    E = phases(nf, nt)
    th = (2 * np.arange(nf) + 1) * np.pi / nt
    # int_0^1 u^k e^{i theta u} du by Gauss-Legendre, 64 points (theta < 64)
    x, w = np.polynomial.legendre.leggauss(64)
    u, w = 0.5 * (x + 1), 0.5 * w
    if th[-1] < 60:
        e = np.exp(1j * th[:, None] * u)
        gam, one = (e * u * w).sum(1), (e * w).sum(1)
    else:
        e1 = np.exp(1j * th)
        gam = np.where(th > 1, (e1 * (1j * th - 1) + 1) / (1j * th) ** 2, (np.exp(1j * th[:, None] * u) * u * w).sum(1))
        one = (e1 - 1) / (1j * th)
    ref = (beta / nt) * (np.einsum("nt,tij->nij", E[:, :-1] * (one - gam)[:, None], g[:-1])
                         + np.einsum("nt,tij->nij", E[:, :-1] * gam[:, None], g[1:]))
    h = G.Handle()
    fw, viol = h.ft_t_to_w(g, beta, nf)
    assert rel(fw, ref) <= 1e-12
    anti = (fw - fw.conj().transpose(0, 2, 1)) / 2j
    assert viol == int((np.linalg.eigvalsh(anti)[:, -1] > 0).sum())
    h.close()


@pytest.mark.gpu
def test_definiteness_shortcut_keeps_the_patch(G):
    """one indefinite G(tau): the eigenvalue path decides as before (oracle's whole transform)"""
    d, nf, nt, beta = 3, 24, 40, 20.0
    f, mom = propagator(d, nf, beta, 5)
    f = f.copy()
    f[3] += 2.0 * np.eye(d)  # a spike that drives G(tau) through zero
    h = G.Handle()
    gt, patched = h.fourier_transform(f, mom, beta, nt)
    ref, rp = O.ft_w2tau(f, mom, beta, nt)
    assert patched == rp == 1
    assert rel(gt, ref) <= 1e-12
    h.close()


@pytest.mark.gpu
def test_tables_follow_the_grid(G):
    """one handle, alternating tau counts: the kept tables belong to the last one"""
    beta = 20.0
    h = G.Handle()
    f, mom = propagator(2, 50, beta, 9)
    first, _ = h.fourier_transform(f, mom, beta, 64)
    h.fourier_transform(f, mom, beta, 77)
    again, _ = h.fourier_transform(f, mom, beta, 64)
    assert np.array_equal(first, again)
    h.close()
