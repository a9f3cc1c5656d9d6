"""The Gauss rule of the density sums beyond N_freq (csrc/freq_points.hip) against the
oracle, which adds every frequency: run lengths at the rule's edges, several octaves of
high_freq, and moments for which the rule is ruled out.  Tolerances are those of the
Schur path against the oracle (1e-12 relative in FP64, 1e-9 FP32 + refinement): the
rule's own error is below 1e-20."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L
from oracle import oracle as O

MU, BETA = 0.15, 40.0


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def rel(a, b):
    return np.max(np.abs(a - b)) / np.max(np.abs(b))


def case(n, nc, nf, scale=1.0):
    Hk = L.random_tb_hk(n, 2, seed=n + nf)
    sig, mom = L.pole_sigma(nc, nf, BETA, n + nf)
    return Hk, sig, mom * scale


def check(G, lat, Hk, sig, mom, hf, method, tol):
    ref = O.greenftn_w(Hk, sig, mom, MU, BETA, high_freq=hf)
    out = lat.greenftn_w(sig, MU, method=method)
    N_ref, dN_ref = O.density(Hk, sig, mom, MU, BETA, high_freq=hf)
    N, dN = lat.density(sig, MU, method=method)
    assert rel(out["gloc"], ref["gloc"]) <= tol
    assert rel(out["num_matrix"], ref["num_matrix"]) <= tol
    assert abs(out["n_total"] - N_ref) <= tol * max(1.0, abs(N_ref))
    assert abs(N - N_ref) <= tol * max(1.0, abs(N_ref))
    assert abs(dN - dN_ref) <= max(tol, 1e-10) * max(1.0, abs(dN_ref))  # as in the density tests
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("n,nc,method,tol", [(6, 3, 1, 1e-12), (9, 5, 2, 1e-9), (7, 5, 1, 1e-12), (12, 8, 1, 1e-12),
                                             (13, 10, 2, 1e-9), (3, 3, 1, 1e-12)])
@pytest.mark.parametrize("nf,hf", [(1, 2), (32, 2), (33, 2), (48, 3), (47, 5), (130, 2), (200, 1)])
def test_sums_against_every_frequency(G, n, nc, method, tol, nf, hf):
    Hk, sig, mom = case(n, nc, nf)
    lat = G.LatticeGF(Hk, nc, nf, BETA, mom, high_freq=hf)
    check(G, lat, Hk, sig, mom, hf, method, tol)
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,nc,method,tol", [(7, 5, 1, 1e-12), (9, 5, 2, 1e-9), (12, 8, 1, 1e-12)])
def test_moments_rule_the_points_out(G, n, nc, method, tol):
    """tail moments 1e3 times larger: |m1| is beyond the rule's bound, so every frequency is
    summed; the same handle returns to the rule (bit for bit) with the first moments"""
    nf = 96
    Hk, sig, mom = case(n, nc, nf)
    big = mom * 1e3
    lat = G.LatticeGF(Hk, nc, nf, BETA, mom)
    first = check(G, lat, Hk, sig, mom, 2, method, tol)
    lat.set_moments(big)
    check(G, lat, Hk, sig, big, 2, method, tol)
    if n <= 16 and nc <= 6:
        dens = O.greenftn_w(Hk, sig, big, MU, BETA, density=True)["density"]
        assert rel(lat.density_matrix(sig, MU), dens) <= 1e-12
    lat.set_moments(mom)
    again = lat.greenftn_w(sig, MU, method=method)
    for key in ("gloc", "num_matrix"):
        assert np.array_equal(first[key], again[key])
    assert first["n_total"] == again["n_total"]
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nf,nc", [(50, 4), (131, 5), (40, 6), (64, 1)])
def test_density_matrix(G, nf, nc):
    Hk, sig, mom = case(11, nc, nf)
    lat = G.LatticeGF(Hk, nc, nf, BETA, mom)
    ref = O.greenftn_w(Hk, sig, mom, MU, BETA, density=True)["density"]
    assert rel(lat.density_matrix(sig, MU), ref) <= 1e-12
    lat.close()


@pytest.mark.gpu
def test_batch_with_and_without_the_rule(G):
    """one batch whose systems differ in whether the rule applies"""
    systems, refs = [], []
    rng = np.random.default_rng(3)
    for i, (n, nc, nf, scale) in enumerate([(7, 5, 96, 1.0), (9, 5, 96, 1e3), (12, 8, 70, 1.0), (11, 8, 70, 1e3),
                                            (6, 3, 20, 1.0)]):
        Hk, sig, mom = case(n, nc, nf, scale)
        tgt = 0.1 * (rng.normal(size=sig.shape) + 1j * rng.normal(size=sig.shape))
        systems.append(dict(Hk=Hk, sigma=sig, moments=mom, beta=BETA, mu=MU, gloc_target=tgt, n_target=0.5 * n))
        ref = O.greenftn_w(Hk, sig, mom, MU, BETA)
        N, _ = O.density(Hk, sig, mom, MU, BETA)
        sb, mb = O.gloc_vjp(Hk, sig, mom, MU, BETA, 2.0 * (ref["gloc"] - tgt), 2.0 * (N - 0.5 * n))
        refs.append((ref, N, sb, mb))
    h = G.Handle()
    b = G.Batch(h, systems, method=1, tune=False, graph=True, prepare=True)
    for _ in range(2):
        b.run()
        for got, (ref, N, sb, mb) in zip(b.results(), refs):
            assert rel(got["gloc"], ref["gloc"]) <= 1e-12
            assert rel(got["num_matrix"], ref["num_matrix"]) <= 1e-12
            assert abs(got["n_total"] - N) <= 1e-12 * max(1.0, abs(N))
            assert rel(got["sigma_bar"], sb) <= 1e-10
            assert abs(got["mu_bar"] - mb) <= 1e-10 * max(1.0, abs(mb))
    b.close()
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,nc", [(6, 3), (9, 8)])
def test_rule_longer_than_one_kernel_argument(G, n, nc):
    """40 x 50 frequencies: six octaves, 96 points, which reach the table in blocks of 64"""
    Hk, sig, mom = case(n, nc, 40)
    lat = G.LatticeGF(Hk, nc, 40, BETA, mom, high_freq=50)
    check(G, lat, Hk, sig, mom, 50, 1, 1e-12)
    lat.close()
