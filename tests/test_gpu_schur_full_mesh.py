"""The Schur kernels on the full meshes of the two large lattices against the plain full inverse,
which shares no kernel with them (48 frequencies, so that the Gauss rule of the density sums takes
part; bound as in test_gpu_schur_forms), and the two Schur methods against each other: they run the
same elimination, so their results are equal to the bit."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def rel(x, ref):
    return float(np.max(np.abs(np.asarray(x) - ref)) / np.max(np.abs(ref)))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["large32", "dp14"])
def test_against_the_full_inverse(G, name):
    w = L.workload(name, seed=1, n_freq=48)
    Hk, sig, beta, mom, ncl = w["Hk"], w["sigma"], w["beta"], w["exact_moments"], w["n_cluster"]
    nf, nc, n = sig.shape[0], sig.shape[1], Hk.shape[1]
    print(f"{name}: nk={Hk.shape[0]} nf={nf}", flush=True)
    lat = G.LatticeGF(Hk, nc, nf, beta, mom, n_cluster=ncl)
    del w, Hk
    rng = np.random.default_rng(2)
    gbar = rng.normal(size=sig.shape) + 1j * rng.normal(size=sig.shape)
    mu = 0.1
    ref = lat.greenftn_w(sig, mu, method=G.PLAIN_F64)
    sb, mb = lat.vjp(sig, mu, gbar, 0.4, method=G.PLAIN_F64)
    n0, dn0 = lat.density(sig, mu, method=G.PLAIN_F64)
    got = []
    for method in (G.SCHUR_F64, G.SCHUR_F32R):
        out = lat.greenftn_w(sig, mu, method=method)
        assert rel(out["gloc"], ref["gloc"]) <= 1e-12 and rel(out["num_matrix"], ref["num_matrix"]) <= 1e-12
        assert abs(out["n_total"] - ref["n_total"]) <= 1e-12 * n
        s, m = lat.vjp(sig, mu, gbar, 0.4, method=method)
        assert rel(s, sb) <= 1e-12 and abs(m - mb) <= 1e-12 * max(1.0, abs(mb))
        N, dN = lat.density(sig, mu, method=method)
        assert abs(N - n0) <= 1e-12 * n and abs(dN - dn0) <= 1e-12 * max(1.0, abs(dn0))
        got.append([out["gloc"], out["num_matrix"], out["n_total"], s, m, N, dN])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,nc", [(3, 1), (9, 3), (14, 5), (14, 6), (20, 10), (18, 16)])
@pytest.mark.parametrize("layout", [0, 1])
def test_schur_methods_are_one(G, n, nc, layout):
    Hk = L.random_tb_hk(n, 4, n)
    sig, mom = L.pole_sigma(nc, 70, 20.0, nc)
    lat = G.LatticeGF(Hk, nc, 70, 20.0, mom)
    lat.set_option(G.capi.OPT_SCHUR_LAYOUT, layout)
    a, b = (lat.loss_grad(sig, 0.1, 0.9 * sig, 1.0, method=m) for m in (G.SCHUR_F64, G.SCHUR_F32R))
    for key in a:
        assert np.array_equal(a[key], b[key]), key
    sr = np.repeat(sig[:1], 30, axis=0)
    for x, y in zip(*(lat.greenftn_real(sr, 0.1, -2.0, 0.1, 0.05, method=m) for m in (G.SCHUR_F64, G.SCHUR_F32R))):
        assert np.array_equal(x, y)
    lat.close()
