"""Schur kernels around their dispatch lines, against the plain full inverse: the forward as one
or two wavefronts per 64 frequencies (n_c = 3..6 around n_d = 6, odd k counts, Matsubara and real
axis), the adjoint as one, two or four (n_c = 4..6), and the column-per-lane buckets with padding and spare lanes.
Bound: two backward-stable inverses of matrices with condition |A| / w_0, about 1e2 here, differ by
a few hundred roundings (2e-14); 1e-12 as for the oracle elsewhere, 1e-11 on the real axis at
eta = 0.05 (condition 1e3)."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def rel(x, ref):
    x, ref = np.asarray(x), np.asarray(ref)
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


SIZES = [(3, 5), (3, 6), (4, 0), (4, 6), (5, 5), (5, 6), (6, 0), (6, 2),
         (7, 0), (7, 5), (9, 3), (10, 22), (11, 1), (13, 4), (14, 18), (15, 2), (16, 16)]


@pytest.mark.gpu
@pytest.mark.parametrize("nc,nd", SIZES)
@pytest.mark.parametrize("nf,target", [(1, 0), (67, 9)])
def test_schur_forms(G, nc, nd, nf, target):
    beta, mu = 20.0, 0.15
    Hk = L.random_tb_hk(nc + nd, 3, nc + nd)
    sig, mom = L.pole_sigma(nc, nf, beta, nc)
    lat = G.LatticeGF(Hk, nc, nf, beta, mom)
    lat.set_option(G.capi.OPT_TARGET_WORKGROUPS, target)
    rng = np.random.default_rng(nc)
    gbar = rng.normal(size=(nf, nc, nc)) + 1j * rng.normal(size=(nf, nc, nc))
    ref = lat.greenftn_w(sig, mu, method=G.PLAIN_F64)
    sb, mb = lat.vjp(sig, mu, gbar, 0.7, method=G.PLAIN_F64)
    n0, dn0 = lat.density(sig, mu, method=G.PLAIN_F64)
    print(f"nc={nc} nd={nd} nf={nf} target={target}", flush=True)
    for method in (G.SCHUR_F64, G.SCHUR_F32R):
        out = lat.greenftn_w(sig, mu, method=method)
        assert rel(out["gloc"], ref["gloc"]) <= 1e-12 and rel(out["num_matrix"], ref["num_matrix"]) <= 1e-12
        assert abs(out["n_total"] - ref["n_total"]) <= 1e-12 * (nc + nd)
        s, m = lat.vjp(sig, mu, gbar, 0.7, method=method)
        assert rel(s, sb) <= 1e-12 and abs(m - mb) <= 1e-12 * max(1.0, abs(mb))
        n, dn = lat.density(sig, mu, method=method)
        assert abs(n - n0) <= 1e-12 * (nc + nd) and abs(dn - dn0) <= 1e-12 * max(1.0, abs(dn0))
    ne = nf + 2
    sr = np.repeat(sig[:1], ne, axis=0)
    g0, t0 = lat.greenftn_real(sr, mu, -3.0, 0.09, 0.05, method=G.PLAIN_F64)
    g1, t1 = lat.greenftn_real(sr, mu, -3.0, 0.09, 0.05, method=G.SCHUR_F64)
    assert rel(g1, g0) <= 1e-11 and rel(t1, t0) <= 1e-11
    lat.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nc,bad", [(5, (0, 0)), (20, (19, 19))])
@pytest.mark.parametrize("want_n", [True, False])
def test_failed_call_leaves_num_matrix(G, nc, bad, want_n):
    """A result that is not finite is an error, and the caller's NumMatrix keeps what it held
    (one element of a block of nc^2 threads is enough to refuse all of them)."""
    import torch
    Hk = L.random_tb_hk(nc + 2, 2, nc)
    sig, mom = L.pole_sigma(nc, 6, 20.0, nc)
    lat = G.LatticeGF(Hk, nc, 6, 20.0, mom)
    sig = sig.copy()
    sig[(3,) + bad] = np.nan
    num = torch.full((nc, nc), 7.0, dtype=torch.complex128, device="cuda")
    with pytest.raises(Exception, match="not finite"):
        lat.greenftn_w_dev(lat.sigma_dev(sig), 0.1, G.PLAIN_F64, num=num, want_n=want_n)
    assert bool((num == 7.0).all())
    lat.close()
