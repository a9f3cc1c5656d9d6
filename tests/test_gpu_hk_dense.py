"""H(R) -> H(k) for hopping lists dense in (R, element) (one product per distinct R) and at
the line to the per-hop form, against the oracle.  Bound: each term's phase differs from the
oracle's by a few eps |phi.R| (phi <= pi), so 8 eps pi |R|_1 sum |t| per element plus rounding of
the sum; 1e-12 covers the lists below (|R|_1 <= 60, at most 12 R of |t| ~ 1)."""
import numpy as np
import pytest

from oracle import oracle as O


@pytest.fixture(scope="module")
def G():
    from dmftpack_amd import gpu
    return gpu


def hops_of(n, Rs, keep, seed, order="R"):
    rng = np.random.default_rng(seed)
    out = []
    for R in Rs:
        for i in range(n):
            for j in range(n):
                if rng.uniform() < keep:
                    out.append((*R, i, j, complex(rng.normal(), rng.normal())))
    if order == "element":
        out.sort(key=lambda h: (h[3], h[4]))
    if order == "shuffled":
        rng.shuffle(out)
    return [(int(h[0]), int(h[1]), int(h[2]), int(h[3]), int(h[4]), h[5]) for h in out]


NEAR = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, -1), (2, 1, 0), (-2, -1, 0), (0, 0, 3)]
FAR = [(20, -20, 20), (-20, 20, -20), (20, 20, 0), (0, -20, 20), (5, 0, 0)]  # a box of 41^3: no index table


@pytest.mark.gpu
@pytest.mark.parametrize("n,nk", [(1, 1), (1, 33), (3, 15), (8, 16), (9, 17), (15, 100), (16, 1), (17, 31), (32, 4099)])
@pytest.mark.parametrize("keep,order", [(1.0, "R"), (0.6, "element"), (0.5, "shuffled"), (0.3, "R")])
def test_dense_lists(G, n, nk, keep, order):
    hops = hops_of(n, NEAR, keep, n * 1000 + nk, order)
    if not hops:
        hops = [(1, 0, 0, 0, 0, 1.0 + 0j)]
    hops += hops[:2]  # duplicates add up
    rng = np.random.default_rng(nk)
    kp = rng.uniform(-np.pi, np.pi, size=(nk, 3))
    h = G.Handle()
    got = G.from_dev_cm(h.hk_from_hr(n, hops, kp))
    assert np.max(np.abs(got - O.hk_from_hr(n, hops, kp))) <= 1e-12
    h.close()


@pytest.mark.gpu
def test_scattered_r(G):
    hops = hops_of(4, FAR, 1.0, 3)
    kp = np.random.default_rng(4).uniform(-np.pi, np.pi, size=(50, 3))
    h = G.Handle()
    got = G.from_dev_cm(h.hk_from_hr(4, hops, kp))
    assert np.max(np.abs(got - O.hk_from_hr(4, hops, kp))) <= 1e-12
    h.close()
