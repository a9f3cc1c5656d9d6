"""The one-kernel upfolding (n_orb <= 32) and the dense R sums at the edges of their tiles,
against the oracle, at the upfolding bar (1e-12 normwise relative): orbital counts around
16 and 32, transforms whose elimination needs row exchanges in every column, padded
bands, R lists on both sides of the dense rule and counts that are no multiple of 14."""
import numpy as np
import pytest

from dmftpack_amd import lattice as L
from oracle import oracle as O

BETA, MU = 40.0, 0.2


def rel(x, ref):
    return float(np.max(np.abs(np.asarray(x) - ref)) / max(np.max(np.abs(ref)), 1e-300))


@pytest.fixture(scope="module")
def gpu():
    from dmftpack_amd import gpu as G
    h = G.Handle()
    yield G, h
    h.close()


def run(h, c, **kw):
    args = (c["dm_model"], c["corr_base"], c["ks_energy"], c["val_to_ks"], c["transform"], c["ks_ortho"],
            c["overlap"], BETA, MU, c["r_idx"], c["kphase"])
    return h.upfold_density(*args, **kw), O.upfold_density(*args)


def check(h, c):
    (D, dmr), (Dr, dmr_r) = run(h, c)
    assert rel(D, Dr) <= 1e-12
    for x in range(3):
        assert rel(dmr[x], dmr_r[x]) <= 1e-12, x


@pytest.mark.gpu
@pytest.mark.parametrize("n,n_orb", [(1, 2), (2, 15), (15, 16), (16, 16), (3, 17), (14, 28), (31, 31), (17, 32), (32, 32),
                                     (9, 33)])
@pytest.mark.parametrize("overlap", [True, False])
def test_orbital_counts(gpu, n, n_orb, overlap):
    G, h = gpu
    check(h, L.upfold_case(n, n_orb, 2, 50 + n_orb, overlap=overlap))


@pytest.mark.gpu
@pytest.mark.parametrize("n_orb", [7, 16, 20, 32])
def test_row_exchanges(gpu, n_orb):
    """transforms and overlaps with zero or tiny leading diagonals: a shifted identity plus noise
    (no column's diagonal entry is its largest)"""
    G, h = gpu
    c = L.upfold_case(4, n_orb, 2, 60 + n_orb)
    nk = c["transform"].shape[0]
    shift = np.roll(np.eye(n_orb), 3, axis=0)
    noise = c["transform"] - np.eye(n_orb)
    for i in range(n_orb):
        noise[:, i, i] = 0.0
    c["transform"] = shift[None] + 0.3 * noise
    flip = np.eye(n_orb)[::-1]
    c["overlap"] = flip[None] + 0.1 * (c["overlap"] - np.eye(n_orb))
    c["overlap"] = 0.5 * (c["overlap"] + c["overlap"].conj().transpose(0, 2, 1))
    assert np.linalg.cond(c["transform"]).max() < 50 and np.linalg.cond(c["overlap"]).max() < 50
    check(h, c)
    assert nk == 8


@pytest.mark.gpu
def test_padded_bands(gpu):
    G, h = gpu
    c = L.upfold_case(6, 19, 2, 71)
    for k in range(1, 8, 2):
        c["val_to_ks"][k, 4:] = -1
        c["dm_model"][k, 4:, :] = 0.0
        c["dm_model"][k, :, 4:] = 0.0
        c["corr_base"][k] = np.eye(6)
    check(h, c)


@pytest.mark.gpu
@pytest.mark.parametrize("n_orb", [5, 12, 35])
@pytest.mark.parametrize("keep", [1.0, 0.7, 0.5, 0.2])
@pytest.mark.parametrize("n_rv", [1, 14, 15, 29])
def test_r_lists(gpu, n_orb, keep, n_rv):
    G, h = gpu
    c = L.upfold_case(3, n_orb, 3, 80 + n_orb)
    rng = np.random.default_rng(n_orb + n_rv)
    Rs = np.unique(rng.integers(-4, 5, size=(4 * n_rv, 3)), axis=0)
    Rs = Rs[rng.permutation(len(Rs))[:n_rv]]
    rows = [(*R, i, j) for R in Rs for i in range(n_orb) for j in range(n_orb) if rng.uniform() < keep]
    rows = np.array(rows, dtype=np.int32)
    c["r_idx"] = rows[rng.permutation(len(rows))]
    check(h, c)
