"""Host side of the library's calls, on the stand-in for the HIP runtime (host_hip.py): which
kernels a call launches with which grids, how much scratch it asks for, and that the host
source of every asynchronous copy lives until the stream is waited for."""
import pytest

from tests import host_hip

FT = """
import ctypes as C
h = rt.handle()
d, nf, nt = 4, 40, 64
f, g = rt.dev(16 * nf * d * d), rt.dev(16 * (nt + 1) * d * d)
mom = rt.dev(np.stack([np.zeros((d, d)), np.eye(d), 0.1 * np.eye(d), np.eye(d)]).astype(np.complex128))
"""


@pytest.mark.parametrize("call", [
    "rt.lib.dmftgpu_ft_w2tau(h, d, nf, nt, 20.0, f, mom, g, None)",
    "rt.lib.dmftgpu_ft_w2tau_points(h, d, nf, 20.0, f, mom, 3, (C.c_double * 3)(0.1, 0.2, 0.3), g)",
])
def test_tail_copy_source_outlives_the_copy(call):
    assert host_hip.run(FT + f"rt.reset()\nrt.check(h, {call})\nresult = rt.stale()") == 0


SPLIT = r"""
import ctypes as C, re
def forms(nk):
    out = []
    for name, grid, block in rt.launches():
        m = re.match(r"void dg::k_lattice_schur<(\d+), (\d+), (\d+), \w+, (\d+)>", name)
        if m:
            mode, parts, chunks = int(m[2]), int(m[4]), grid[1]
            out.append((mode, int(m[3]) // parts, parts, -(-nk // chunks), chunks * grid[0]))
    return out
result = []
for nc, nd in ((3, 6), (4, 0), (4, 6), (5, 0), (5, 9), (6, 0), (6, 8)):
    for nk, nf in ((64, 64), (512, 64), (512, 256), (1000, 512), (1728, 512), (4096, 512)):
        h = rt.handle()
        rt.prepare(h, nc + nd, nc, nk, nf)
        s, g, num = rt.dev(16 * nf * nc * nc), rt.dev(16 * nf * nc * nc), rt.dev(16 * nc * nc)
        rt.reset()
        call
        result.append((nc, nd, nk, nf, forms(nk)))
        rt.lib.dmftgpu_destroy(h)
"""


def test_split_walk_has_a_k_for_every_wavefront():
    """Matsubara forward and adjoint, real axis summed: where wavefronts split a chunk's k walk, the
    chunks are multiples of their number and there are 256 workgroups of them"""
    calls = ["rt.check(h, rt.lib.dmftgpu_gloc_loss_grad(h, 1, s, 0.1, g, 1.0, g, num, None, None, s, None))",
             "rt.check(h, rt.lib.dmftgpu_greenftn_real(h, 1, nf, -1.0, 0.01, 0.05, s, 0.1, g, None))"]
    seen = set()
    for call in calls:
        for nc, nd, nk, nf, forms in host_hip.run(SPLIT.replace("call", call)):
            assert forms, (nc, nd, nk, nf)
            for mode, width, parts, per_chunk, groups in forms:
                assert width in (64, 128)
                if parts > 1:
                    assert per_chunk % parts == 0 and groups >= 256, (nc, nd, nk, nf, mode, parts, per_chunk, groups)
                seen.add((mode, parts))
    # adjoint in four, in two (n_c = 6) and alone, forward and real axis in two and alone
    assert seen >= {(2, 4), (2, 2), (2, 1), (0, 2), (0, 1), (5, 2), (5, 1)}


def test_band_spectra_do_no_k_twice():
    """one k per workgroup: no split walk, but for n_c = 6 without (many) d orbitals, which gains from it"""
    call = "rt.check(h, rt.lib.dmftgpu_greenftn_real_k(h, 1, nf, -1.0, 0.01, 0.05, s, 0.1, rt.dev(16 * nk * nf * nc * nc), None))"
    for nc, nd, nk, nf, forms in host_hip.run(SPLIT.replace("call", call)):
        assert [f[2] for f in forms] == [2 if nc == 6 and nd < 2 else 1], (nc, nd, nk, nf, forms)


def test_frequency_rule_needs_no_host_memory_after_the_call():
    """two grids one after the other with no wait between: the second preparation must not take the
    first one's rule from under its copy"""
    assert host_hip.run("""
        h = rt.handle()
        rt.reset()
        for nf in (4000, 200, 100):
            rt.prepare(h, 5, 3, 8, nf)
        result = rt.stale()
    """) == 0


def test_preparation_reads_only_what_it_queued_on_its_own_stream():
    """the same grid prepared on one stream and then on another queues the same work: nothing that
    the first stream may still be writing is read by the second"""
    work = host_hip.run("""
        import ctypes as C
        h = rt.handle(C.c_void_p(0x1000))
        result = []
        for stream in (0x1000, 0x2000):
            rt.check(h, rt.lib.dmftgpu_set_stream(h, C.c_void_p(stream)))
            rt.reset()
            rt.prepare(h, 5, 3, 8, 100)
            result.append([e.replace(str(stream), "S") for e in rt.events() if not e.startswith("malloc")])
    """)
    assert work[0] == work[1] and len(work[0]) > 3


def test_transform_tables_are_kept_while_the_stream_is():
    counts = host_hip.run("""
        import ctypes as C
        h = rt.handle(C.c_void_p(0x1000))
        d, nf, nt = 2, 40, 64
        f, g = rt.dev(16 * nf * d * d), rt.dev(16 * (nt + 1) * d * d)
        result = []
        for stream in (0x1000, 0x1000, 0x2000):
            rt.check(h, rt.lib.dmftgpu_set_stream(h, C.c_void_p(stream)))
            rt.reset()
            rt.check(h, rt.lib.dmftgpu_ft_tau2w(h, d, nf, nt, 20.0, g, f, None))
            result.append(sum("k_czt_phases" in name for name, _, _ in rt.launches()))
    """)
    assert counts == [1, 0, 1]


def test_small_tau_transforms_take_one_launch_and_the_causality_test():
    """a tau -> iw transform of a few hundred points: no FFTs, whose launches cost more than its sums"""
    names = host_hip.run("""
        h = rt.handle()
        result = []
        for d, nf, nt in ((1, 64, 128), (5, 200, 400), (5, 1000, 2000)):
            f, g = rt.dev(16 * nf * d * d), rt.dev(16 * (nt + 1) * d * d)
            for _ in range(2):  # the tables are kept
                rt.reset()
                rt.check(h, rt.lib.dmftgpu_ft_tau2w(h, d, nf, nt, 20.0, g, f, None))
            result.append([name for name, _, _ in rt.launches()])
    """)
    assert [len(n) for n in names] == [2, 2, 4]
    assert all("k_not_posdef" in n[-1] for n in names)


@pytest.mark.parametrize("d,nf,nt", [(32, 65536, 131072), (10, 65536, 131072), (4, 100000, 3000), (32, 3000, 100000)])
def test_scratch_of_the_tau_transforms(d, nf, nt):
    """a copy of each grid and a bounded number of partial sums: not a partial sum of the whole
    output for every 2048 inputs (69 GB at the first of these sizes)"""
    to_tau, to_w = host_hip.run(f"""
        import ctypes as C
        d, nf, nt = {d}, {nf}, {nt}
        f, g = rt.dev(16 * nf * d * d), rt.dev(16 * (nt + 1) * d * d)
        mom = rt.dev(np.stack([np.zeros((d, d)), np.eye(d), 0.1 * np.eye(d), np.eye(d)]).astype(np.complex128))
        result = []
        for call in ("w2tau", "tau2w"):
            h = rt.handle()
            rt.reset()
            before = rt.peak()
            if call == "w2tau":
                rt.check(h, rt.lib.dmftgpu_ft_w2tau(h, d, nf, nt, 20.0, f, mom, g, None))
            else:
                rt.check(h, rt.lib.dmftgpu_ft_tau2w(h, d, nf, nt, 20.0, g, f, None))
            result.append(rt.peak() - before)
            rt.lib.dmftgpu_destroy(h)
    """)
    grids = 16 * d * d * (nf + nt + 1)
    eig = 16 * d * d * nf  # tau -> iw: (F - F^H)/2i for the eigensolver
    assert to_tau <= grids + 2 ** 30 and to_w <= grids + eig + 2 ** 30, (to_tau, to_w, grids)


def test_dense_hopping_lists_are_told_from_sparse_ones_in_any_order():
    """H(k) takes the dense sums exactly where at least half of all (R, element) pairs are listed:
    lists around that line, grouped by R, shuffled, element by element, with R far apart, with
    pairs listed twice"""
    cases = host_hip.run("""
        import ctypes as C
        rng = np.random.default_rng(5)
        h = rt.handle()
        result = []
        for n, n_r in ((1, 1), (1, 40), (3, 7), (6, 19), (6, 130), (2, 1000)):
            R = np.unique(rng.integers(-6, 7, size=(4 * n_r, 3)), axis=0)[:n_r]
            for scale in (1, 1, 40000000):
                pairs = np.array([(*(scale * r), i, j) for r in R for i in range(n) for j in range(n)], np.int32)
                full = len(pairs)
                for keep in {1, full // 4, (full + 1) // 2 - 1, (full + 1) // 2, (full + 1) // 2 + 1, full}:
                    if keep < 1: continue
                    pick = np.sort(rng.permutation(full)[:keep])
                    by_element = pick[np.lexsort((pick, pairs[pick, 3], pairs[pick, 4]))]
                    for rows in (pick, rng.permutation(pick), by_element, np.repeat(pick, 2)):
                        idx = np.ascontiguousarray(pairs[rows])
                        t = np.ones(2 * len(idx))
                        distinct = len(np.unique(idx[:, :3], axis=0))
                        rt.reset()
                        rt.check(h, rt.lib.dmftgpu_hk_from_hr(h, n, len(idx), idx.ctypes.data_as(C.POINTER(C.c_int)),
                                                              t.ctypes.data_as(C.POINTER(C.c_double)), 4,
                                                              rt.dev(96), rt.dev(64 * n * n)))
                        dense = any("k_hk_dense" in name for name, _, _ in rt.launches())
                        result.append([bool(distinct * n * n <= 2 * len(idx)), dense, rt.stale()])
    """)
    assert all(want == got and not stale for want, got, stale in cases)
    assert {want for want, _, _ in cases} == {True, False} and len(cases) > 300


def test_eigensolver_form_by_size_and_count():
    """17 to 29 rows: the LDS kernel where one round of it ends before a round of the 32-lane slots
    (or needs no more rounds); from 30 on, for many matrices, and without vectors the slots"""
    names = host_hip.run("""
        result = []
        for n, nk in ((17, 5000), (25, 5000), (26, 1), (26, 1700), (26, 2000), (26, 2700), (26, 4096), (27, 1200),
                      (27, 1700), (28, 1024), (28, 1100), (29, 512), (29, 2000), (30, 64), (32, 1)):
            h = rt.handle()
            rt.prepare(h, n, 5, nk, 8)
            rt.reset()
            rt.check(h, rt.lib.dmftgpu_update_moments(h, rt.dev(16 * 4 * 25)))
            result.append([n, nk, any("k_herm_eig(" in name for name, _, _ in rt.launches())])
            rt.lib.dmftgpu_destroy(h)
    """)
    slots = {(26, 2000), (26, 4096), (27, 1700), (28, 1100), (29, 2000), (30, 64), (32, 1)}
    assert {(n, nk) for n, nk, lds in names if not lds} == slots
