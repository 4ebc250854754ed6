"""What the host code plans and launches, on the CPU (hip_record.cpp plays the HIP runtime)."""
import os

import pytest

import recorded as R

LDS = 160 * 1024  # of a workgroup on gfx950


@pytest.mark.skipif(not os.path.exists(R.READELF), reason="llvm-readelf not available")
@pytest.mark.parametrize("ncat", range(1, 9))
def test_lds_of_every_launch_fits(ncat):
    """4 states, both forms and scaling modes, short and long alignments and every kind of op list
    (post-order, all directions, the moves of all branches); no call is refused."""
    got = R.run(f"""
    out, ncat = [], {ncat}
    for taxa in (5, 9, 12, 20, 30, 38, 40, 41, 64, 100, 160):
        for nptn in (1, 1000, 16000, 64 * 512, 64 * 512 + 1):
            if nptn > 16000 and taxa not in (20, 41, 100):
                continue
            p = S.make_problem(4, taxa, 1, np.random.default_rng(taxa), ncat=ncat, compress=False)
            p.states, p.freq, p.nptn = np.repeat(p.states, nptn, 1), np.ones(nptn), nptn
            internal = [(u, int(v)) for u in range(taxa, 2 * taxa - 2) for v in p.nei[u] if v > u]
            for prec, safe in ((G.FP64, 0), (G.FP64, 1), (G.FP32, 0)):
                t = G.Tree(p, precision=prec, scaling=safe, all_directions=2 if taxa <= 100 and nptn <= 1000 else 1)
                rc = [called(t.full_traversal)]
                G.lib().plk_tree_clear_all(t.h)
                rc.append(called(t.derivs, 0, int(p.nei[0, 0])))
                G.lib().plk_tree_clear_all(t.h)
                rc.append(called(t.all_branch_derivs))
                if taxa <= 100 and nptn <= 1000 and prec == G.FP64:
                    G.lib().plk_tree_clear_all(t.h)
                    rc.append(called(t.nni_evaluate, internal))
                out.append((taxa, nptn, prec, safe, rc, sorted(set((n, l) for n, l, _ in launches()))))
                t.close()
    print(json.dumps(out))
    """)
    static = R.static_lds()
    for taxa, nptn, prec, safe, rc, kernels in got:
        assert not any(rc), (taxa, nptn, prec, safe, rc)
        assert any("k_traverse_dna" in name for name, _ in kernels)
        for name, lds in kernels:
            assert lds + static[name] <= LDS, (taxa, nptn, prec, safe, name, lds)


@pytest.mark.parametrize("prec", ["FP64", "FP32"])
def test_failed_launch_keeps_the_transition_matrices_to_come(prec):
    """After a refused traversal the next call forms P(t) of all queued ops, whichever kernel it
    takes, and of its own branch once."""
    got = R.run(f"""
    p = S.make_problem(4, 12, 300, np.random.default_rng(1), compress=False)
    w = int(p.nei[0, 0])
    out = []
    for waves in (0, 1, -1):
        calls = []
        for fails in (0, 1, 3):
            t = G.Tree(p, precision=G.{prec})
            rec.rec_fail(b"k_traverse")
            rc = [called(t.loglik, 0, w) for _ in range(fails)]
            rec.rec_fail(b"")
            t.set_level_waves(waves)
            launches()
            rc.append(called(t.loglik, 0, w))
            calls.append((rc, launches()))
            t.close()
        out.append(calls)
    print(json.dumps(out))
    """)
    for fresh, *after in got:
        assert fresh[0] == [0]
        for rc, kernels in after:
            assert all(rc[:-1]) and rc[-1] == 0
            assert kernels == fresh[1]


def test_exchange_places_after_a_failed_solve():
    """Every one-launch solve finds its exchange places empty, also after launches that failed."""
    got = R.run("""
    p = S.make_problem(4, 12, 300, np.random.default_rng(1), compress=False)
    t = G.Tree(p, all_directions=2)
    w, inner = int(p.nei[0, 0]), [(u, int(v)) for u in range(12, 22) for v in p.nei[u] if v > u]
    out = []
    for step in ("one", "all", "one", "all", "", "one", "all", "", "one", "one", "all", "all"):
        rec.rec_fail(b"" if step else b"k_newton_solve")
        if step != "all":
            rc = called(t.optimize_one, 0, w)
        if step != "one":
            rc = called(t.nni_evaluate, inner)
        out.append((step, rc, rec.rec_dirty()))
    print(json.dumps([out, [n for n, _, _ in launches() if "newton_solve" in n]]))
    """)
    assert all((rc == 0) == bool(step) for step, rc, _ in got[0])
    assert any("solve_multi" in n for n in got[1]) and any("solveI" in n for n in got[1])
    assert not any(dirty for _, _, dirty in got[0]), got[0]


def test_exchange_places_are_allocated_for_solves_only():
    """Derivatives of all branches allocate none (8 + 24 bytes a branch and tile is what they need), nor
    do sizes that the one-launch solve does not take; all is given back."""
    got = R.run("""
    out = []
    for nptn in (6400, 64 * 1500):
        p = S.make_problem(4, 12, 1, np.random.default_rng(1), compress=False)
        p.states, p.freq, p.nptn = np.repeat(p.states, nptn, 1), np.ones(nptn), nptn
        before = rec.rec_bytes()
        t = G.Tree(p, all_directions=2)
        t.full_traversal()
        inner = [(u, int(v)) for u in range(12, 22) for v in p.nei[u] if v > u]
        sizes = [rec.rec_bytes()]
        for f in (t.all_branch_derivs, lambda: t.nni_evaluate(inner)):
            called(f)
            sizes.append(rec.rec_bytes())
        t.close()
        out.append((nptn // 64, len(inner), [b - a for a, b in zip(sizes, sizes[1:])], rec.rec_bytes() - before))
    print(json.dumps(out))
    """)
    for tiles, moves, (derivs, nni), left in got:
        slack = 1 << 20  # parameters, queued ops and their P(t)
        assert derivs <= 2 * 12 * 32 * tiles + slack, (tiles, derivs)
        assert nni <= (2 * moves * 144 * tiles if tiles <= 1024 else 0) + slack, (tiles, nni)
        assert left == 0


@pytest.mark.skipif(not os.path.exists(R.READELF), reason="llvm-readelf not available")
@pytest.mark.parametrize("n", [4, 20, 61])
def test_a_solve_takes_a_quarter_of_the_places(n):
    """The workgroups of one branch wait for each other: four solves of different streams must fit the
    256 compute units together, by wavefronts (16 a compute unit, 61 states 8) and by LDS."""
    got = R.run(f"""
    out, n = [], {n}
    for ncat in range(1, 9):
        for tiles in (1, 15, 64, 100, 128, 129, 255, 256, 257, 400, 512, 513, 700, 1024, 1025, 2047, 2048, 4096, 4097):
            p = S.make_problem(n, 4, 1, np.random.default_rng(1), ncat=ncat, compress=False)
            p.nptn = 64 * tiles
            p.states, p.freq = np.repeat(p.states, p.nptn, 1), np.ones(p.nptn)
            t = G.Tree(p, all_directions=2)
            rec.rec_finish(1)
            called(t.optimize_one, 0, int(p.nei[0, 0]))
            called(t.nni_evaluate, [(4, 5)])
            out.append((ncat, tiles, [k for k in launches() if "newton_solve" in k[0]]))
            t.close()
    print(json.dumps(out))
    """)
    static, seen = R.static_lds(), 0
    for ncat, tiles, solves in got:
        for name, _, blocks in solves:
            places = min(LDS // static[name], (8 if n == 61 else 16) // ncat) * 256
            blocks //= 2 if "multi" in name else 1  # two moves of one branch
            assert 4 * blocks <= places, (ncat, tiles, name, blocks, places)
            seen += 1
    assert seen > 100


def test_solves_whose_waits_end_are_not_tried_again_at_once():
    """A solve whose wait ends has lost that time: the context goes back to one launch per evaluation
    for a while, longer each time in a row, until a one-launch solve finishes or the bound is set."""
    got = R.run("""
    p = S.make_problem(4, 12, 300, np.random.default_rng(1), compress=False)
    t = G.Tree(p)
    w = int(p.nei[0, 0])
    def tries(n, finish):
        rec.rec_finish(finish)
        for _ in range(n):
            called(t.optimize_one, 0, w)
        return sum("newton_solve" in k[0] for k in launches())
    out = [tries(50, 1), tries(250, 0), tries(700, 0), tries(2000, 0), tries(8000, 1)]
    tries(1, 0)
    one, ended = ctypes.c_int64(), ctypes.c_int64()
    G.lib().plk_get_solve_counts(t.context(), ctypes.byref(one), ctypes.byref(ended))
    out += [one.value, ended.value]
    G.lib().plk_set_solve_wait(t.context(), 20000)
    out.append(tries(5, 1))
    print(json.dumps(out))
    """)
    # pauses of 256, 512, 1,024 and 2,048 solves, one try between two of them; then 256 again
    assert got[:5] == [50, 1, 2, 1, 8000 - 2048 + (50 + 250 + 700 + 2000) - (50 + 4 + 256 + 512 + 1024)]
    assert got[5:] == [50 + got[4], 5, 5]


def test_codon_launch_fills_the_device():
    """61 states in FP64: a long alignment gets as many workgroups as eight wavefronts a compute unit
    hold, whatever the number of categories and the scaling."""
    got = R.run("""
    out = []
    for ncat in range(1, 9):
        for safe in (0, 1):
            p = S.make_problem(61, 4, 1, np.random.default_rng(1), ncat=ncat, compress=False)
            p.nptn = 64 * 400
            p.states, p.freq = np.repeat(p.states, p.nptn, 1), np.ones(p.nptn)
            t = G.Tree(p, scaling=safe)
            called(t.full_traversal)
            for i in range(rec.rec_count()):
                if b"k_traverse_f64_codon" in rec.rec_name(i):
                    out.append((ncat, safe, rec.rec_blocks(i) * rec.rec_threads(i) // 64))
            rec.rec_clear()
            t.close()
    print(json.dumps(out))
    """)
    assert len(got) == 16
    for ncat, safe, wavefronts in got:
        assert wavefronts >= 256 * (8 if safe else 8 // ncat * ncat), (ncat, safe, wavefronts)


def test_small_mixed_batch_is_two_launches():
    """FP32 partitions of both data types whose items the device takes at once: one P(t) launch, one
    traversal (more items: one of each per kernel)."""
    got = R.run("""
    out = []
    for sizes in ((300, 200, 64), (64 * 255, 64 * 257), (64 * 256, 64 * 257), (300,)):
        trees = []
        for i, nptn in enumerate(sizes):
            p = S.make_problem(20 if i == 0 and len(sizes) > 1 else 4, 5, nptn, np.random.default_rng(i), compress=False)
            trees.append(G.Tree(p, precision=G.FP32))
        b = G.Batch(trees)
        launches()
        rc = called(b.loglik, [(0, int(t.p.nei[0, 0])) for t in trees], clear=True)
        out.append((rc, [n for n, _, _ in launches() if "pmatrix" in n or "traverse" in n]))
        b.close()
    print(json.dumps(out))
    """)
    assert [(rc, len(k)) for rc, k in got] == [(0, 2), (0, 2), (0, 4), (0, 2)], got


@pytest.mark.skipif(not os.path.exists(R.READELF), reason="llvm-readelf not available")
def test_fp32_derivative_kernels_leave_room_for_two_wavefronts():
    """20 states: 256 vector registers at most (matrices read ahead of the category loop took 280)."""
    kernels = {n: v for n, (_, v) in R.kernel_notes().items()
               if any(k in n for k in ("k_multi_derivs_f32ILi20E", "k_multi_newtonILi20ELb1E", "k_theta_f32ILi20E"))}
    assert len(kernels) == 3 and max(kernels.values()) <= 256, kernels
