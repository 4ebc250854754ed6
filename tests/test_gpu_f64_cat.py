"""FP64 20-state traversal on the matrix cores: every category count (1-2 put pattern groups
into the idle blocks, 5-8 take two wavefronts), both widths (one and two patterns per
column; the wider from one wavefront per SIMD on), ragged ends, NORM and SAFE with forced
rescaling, against the vector form and the oracle: logL within 1e-10 relative, derivatives
1e-9, scale counts equal (partial vectors are compared in test_gpu_f64_mfma.py).  Batched launches equal the same contexts alone bit for bit, also after a form switch."""
import sys

import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def rel(a, b):
    return abs(a - b) / max(abs(b), 1e-300)


def check(p, safe, depth):
    gm, gv = G.Tree(p, scaling=safe), G.Tree(p, scaling=safe)
    gv.set_f64_form(0)
    o = S.Oracle(p, safe=bool(safe), nthreads=8)
    a, b = 0, int(p.nei[0, 0])
    lm, pm = gm.loglik(a, b, with_patterns=True)
    lo, po = o.loglik(a, b, with_patterns=True)
    assert rel(lm, lo) <= 1e-10 and rel(lm, gv.loglik(a, b)) <= 1e-10
    np.testing.assert_allclose(pm, po, rtol=1e-10, atol=1e-10)
    dm, do = gm.derivs(a, b)[:2], o.derivs(a, b)[:2]
    for x, y in zip(dm, do):
        assert abs(x - y) <= 1e-9 * max(1.0, abs(y))
    top = 0
    for w in range(p.ntaxa, 2 * p.ntaxa - 2, max(1, (p.ntaxa - 2) // 3)):
        d = int(p.nei[w, 0])
        assert rel(gm.loglik(d, w), lo) <= 1e-10
        _, sm = gm.partial(d, w, safe=bool(safe))
        _, so = o.partial(d, w, safe=bool(safe))
        assert np.array_equal(sm, so)
        top = max(top, int(so.max()))
    assert top >= depth
    gm.close()
    gv.close()


@pytest.mark.parametrize("safe", [0, 1], ids=["norm", "safe"])
@pytest.mark.parametrize("ncat", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("wide", [0, 1], ids=["pg1", "pg2"])
def test_categories_and_widths(ncat, safe, wide):
    units = max(1, G.device_units())
    # the wider form starts above one wavefront per SIMD: 16 patterns per compute unit with
    # 3-4 categories, half with 5-8 (two wavefronts a unit), twice with 2
    limit = 16 * units * (2 if ncat == 2 else 1) // (2 if ncat > 4 else 1)
    nptn = limit + 1 if wide else 131
    rng = np.random.default_rng(100 * ncat + 10 * safe + wide)
    p = S.make_problem(20, 7, nptn, rng, ncat=ncat, mean_len=0.3, ambiguous=0.05, compress=False)
    say("cat", ncat, "safe", safe, "patterns", p.nptn)
    check(p, safe, 0)


@pytest.mark.parametrize("safe", [0, 1], ids=["norm", "safe"])
@pytest.mark.parametrize("ncat", [1, 2, 4, 6])
def test_forced_rescaling(ncat, safe):
    rng = np.random.default_rng(ncat)
    p = S.make_problem(20, 90, 70, rng, ncat=ncat, tree=S.caterpillar_tree(90, 1.5), ambiguous=0.05)
    say("rescaling", ncat, "safe", safe, p.nptn)
    check(p, safe, 1)  # at least one rescaling seen at the sampled nodes


def test_batch_equals_alone():
    rng = np.random.default_rng(5)
    probs = [S.make_problem(n, 9, sites, rng, ncat=ncat, ambiguous=0.03, compress=False)
             for n, sites, ncat in [(20, 1, 4), (20, 33, 1), (4, 65, 4), (20, 5000, 3), (20, 64, 2), (4, 700, 2), (20, 129, 4)]]
    trees = [G.Tree(p) for p in probs]
    br = [(0, int(p.nei[0, 0])) for p in probs]
    batch = G.Batch(trees)
    for form in (1, 0, -1):  # switched on the live batch
        trees[3].set_f64_form(form)
        alone = np.array([t.full_traversal() for t in trees])
        for _ in range(3):
            vals, _ = batch.loglik(br, clear=True)
            assert np.array_equal(vals, alone), form
        for p, v in zip(probs, vals):
            assert rel(v, S.Oracle(p, nthreads=4).loglik(0, int(p.nei[0, 0]))) <= 1e-10
    batch.close()
