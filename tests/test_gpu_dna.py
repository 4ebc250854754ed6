"""4-state traversal (one wavefront per 16 patterns and all categories): every category count,
lists that a workgroup stages and longer ones, ragged ends, NORM and SAFE with forced rescaling.
FP64 against the category-split kernel and the oracle: logL and per-pattern logL 1e-10
relative, derivatives 1e-9, scale counts equal.  FP32: the same sums in the same order as
the category-split kernel, so equal to the bit.  A batch equals its contexts alone."""
import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


def rel(a, b):
    return abs(a - b) / max(abs(b), 1e-300)


@pytest.mark.parametrize("form", ["norm", "safe", "fp32"])
@pytest.mark.parametrize("ncat", [1, 2, 3, 4, 5, 8])
@pytest.mark.parametrize("ntaxa,depth", [(9, 0), (150, 1)], ids=["staged", "long"])
def test_forms(ntaxa, depth, ncat, form):
    rng = np.random.default_rng(ncat)
    tree = S.caterpillar_tree(ntaxa, 1.5) if depth else None
    p = S.make_problem(4, ntaxa, 131, rng, ncat=ncat, mean_len=0.3, ambiguous=0.05, tree=tree, compress=False)
    print("4 states", ntaxa, ncat, form, flush=True)
    safe, prec = form == "safe", G.FP32 if form == "fp32" else G.FP64
    g, h = G.Tree(p, scaling=safe, precision=prec), G.Tree(p, scaling=safe, precision=prec)
    h.set_level_waves(0)
    o = S.Oracle(p, safe=safe, nthreads=8)
    top = 0
    for a, w in [(0, int(p.nei[0, 0]))] + [(int(p.nei[w, 0]), w) for w in range(ntaxa, 2 * ntaxa - 2, max(1, ntaxa // 4))]:
        lg, pg = g.loglik(a, w, with_patterns=True)
        lh, ph = h.loglik(a, w, with_patterns=True)
        lo, po = o.loglik(a, w, with_patterns=True)
        if form == "fp32":
            assert lg == lh and np.array_equal(pg, ph) and rel(lg, lo) <= 1e-6
            continue
        assert rel(lg, lo) <= 1e-10 and rel(lg, lh) <= 1e-10
        np.testing.assert_allclose(pg, po, rtol=1e-10, atol=1e-10)
        for x, y in zip(g.derivs(a, w)[:2], o.derivs(a, w)[:2]):
            assert abs(x - y) <= 1e-9 * max(1.0, abs(y))
        _, sg = g.partial(a, w, safe=safe)
        _, sh = h.partial(a, w, safe=safe)
        assert np.array_equal(sg, sh)
        top = max(top, int(sg.max()))
    assert form == "fp32" or top >= depth
    g.close()
    h.close()


@pytest.mark.parametrize("form", ["norm", "safe", "fp32"])
def test_batch_equals_alone(form):
    rng = np.random.default_rng(6)
    probs = [S.make_problem(4, taxa, sites, rng, ncat=ncat, ambiguous=0.03, compress=False)
             for taxa, sites, ncat in [(9, 1, 4), (70, 65, 1), (9, 700, 2), (140, 129, 3), (30, 64, 4)]]
    safe, prec = form == "safe", G.FP32 if form == "fp32" else G.FP64
    trees = [G.Tree(p, scaling=safe, precision=prec) for p in probs]
    batch = G.Batch(trees)
    for waves in (-1, 0, -1):  # switched on the live batch
        trees[2].set_level_waves(waves)
        alone = np.array([t.full_traversal() for t in trees])
        for _ in range(3):
            vals, _ = batch.loglik([(0, int(p.nei[0, 0])) for p in probs], clear=True)
            assert np.array_equal(vals, alone), waves
    batch.close()
