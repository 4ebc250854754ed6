"""4 states with five to eight categories, where a workgroup's LDS holds fewer buffers or no P(t)
data: gradients, NNI moves and logL on random trees.  FP64 against the oracle (derivatives and
scores 1e-9 relative, lengths 2e-6); FP32 against the category-split kernel, which forms the
same sums in the same order, so equal to the bit."""
import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["norm", "safe", "fp32"])
@pytest.mark.parametrize("ncat", [5, 6, 8])
@pytest.mark.parametrize("ntaxa", [12, 20, 40])
def test_gradient_and_moves(ntaxa, ncat, form):
    p = G.Problem(G.SEQ_DNA, ntaxa, 700, ncat=ncat, seed=ntaxa + ncat)
    print("4 states, categories", ntaxa, ncat, form, flush=True)
    kw = {"scaling": form == "safe", "precision": G.FP32 if form == "fp32" else G.FP64, "all_directions": 2}
    inner = [(u, int(v)) for u in range(ntaxa, 2 * ntaxa - 2) for v in p.nei[u] if v > u]
    g = G.Tree(p, **kw)
    br, df, ddf = g.all_branch_derivs()
    scores, lens = g.nni_evaluate(inner)
    if form == "fp32":
        h = G.Tree(p, **kw)
        h.set_level_waves(0)
        _, df2, ddf2 = h.all_branch_derivs()
        scores2, lens2 = h.nni_evaluate(inner)
        for x, y in ((df, df2), (ddf, ddf2), (scores, scores2), (lens, lens2)):
            assert np.array_equal(x, y)
        return
    o = S.Oracle(p, safe=form == "safe", nthreads=8)
    for (u, v), x, y in zip(br, df, ddf):
        d1, d2, _ = o.derivs(u, v)
        assert abs(x - d1) <= 1e-9 * max(1.0, abs(d1)) and abs(y - d2) <= 1e-9 * max(1.0, abs(d2)), (u, v)
    for i in range(0, len(inner), max(1, len(inner) // 6)):
        for m in (0, 1):
            so, lo = o.nni_eval(*inner[i], m)
            assert abs(scores[i, m] - so) <= 1e-9 * abs(so), (inner[i], m)
            assert np.all(np.abs(lens[i, m] - lo) <= 2e-6 * np.maximum(1.0, lo)), (inner[i], m)


@pytest.mark.parametrize("ncat", [5, 8])
@pytest.mark.parametrize("ntaxa", [34, 37, 38, 39, 40, 41, 42, 63, 64, 65])
def test_fp32_logl_around_the_staging_limit(ntaxa, ncat):
    p = S.make_problem(4, ntaxa, 200, np.random.default_rng(ntaxa), ncat=ncat, ambiguous=0.03, compress=False)
    print("4 states, staging limit", ntaxa, ncat, flush=True)
    g, h = G.Tree(p, precision=G.FP32), G.Tree(p, precision=G.FP32)
    h.set_level_waves(0)
    lg, pg = g.loglik(0, int(p.nei[0, 0]), with_patterns=True)
    lh, ph = h.loglik(0, int(p.nei[0, 0]), with_patterns=True)
    assert lg == lh and np.array_equal(pg, ph)
    assert abs(lg - S.Oracle(p).loglik(0, int(p.nei[0, 0]))) <= 1e-6 * abs(lg)
