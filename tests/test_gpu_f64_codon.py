"""FP64 61-state traversal on the matrix cores: every category count, NORM (the categories of four
patterns meet at a barrier) and SAFE, ragged ends, more units than workgroups that stay on the
device, and forced rescaling, against the vector form and the oracle: logL 1e-10 relative,
derivatives 1e-9, scale counts equal (patterns one by one are compared in test_gpu_f64_mfma.py)."""
import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


def rel(a, b):
    return abs(a - b) / max(abs(b), 1e-300)


def check(p, safe, depth):
    g, h = G.Tree(p, scaling=safe), G.Tree(p, scaling=safe)
    h.set_f64_form(0)
    o = S.Oracle(p, safe=bool(safe), nthreads=8)
    T, top = p.ntaxa, 0
    for a, w in [(0, int(p.nei[0, 0])), (int(p.nei[T + 1, 0]), T + 1)]:
        lg, lo = g.loglik(a, w), o.loglik(a, w)
        assert rel(lg, lo) <= 1e-10 and rel(lg, h.loglik(a, w)) <= 1e-10
        for x, y in zip(g.derivs(a, w)[:2], o.derivs(a, w)[:2]):
            assert abs(x - y) <= 1e-9 * max(1.0, abs(y))
    for w in range(T, 2 * T - 2, max(1, (T - 2) // 4)):
        d = int(p.nei[w, 0])
        _, sg = g.partial(d, w, safe=bool(safe))
        _, so = o.partial(d, w, safe=bool(safe))
        assert np.array_equal(sg, so)
        top = max(top, int(so.max()))
    assert top >= depth
    g.close()
    h.close()


@pytest.mark.parametrize("safe", [0, 1], ids=["norm", "safe"])
@pytest.mark.parametrize("ncat,nptn", [(1, 65), (2, 17), (3, 131), (4, 1), (4, 2500), (5, 66), (8, 33)])
def test_categories(ncat, nptn, safe):
    # (2,500 patterns: 160 units of 16 patterns x 4 categories = 640, above two a compute unit)
    rng = np.random.default_rng(10 * ncat + nptn)
    p = S.make_problem(61, 6, nptn, rng, ncat=ncat, mean_len=0.4, ambiguous=0.05, compress=False)
    print("61 states", ncat, nptn, safe, flush=True)
    check(p, safe, 0)


@pytest.mark.parametrize("safe", [0, 1], ids=["norm", "safe"])
@pytest.mark.parametrize("ncat", [1, 4, 6])
def test_forced_rescaling(ncat, safe):
    rng = np.random.default_rng(ncat)
    p = S.make_problem(61, 70, 40, rng, ncat=ncat, tree=S.caterpillar_tree(70, 1.5), ambiguous=0.05)
    print("61 states rescaling", ncat, safe, flush=True)
    check(p, safe, 1)
