"""FP32 61 states: a tile run as four 16-pattern units (while all are resident: up to 128 tiles with 4
categories, 64 with more, on 256 compute units; the last two sizes lie beyond) against the
pattern-block shape (up to 4 categories: equal to the bit) and the oracle (1e-6)."""
import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncat,nptn", [(1, 17), (4, 1), (4, 300), (6, 40), (4, 8300), (6, 4200)])
def test_units_match_whole_tiles(ncat, nptn):
    p = S.make_problem(61, 6, nptn, np.random.default_rng(ncat + nptn), ncat=ncat, mean_len=0.4, ambiguous=0.05,
                       compress=False)
    print("61 states fp32", ncat, nptn, flush=True)
    g = G.Tree(p, precision=G.FP32)
    v = g.full_traversal()
    want = S.Oracle(p, nthreads=8).loglik(0, int(p.nei[0, 0]))
    assert abs(v - want) <= 1e-6 * abs(want)
    if ncat <= 4:
        g.set_tile_shape(0)
        assert g.full_traversal() == v
    g.close()


@pytest.mark.parametrize("ncat", [1, 4, 8])
def test_few_jobs_give_the_same_matrices(ncat):
    """P(t) of a few ops at a time (a workgroup per 16 rows) and of the whole list (matrix cores)
    are equal to the bit."""
    p = S.make_problem(61, 40, 30, np.random.default_rng(ncat), ncat=ncat, mean_len=0.2, ambiguous=0.05, compress=False)
    print("61 states fp32 P(t)", ncat, flush=True)
    g = G.Tree(p, precision=G.FP32)
    v = g.full_traversal()
    for u in range(40, 78, 9):
        w = int(p.nei[u, 0])
        t = g.get_length(u, w)
        g.set_length(u, w, 2 * t)
        assert g.compute_likelihood() != v
        g.set_length(u, w, t)
        assert g.compute_likelihood() == v
    g.close()
