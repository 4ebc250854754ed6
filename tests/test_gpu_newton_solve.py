"""A branch solve in one launch (dev_newton.h): sizes around a tile, a workgroup of four tiles and
the launch rule, every state count and wide category counts.  The solve takes the steps of
minimizeNewton driven from the host and adds in the same order, so lengths and evaluation
counts are equal to the bit; the many-branch form gives the same lengths whatever the
number of branches of the launches before it."""
import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu

# (states, patterns, categories): one tile and its edges; eight categories with one workgroup per
# tile up to 128 tiles, four tiles each with a remainder, the last size of that form
# (512 tiles), and past it
CASES = [(4, 1, 4), (4, 64, 1), (4, 65, 5), (4, 128 * 64, 8), (4, 128 * 64 + 1, 8), (4, 130 * 64 - 3, 8),
         (4, 512 * 64, 8), (4, 512 * 64 + 1, 8), (20, 63, 1), (20, 200, 4), (20, 129, 8), (61, 65, 1), (61, 70, 8)]


@pytest.mark.parametrize("form", ["norm", "safe", "fp32"])
@pytest.mark.parametrize("n,nptn,ncat", CASES)
def test_one_launch_equals_host_loop(n, nptn, ncat, form):
    p = S.make_problem(n, 5, nptn, np.random.default_rng(nptn + ncat), ncat=ncat, mean_len=0.3, compress=False)
    print("newton solve", n, nptn, ncat, form, flush=True)
    kw = {"scaling": form == "safe", "precision": G.FP32 if form == "fp32" else G.FP64}
    dev, host = G.Tree(p, **kw), G.Tree(p, **kw)
    host.set_newton(False)
    for u, v in [(0, int(p.nei[0, 0])), (5, int(max(p.nei[5])))]:
        assert dev.optimize_one(u, v) == host.optimize_one(u, v)
    assert dev.counters()[1] == host.counters()[1]


def test_many_branches_after_fewer():
    p = S.make_problem(4, 12, 500, np.random.default_rng(3), mean_len=0.2, compress=False)
    g = G.Tree(p, all_directions=True)
    br, _, _ = g.all_branch_derivs()

    def ref(frm, to):
        return -(to + 1) if to < p.ntaxa else 3 * (to - p.ntaxa) + [int(x) for x in p.nei[to]].index(frm)

    refs = [(ref(v, u), ref(u, v)) for u, v in br]
    guess = [g.get_length(u, v) for u, v in br]
    first, logl, _ = g.newton_multi(refs, guess)
    for k in (3, 1, len(refs), 7, len(refs)):
        out, lg, st = g.newton_multi(refs[:k], guess[:k])
        assert np.all(st == 0) and np.array_equal(out, first[:k]) and np.array_equal(lg, logl[:k])


def test_ended_waits_give_the_same_solves():
    """With waits of no length the solves go on with one launch per evaluation; the exchange
    places are clean for the next solve."""
    p = S.make_problem(4, 12, 3000, np.random.default_rng(4), mean_len=0.2, compress=False)
    g, h = G.Tree(p, all_directions=True), G.Tree(p, all_directions=True)
    br, _, _ = g.all_branch_derivs()
    h.all_branch_derivs()

    def ref(frm, to):
        return -(to + 1) if to < p.ntaxa else 3 * (to - p.ntaxa) + [int(x) for x in p.nei[to]].index(frm)

    refs = [(ref(v, u), ref(u, v)) for u, v in br]
    guess = [g.get_length(u, v) for u, v in br]
    first, logl, _ = g.newton_multi(refs, guess)
    assert G.lib().plk_set_solve_wait(h.context(), -1) == -1
    for wait in (0, 20000, 0):
        assert G.lib().plk_set_solve_wait(h.context(), wait) == 0
        out, lg, st = h.newton_multi(refs, guess)
        assert np.all(st == 0) and np.array_equal(out, first) and np.array_equal(lg, logl)
    for k, (u, v) in enumerate(br[:6]):
        assert G.lib().plk_set_solve_wait(h.context(), 20000 * (k % 2)) == 0
        assert g.optimize_one(u, v) == h.optimize_one(u, v)
