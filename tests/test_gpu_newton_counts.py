"""Which way the Newton solves went (plk_get_solve_counts): in one launch wherever the launch
rule takes them, never beyond it, and on by one launch per evaluation where a wait ends."""
import ctypes

import numpy as np
import pytest

import gems_amd as G
import support as S

pytestmark = pytest.mark.gpu


def counts(t):
    one, ended = ctypes.c_int64(), ctypes.c_int64()
    assert G.lib().plk_get_solve_counts(t.context(), ctypes.byref(one), ctypes.byref(ended)) == 0
    return one.value, ended.value


# (states, patterns, categories, in one launch): 256 compute units; 4 states take up to 1,024
# tiles of four categories and 512 of eight, 20 states 256 and 128, 61 states 128 and 64
CASES = [(4, 1, 4, True), (4, 5000, 1, True), (4, 1024 * 64, 4, True), (4, 1024 * 64 + 1, 4, False), (4, 512 * 64, 8, True),
         (4, 512 * 64 + 1, 8, False), (20, 256 * 64, 4, True), (20, 256 * 64 + 1, 4, False), (61, 128 * 64, 4, True),
         (61, 128 * 64 + 1, 4, False)]


@pytest.mark.skipif(G.device_count() > 0 and G.device_units() != 256, reason="sizes of 256 compute units")
@pytest.mark.parametrize("n,nptn,ncat,fits", CASES)
def test_one_launch_where_the_rule_says(n, nptn, ncat, fits):
    p = S.make_problem(n, 5, nptn, np.random.default_rng(nptn), ncat=ncat, mean_len=0.3, compress=False)
    print("solve counts", n, nptn, ncat, flush=True)
    t = G.Tree(p, all_directions=2)
    assert counts(t) == (0, 0)
    for u, v in [(0, int(p.nei[0, 0])), (5, int(max(p.nei[5])))]:
        t.optimize_one(u, v)
    assert counts(t) == (2 if fits else 0, 0)
    t.nni_evaluate([(u, int(v)) for u in range(5, 8) for v in p.nei[u] if v > u])
    one, ended = counts(t)
    assert ended == 0 and (one >= 2 + 4 * 5 if fits else one == 0)


def test_ended_waits_are_counted_and_stop_the_tries():
    p = S.make_problem(4, 12, 3000, np.random.default_rng(4), mean_len=0.2, compress=False)
    t, h = G.Tree(p), G.Tree(p)
    h.set_newton(False)
    edges = [(u, int(v)) for u in range(22) for v in p.nei[u] if v > u]
    assert G.lib().plk_set_solve_wait(t.context(), 0) == 0
    for e in edges:
        assert t.optimize_one(*e) == h.optimize_one(*e)
    one, ended = counts(t)
    assert ended >= 1 and one + ended < len(edges)
    assert G.lib().plk_set_solve_wait(t.context(), 20000) == 0
    for e in edges:
        assert t.optimize_one(*e) == h.optimize_one(*e)
    assert counts(t) == (one + len(edges), ended)
