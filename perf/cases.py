"""Performance cases of the likelihood engine: what a phylogenetics program has it do.

A case is one alignment (or a set of them) on a tree and one call, or one short sequence of
calls, of the public API (gems_amd, the C ABI behind it):

  logl      full post-order traversal of a tree + branch logL (computeLikelihood after a model
            or topology change), FP64 or FP32 form, with or without the site-wise logL
  gradient  df/ddf of every branch for new branch lengths: both directions of every branch
  newton    one optimizeAllBranches round on a candidate tree (device-resident Newton)
  nni       both NNI moves of every internal branch, five branch solves each
  batch     logL of many unlinked partitions at once
  rell      logL of a candidate tree, then RELL scores of the bootstrap replicates
  serve     a burst of requests through the serving loop

The alignments are simulated along a random Yule tree under the model they are evaluated with
(reversible, discrete Gamma), with a few percent of gaps and, for DNA, ambiguity codes, and
compressed to patterns; so sizes are in sites and the pattern counts come out odd.
"""
import math
import random
import types

import numpy as np
import torch

import gems_amd as G

DNA, PROTEIN, CODON = "dna", "protein", "codon"
STATES = {DNA: 4, PROTEIN: 20, CODON: 61}
SEQ = {DNA: G.SEQ_DNA, PROTEIN: G.SEQ_PROTEIN, CODON: G.SEQ_CODON}
UNKNOWN = {DNA: 18, PROTEIN: 23, CODON: 61}
GAMMA_SHAPE = {DNA: 0.5, PROTEIN: 0.8, CODON: 0.5}
MEAN_LENGTH = {DNA: 0.1, PROTEIN: 0.2, CODON: 0.1}


def device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# --------------------------------------------------------------------------------------
# the cases

def listed():
    def logl(name, data, taxa, sites, precision, safe=False, sitewise=False, ncat=4, pinv=0.0):
        return {"name": name, "kind": "logl", "data": data, "taxa": taxa, "sites": sites, "precision": precision,
                "safe": safe, "sitewise": sitewise, "ncat": ncat, "pinv": pinv}

    return [
        # a single gene of a small study: the smallest call, all latency
        logl("dna_gene", DNA, 12, 400, "fp64"),
        # an ordinary DNA data set (32 taxa, 10,000 sites)
        logl("dna_ordinary", DNA, 32, 10000, "fp64"),
        # the largest request of a serving mix: 512 taxa, 100,000 sites
        logl("dna_large_fp32", DNA, 512, 100000, "fp32"),
        # the benchmark's protein problem in both forms; the FP64 one with the site-wise logL
        # that topology tests read
        logl("protein_fp32", PROTEIN, 100, 50000, "fp32"),
        logl("protein_fp64", PROTEIN, 100, 50000, "fp64", sitewise=True),
        # the codon problem in both forms (FP64 in the SAFE scaling mode codon runs use)
        logl("codon_fp64", CODON, 48, 5000, "fp64", safe=True, sitewise=True),
        logl("codon_fp32", CODON, 48, 5000, "fp32"),
        # one gradient of a branch-length optimiser on a protein gene set
        {"name": "protein_gradient", "kind": "gradient", "data": PROTEIN, "taxa": 50, "sites": 4000, "precision": "fp64",
         "safe": False, "ncat": 4},
        # a candidate tree of a tree search: one round of branch-length optimisation
        {"name": "dna_newton", "kind": "newton", "data": DNA, "taxa": 64, "sites": 5000, "precision": "fp64", "safe": False,
         "ncat": 4},
        # the NNI neighbourhood of a tree during the search
        {"name": "dna_nni", "kind": "nni", "data": DNA, "taxa": 40, "sites": 3000, "precision": "fp64", "safe": False,
         "ncat": 4},
        # a phylogenomic data set of 300 unlinked genes on 64 taxa, 70 % DNA, 30 % protein
        {"name": "genes_300", "kind": "batch", "taxa": 64, "genes": 300, "protein": 0.3, "precision": "fp64"},
        # a burst of eight requests: DNA and protein, half of them with a branch optimisation
        {"name": "serve_8", "kind": "serve", "requests": 8, "max_taxa": 128, "max_sites": 20000, "precision": "fp64"},
    ]


def spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["logl"] * 6 + ["gradient", "newton", "nni", "batch", "rell", "serve"])
    data = rng.choice([DNA, PROTEIN, CODON]) if kind == "logl" else rng.choice([DNA, DNA, PROTEIN])
    ncat = rng.choice([4, 4, 4, 4, 1, 2, 3, 6, 8])
    safe = rng.random() < 0.3
    if kind == "logl":
        most_taxa, most_sites, cells = {DNA: (512, 100000, 4e7), PROTEIN: (200, 50000, 4e6), CODON: (64, 6000, 2e5)}[data]
        taxa = spread(rng, 6, most_taxa)
        sites = spread(rng, 120, min(most_sites, cells * 4 / max(ncat, 4) / taxa))
        precision = rng.choice(["fp64", "fp32"])
        pinv = rng.choice([0.0, 0.0, 0.0, 0.2]) if data == DNA else 0.0
        return {"kind": kind, "data": data, "taxa": taxa, "sites": sites, "precision": precision, "safe": safe,
                "sitewise": precision == "fp64" and rng.random() < 0.5, "ncat": ncat, "pinv": pinv}
    if kind in ("gradient", "newton", "nni"):
        most = {"gradient": (60, 5000), "newton": (64, 6000), "nni": (40, 4000)}[kind]
        return {"kind": kind, "data": data, "taxa": spread(rng, 6, most[0] if data == DNA else most[0] // 2),
                "sites": spread(rng, 150, most[1] if data == DNA else most[1] // 2), "precision": "fp64", "safe": safe,
                "ncat": rng.choice([4, 4, 4, 2, 6])}
    if kind == "batch":
        return {"kind": kind, "taxa": spread(rng, 8, 64), "genes": spread(rng, 8, 300),
                "protein": rng.choice([0.0, 0.3, 0.5]), "precision": "fp64"}
    if kind == "rell":
        return {"kind": kind, "data": data, "taxa": spread(rng, 8, 64), "sites": spread(rng, 400, 30000),
                "replicates": spread(rng, 100, 1000), "precision": "fp64", "safe": False, "ncat": 4}
    return {"kind": kind, "requests": rng.randint(2, 8), "max_taxa": spread(rng, 24, 128),
            "max_sites": spread(rng, 1500, 20000), "precision": rng.choice(["fp64", "fp32"])}


# --------------------------------------------------------------------------------------
# models, trees and alignments

CODE = "FFLLSSSSYY**CC*WLLLLPPPPHHQQRRRRIIIMTTTTNNKKSSRRVVVVAAAADDEEGGGG"  # standard code, T C A G order


def exchangeabilities(data, rng):
    n = STATES[data]
    if data != CODON:
        e = rng.gamma(1.0, 1.0, (n, n)) + 0.02
        e = np.triu(e, 1)
        return e + e.T
    codons = [(a, b, c) for a in range(4) for b in range(4) for c in range(4) if CODE[16 * a + 4 * b + c] != "*"]
    kappa, omega = 2.0 + rng.random(), 0.2 + 0.2 * rng.random()
    e = np.zeros((n, n))
    for i, p in enumerate(codons):
        for j, q in enumerate(codons):
            diff = [k for k in range(3) if p[k] != q[k]]
            if len(diff) != 1:
                continue
            x, y = p[diff[0]], q[diff[0]]
            rate = kappa if {x, y} in ({0, 1}, {2, 3}) else 1.0  # T<->C, A<->G
            if CODE[16 * p[0] + 4 * p[1] + p[2]] != CODE[16 * q[0] + 4 * q[1] + q[2]]:
                rate *= omega
            e[i, j] = rate
    return e


def gamma_rates(shape, ncat):
    """Mean rates of ncat equally likely categories of a Gamma(shape) of mean 1."""
    if ncat == 1:
        return np.ones(1)
    a = torch.tensor(shape, dtype=torch.float64)
    q = torch.arange(1, ncat, dtype=torch.float64) / ncat
    lo, hi = torch.zeros_like(q), torch.full_like(q, 1000.0)
    for _ in range(200):
        mid = 0.5 * (lo + hi)
        below = torch.special.gammainc(a, mid) < q
        lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
    cum = torch.special.gammainc(a + 1.0, lo)
    edges = torch.cat([torch.zeros(1, dtype=torch.float64), cum, torch.ones(1, dtype=torch.float64)])
    r = ((edges[1:] - edges[:-1]) * ncat).numpy()
    return r / r.mean()


def model(data, ncat, rng, pinv=0.0):
    """Reversible model: eigen system U, lambda, U^-1, category rates and weights, tip vectors."""
    n, su = STATES[data], UNKNOWN[data]
    pi = rng.dirichlet(np.full(n, 5.0)) + 0.002
    pi /= pi.sum()
    q = exchangeabilities(data, rng) * pi[None, :]
    np.fill_diagonal(q, 0.0)
    np.fill_diagonal(q, -q.sum(1))
    q /= -(pi * np.diag(q)).sum()
    s = np.sqrt(pi)
    sym = s[:, None] * q / s[None, :]
    lam, v = np.linalg.eigh(0.5 * (sym + sym.T))
    lam[-1] = 0.0  # eigh sorts ascending: the last eigenvalue is the stationary one
    evec, inv = np.ascontiguousarray(v / s[:, None]), np.ascontiguousarray(v.T * s[None, :])
    real = np.ones((su + 1, n))
    real[:n] = np.eye(n)
    if data == DNA:
        for code in range(4, 18):
            real[code] = [(code - 3) >> j & 1 for j in range(4)]
    if data == PROTEIN:
        for code, pair in ((20, (2, 3)), (21, (5, 6)), (22, (9, 10))):
            real[code] = 0.0
            real[code, list(pair)] = 1.0
    shape = GAMMA_SHAPE[data] * (0.7 + 0.6 * rng.random())
    rates = gamma_rates(shape, ncat)
    return types.SimpleNamespace(data=data, n=n, su=su, seq_type=SEQ[data], pi=pi, eval=lam, evec=evec, inv_evec=inv,
                                 rates=rates / (1.0 - pinv), props=np.full(ncat, (1.0 - pinv) / ncat), ncat=ncat,
                                 tip_real=real, tip_lh=np.ascontiguousarray(real @ inv.T), pinv=pinv)


def yule(taxa, mean, rng):
    """Random binary tree, leaves 0..taxa-1: neighbour table (2 taxa - 2, 3) and branch lengths."""
    nei = np.full((2 * taxa - 2, 3), -1, dtype=np.int32)
    nei[taxa] = (0, 1, 2)
    nei[:3, 0] = taxa
    for leaf in range(3, taxa):
        new, old = taxa + leaf - 2, int(rng.integers(0, leaf))  # a leaf splits
        up = int(nei[old, 0])
        nei[up, list(nei[up]).index(old)] = new
        nei[new] = (up, old, leaf)
        nei[old, 0] = nei[leaf, 0] = new
    return nei, lengths(nei, mean, rng)


def lengths(nei, mean, rng):
    blen = np.zeros(nei.shape)
    for u in range(nei.shape[0]):
        for k in range(3):
            v = int(nei[u, k])
            if v > u:
                blen[u, k] = blen[v, list(nei[v]).index(u)] = rng.exponential(mean) + 1e-4
    return blen


def order(nei):
    """(parent, node) pairs in pre-order from leaf 0."""
    out, stack = [], [(0, int(nei[0, 0]))]
    while stack:
        dad, v = stack.pop()
        out.append((dad, v))
        stack += [(v, int(x)) for x in nei[v] if x >= 0 and x != dad]
    return out


def edge(nei, blen, u, v):
    return float(blen[u, list(nei[u]).index(v)])


def transition(m, lens, dev, derivative=0):
    """(len(lens), ncat, n, n) matrices d^k/dt^k exp(Q r_c t) in 64 bits."""
    t = torch.tensor(np.asarray(lens), dtype=torch.float64, device=dev)
    cof = torch.tensor(np.outer(m.rates, m.eval), device=dev)
    e = torch.exp(cof[None] * t[:, None, None]) * cof[None] ** derivative
    u, ui = torch.tensor(m.evec, device=dev), torch.tensor(m.inv_evec, device=dev)
    return torch.matmul(u[None, None] * e[:, :, None, :], ui.expand(len(lens), m.ncat, m.n, m.n).contiguous())


def alignment(m, nei, blen, sites, taxa, rng):
    """States simulated along the tree, as patterns: (taxa, nptn) uint8, their counts, each site's pattern."""
    dev = device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(rng.integers(1 << 40)))
    rand = lambda *shape: torch.rand(*shape, generator=gen, device=dev)  # noqa: E731
    pairs = order(nei)
    p = transition(m, [edge(nei, blen, u, v) for u, v in pairs], dev).clamp_(min=0).cumsum(-1).float()
    cat = (rand(sites) * m.ncat).long().clamp_(max=m.ncat - 1)
    fixed = rand(sites) < m.pinv
    root = torch.searchsorted(torch.tensor(np.cumsum(m.pi), dtype=torch.float32, device=dev), rand(sites))
    state = {0: root.clamp_(max=m.n - 1)}
    rows = torch.empty(taxa, sites, dtype=torch.long, device=dev)
    rows[0] = state[0]
    last = {}
    for k, (u, v) in enumerate(pairs):
        s = (rand(sites, 1) > p[k][cat, state[u]]).sum(-1).clamp_(max=m.n - 1)
        s = torch.where(fixed, state[u], s)
        if v < taxa:
            rows[v] = s
        else:
            state[v] = s
            last[v] = 2
        if u in last:
            last[u] -= 1
            if not last[u]:
                del state[u]
    if m.data == DNA:  # ambiguity codes that allow the true state (R, Y, ... as code = mask + 3)
        mask = (rand(taxa, sites) * 14).long() + 1
        mask |= torch.ones_like(rows) << rows
        single = (mask & (mask - 1)) == 0
        rows = torch.where((rand(taxa, sites) < 0.004) & ~single, mask + 3, rows)
    rows[rand(taxa, sites) < 0.02] = m.su
    weights = torch.randint(-(1 << 62), 1 << 62, (taxa,), generator=gen, device=dev)
    _, inverse, counts = torch.unique((rows * weights[:, None]).sum(0), return_inverse=True, return_counts=True)
    first = torch.full_like(counts, sites).scatter_reduce_(0, inverse, torch.arange(sites, device=dev), "amin")
    first, at = torch.sort(first)
    rank = torch.empty_like(at).scatter_(0, at, torch.arange(len(at), device=dev))
    return rows[:, first].to(torch.uint8).cpu().numpy(), counts[at].double().cpu().numpy(), rank[inverse].cpu().numpy()


def problem(data, taxa, sites, seed, ncat=4, pinv=0.0, tree=None):
    """What a program holds before it calls the engine; the attributes gems_amd.Tree reads."""
    rng = np.random.default_rng([abs(int(seed)), taxa, sites])
    m = model(data, ncat, rng, pinv)
    nei, blen = yule(taxa, MEAN_LENGTH[data], rng) if tree is None else (tree, lengths(tree, MEAN_LENGTH[data], rng))
    states, freq, m.site_pattern = alignment(m, nei, blen, sites, taxa, rng)
    m.ntaxa, m.nptn, m.nsites, m.states, m.freq, m.nei, m.blen, m.invar = taxa, states.shape[1], sites, states, freq, nei, blen, None
    if pinv:
        # invariant-site mass: p_inv times the frequency of the states every taxon allows
        allowed = np.ones((m.nptn, m.n), dtype=bool)
        for row in states:
            allowed &= m.tip_real[row] > 0
        m.invar = pinv * (allowed @ m.pi)
    return m


def gene_sizes(case, rng):
    """Lognormal gene lengths, median 500 sites, clipped to [100, 5000]."""
    out = []
    for _ in range(case["genes"]):
        data = PROTEIN if rng.random() < case["protein"] else DNA
        out.append((data, int(np.clip(round(rng.lognormal(math.log(500.0), 1.0)), 100, 5000))))
    return out


def genes(case, seed):
    # the sizes are the data set's own; the sequences, models and lengths come from the seed
    sizes = gene_sizes(case, np.random.default_rng([3, case["genes"], case["taxa"]]))
    tree = yule(case["taxa"], 0.1, np.random.default_rng([int(seed), 1]))[0]
    return [problem(data, case["taxa"], sites, 1000 * int(seed) + i, tree=tree) for i, (data, sites) in enumerate(sizes)]


def request_sizes(case):
    rng = random.Random(case["requests"] * 7919 + case["max_taxa"])
    return [(rng.choice([DNA, PROTEIN]), spread(rng, 16, case["max_taxa"]), spread(rng, 1000, case["max_sites"]), i % 2 == 1)
            for i in range(case["requests"])]


def requested(case, seed):
    return [problem(data, taxa, sites, 1000 * int(seed) + i) for i, (data, taxa, sites, _) in enumerate(request_sizes(case))]


def one_problem(case, seed):
    return problem(case["data"], case["taxa"], case["sites"], seed, case["ncat"], case.get("pinv", 0.0))


def replicates(case, p):
    """Bootstrap pattern counts: each replicate draws the alignment's sites with replacement."""
    dev, ns = device(), case["replicates"]
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(p.nptn) * 31 + int(p.states[:, 0].sum()))
    cum = torch.tensor(np.cumsum(p.freq), device=dev)
    counts = torch.zeros(ns, p.nptn, device=dev)
    for at in range(0, ns, 64):
        rows = min(64, ns - at)
        u = torch.rand(rows, p.nsites, generator=gen, device=dev, dtype=torch.float64) * p.nsites
        hit = torch.searchsorted(cum, u, right=True).clamp_(max=p.nptn - 1)
        flat = (hit + torch.arange(rows, device=dev)[:, None] * p.nptn).reshape(-1)
        counts[at:at + rows] = torch.bincount(flat, minlength=rows * p.nptn).reshape(rows, p.nptn).float()
    return counts.cpu().numpy()


# --------------------------------------------------------------------------------------
# the engine's side

def tree_of(p, case, directions=0):
    return G.Tree(p, precision=G.FP32 if case["precision"] == "fp32" else G.FP64,
                  scaling=G.SAFE if case.get("safe") else G.NORM, all_directions=directions)


def prepare(case, seed):
    kind = case["kind"]
    s = types.SimpleNamespace(case=case)
    if kind == "batch":
        s.trees = [tree_of(p, case) for p in genes(case, seed)]
        s.batch = G.Batch(s.trees)
        s.branches = [(0, int(t.p.nei[0, 0])) for t in s.trees]
        return s
    if kind == "serve":
        s.server = G.Server(nworkers=4)
        s.requests = [G.Request(p, kind=G.REQ_OPT_BRANCH if opt else G.REQ_LOGL,
                                precision=G.FP32 if case["precision"] == "fp32" else G.FP64,
                                opt_branch=(p.ntaxa, int(p.nei[p.ntaxa, 0])))
                      for p, (_, _, _, opt) in zip(requested(case, seed), request_sizes(case))]
        return s
    p = one_problem(case, seed)
    s.p, s.branch = p, (0, int(p.nei[0, 0]))
    s.tree = tree_of(p, case, {"gradient": 1, "nni": 2}.get(kind, 0))
    s.nei, s.blen = np.ascontiguousarray(p.nei), np.ascontiguousarray(p.blen)
    if kind == "rell":
        s.rell = G.Rell(replicates(case, p))
    if kind == "nni":
        s.internal = [(u, int(v)) for u in range(p.ntaxa, 2 * p.ntaxa - 2) for v in p.nei[u] if v > u]
    return s


def candidate(s):
    """Put a candidate tree (topology and branch lengths) in: every partial is out of date."""
    rc = G.lib().plk_tree_set_topology(s.tree.h, s.nei.ctypes.data_as(G._ip), s.blen.ctypes.data_as(G._dp))
    if rc:
        raise RuntimeError(f"plk_tree_set_topology: {rc}")


def run(s):
    kind = s.case["kind"]
    if kind == "logl":
        if not s.case["sitewise"]:
            return {"logl": s.tree.full_traversal()}
        G.lib().plk_tree_clear_all(s.tree.h)
        logl, per_pattern = s.tree.loglik(*s.branch, with_patterns=True)
        return {"logl": logl, "sites": per_pattern[s.p.site_pattern]}
    if kind == "gradient":
        candidate(s)
        _, df, ddf = s.tree.all_branch_derivs()
        return {"df": df, "ddf": ddf}
    if kind == "newton":
        candidate(s)
        logl = s.tree.optimize_all(iterations=1)
        pairs = order(s.nei)
        return {"logl": logl, "lengths": np.array([s.tree.get_length(u, v) for u, v in pairs])}
    if kind == "nni":
        candidate(s)
        scores, lens = s.tree.nni_evaluate(s.internal)
        return {"scores": scores, "lengths": lens}
    if kind == "batch":
        per_gene, total = s.batch.loglik(s.branches, clear=True)
        return {"logl": per_gene, "total": total}
    if kind == "rell":
        candidate(s)
        logl = s.tree.compute_likelihood()
        return {"logl": logl, "scores": s.rell.eval(s.tree.context())}
    for r in s.requests:
        s.server.submit(r)
    s.server.drain()
    done = [r.result() for r in s.requests]
    if any(d["status"] for d in done):
        raise RuntimeError("a request failed")
    opt = [d["opt_len"] for d, r in zip(done, s.requests) if r.r.kind == G.REQ_OPT_BRANCH]
    return {"before": [d["logl_before"] for d in done], "after": [d["logl_after"] for d in done], "length": opt}


# --------------------------------------------------------------------------------------
# what a pass cannot do without

def traversal_work(data, taxa, patterns, ncat, width, updates=None):
    """Tip states and pattern weights read, every partial written once; textbook pruning flops."""
    n = STATES[data]
    updates = (taxa - 2) if updates is None else updates
    return (updates * patterns * ncat * n * width + taxa * patterns + 16 * patterns,
            updates * patterns * ncat * (4 * n * n + n) + patterns * ncat * (2 * n * n + 3 * n))


def patterns_of(data, taxa, sites):
    """About how many patterns the simulated sites compress to (short trees repeat columns)."""
    few = {DNA: 0.35, PROTEIN: 0.15, CODON: 0.2}[data]
    return int(sites * (1.0 - few * math.exp(-taxa / 40.0)))


def work(case):
    kind, width = case["kind"], 4 if case["precision"] == "fp32" else 8
    if kind == "batch":
        sizes = [(data, case["taxa"], sites) for data, sites in gene_sizes(case, np.random.default_rng([3, case["genes"], case["taxa"]]))]
        w = [traversal_work(d, t, patterns_of(d, t, s), 4, width) for d, t, s in sizes]
    elif kind == "serve":
        w = [traversal_work(d, t, patterns_of(d, t, s), 4, width) for d, t, s, _ in request_sizes(case)]
        w += [(t * patterns_of(d, t, s), 0) for d, t, s, _ in request_sizes(case)]  # the alignment comes from the host
    else:
        data, taxa, ncat = case["data"], case["taxa"], case["ncat"]
        ptn, n = patterns_of(data, taxa, case["sites"]), STATES[data]
        branches = 2 * taxa - 3
        product = ptn * ncat * n  # one branch: node x dad partials
        if kind in ("logl", "rell"):
            w = [traversal_work(data, taxa, ptn, ncat, width)]
        if kind == "rell":
            w.append((4 * case["replicates"] * ptn + 8 * ptn, 2 * case["replicates"] * ptn))
        if kind == "gradient":
            w = [traversal_work(data, taxa, ptn, ncat, width, 3 * (taxa - 2)), (0, branches * product * 7)]
        if kind == "newton":
            # partials to the first branch, about one more per branch on the way through the
            # tree, and five evaluations of each branch's derivatives
            w = [traversal_work(data, taxa, ptn, ncat, width, 3 * (taxa - 2)), (branches * product * width, branches * 5 * product * 6)]
        if kind == "nni":
            moves = 2 * (taxa - 3)
            w = [traversal_work(data, taxa, ptn, ncat, width, 3 * (taxa - 2) + 6 * moves), (0, moves * 5 * 5 * product * 7)]
    return {"bytes": float(sum(b for b, _ in w)), "flops": float(sum(f for _, f in w))}


# --------------------------------------------------------------------------------------
# the same in 64 bits with plain torch

class Exact:
    """Felsenstein pruning of one problem in real space, renormalised at every node."""

    def __init__(self, p):
        self.p, self.dev = p, device()
        self.pairs = order(p.nei)
        self.lens = [edge(p.nei, p.blen, u, v) for u, v in self.pairs]
        self.mats = transition(p, self.lens, self.dev)
        self.tip = torch.tensor(p.tip_real, device=self.dev)
        self.pi = torch.tensor(p.pi, device=self.dev)
        self.props = torch.tensor(p.props, device=self.dev)
        self.rows = torch.tensor(p.states.astype(np.int64), device=self.dev)
        self.freq = torch.tensor(p.freq, device=self.dev)

    def across(self, mats, ref):
        """(ncat, nptn, n): the matrices of a branch times what hangs at its far end."""
        if isinstance(ref, int):
            table = torch.matmul(self.tip.expand(self.p.ncat, *self.tip.shape).contiguous(), mats.transpose(1, 2).contiguous())
            return table[:, self.rows[ref]]
        return torch.matmul(ref, mats.transpose(1, 2).contiguous())

    def down(self, keep=False):
        """Partials of every node's subtree seen from leaf 0 (all kept, or the last one only) and log scales."""
        self.kids = {}
        for k, (u, v) in enumerate(self.pairs):
            self.kids.setdefault(u, []).append((k, v))
        log = torch.zeros(self.p.nptn, dtype=torch.float64, device=self.dev)
        part = {}
        for u, v in reversed(self.pairs):
            if v < self.p.ntaxa:
                part[v] = v
                continue
            prod = None
            for k, x in self.kids[v]:
                a = self.across(self.mats[k], part[x] if keep else part.pop(x))
                prod = a if prod is None else prod * a
            top = prod.amax(2).amax(0)
            part[v] = prod / top[None, :, None]
            log += torch.log(top)
        return part, log

    def patterns(self):
        part, log = self.down()
        v = self.pairs[0][1]
        far = self.across(self.mats[0], part[v])
        lh = (self.tip[self.rows[0]][None] * far * self.pi).sum(2)
        logl = torch.log((self.props[:, None] * lh).sum(0)) + log
        if self.p.invar is not None:
            logl = torch.logaddexp(logl, torch.log(torch.tensor(self.p.invar, device=self.dev)))
        return logl

    def logl(self):
        return float((self.patterns() * self.freq).sum())

    def gradient(self):
        part, _ = self.down(keep=True)
        d1, d2 = transition(self.p, self.lens, self.dev, 1), transition(self.p, self.lens, self.dev, 2)
        rest, found = {0: 0}, {}  # rest[k]: what the branch's upper end sees, without the branch
        for k, (u, v) in enumerate(self.pairs):
            up = rest.pop(k)
            near = self.tip[self.rows[up]][None] if isinstance(up, int) else up
            lh, l1, l2 = ((self.props[:, None] * (near * self.across(m[k], part[v]) * self.pi).sum(2)).sum(0)
                          for m in (self.mats, d1, d2))
            g = l1 / lh
            found[min(u, v), max(u, v)] = (float((self.freq * g).sum()), float((self.freq * (l2 / lh - g * g)).sum()))
            for j, x in self.kids.get(v, []):
                r = self.across(self.mats[k], up)
                for i, y in self.kids[v]:
                    if y != x:
                        r = r * self.across(self.mats[i], part[y])
                rest[j] = r / r.amax(2).amax(0)[None, :, None]
        pairs = [(u, int(v)) for u in range(self.p.nei.shape[0]) for v in self.p.nei[u] if v > u]
        return {"df": np.array([found[e][0] for e in pairs]), "ddf": np.array([found[e][1] for e in pairs])}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("newton", "nni"):
        return None  # iterative searches
    if kind == "batch":
        per_gene = np.array([Exact(p).logl() for p in genes(case, seed)])
        return {"logl": per_gene, "total": float(per_gene.sum())}
    if kind == "serve":
        logl = [Exact(p).logl() for p in requested(case, seed)]
        opt = [r[3] for r in request_sizes(case)]
        return {"before": logl, "after": [None if o else v for v, o in zip(logl, opt)], "length": [None for o in opt if o]}
    p = one_problem(case, seed)
    if kind == "gradient":
        return Exact(p).gradient()
    per_pattern = Exact(p).patterns()
    logl = float((per_pattern * torch.tensor(p.freq, device=per_pattern.device)).sum())
    if kind == "rell":
        counts = torch.tensor(replicates(case, p), dtype=torch.float64, device=per_pattern.device)
        return {"logl": logl, "scores": (counts * per_pattern.float().double()).sum(1).cpu().numpy()}
    if not case["sitewise"]:
        return {"logl": logl}
    return {"logl": logl, "sites": per_pattern.cpu().numpy()[p.site_pattern]}
