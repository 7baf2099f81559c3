"""Timed cases of the PMM engine, through its public entry points.

Every case is the work of one call (or one short sequence of calls) that a
program built on this package makes: a likelihood, an EM run, a gradient, an
E-step with posteriors, a quartet-local NNI round, a served request.  Sizes
are those of the benchmark's and the tests' workloads: 250 leaves x 30 sites
up to 50,000 leaves x 500 sites, alphabets of 2 to 60 states, EM from the
uniform start (branches 0.05, nu = phi = 0.5).

Inputs are made from the seed alone: random binary trees with uniform splits
(the Yule model's), priors Dirichlet(1) per site, characters simulated under
the PMM model.  ``exact`` evaluates the same model in plain torch in 64 bits:
the two-value form of the inside pass, its adjoint by hand, the M-step by
bisection.
"""
import math

import numpy as np
import torch

from laml_amd import sim
from laml_amd.autograd import neg_log_likelihood
from laml_amd.forest import Forest, SiteTable
from laml_amd.serving import SolveRequest, solve_alone
from laml_amd.ultra import HeightModel

DMIN, DMAX = 0.005, 10.0
TRUE_NU, TRUE_PHI = 0.1, 0.1
M_LO, M_HI = 5, 60


def _case(name, kind, leaves, sites, problems=1, variants=0, leaves_lo=0, iters=5, tol=0.0):
    """leaves_lo: 0, or the smallest tree of a batch whose sizes are spread
    up to ``leaves``; variants: NNI variants of one tree of ``leaves`` leaves
    that a batch holds besides its ``problems`` trees."""
    c = dict(kind=kind, leaves=leaves, sites=sites, problems=problems, variants=variants, leaves_lo=leaves_lo,
             iters=iters, tol=tol)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one likelihood of a small lineage tree: the smallest call (a user's own
        # optimiser or a parameter scan makes it many times)
        _case("nll 250x30", "nll", 250, 30),
        # EM of a small tree until it converges: the ordinary interactive fit
        _case("em 250x30", "em", 250, 30, iters=1000, tol=1e-8),
        # the same tree under the ultrametric constraint (the command line's
        # usual setting), five EM steps
        _case("em ultrametric 250x30", "ultra", 250, 30),
        # E-step and posteriors to the host: the annotation output of a fit
        _case("posteriors 1000x100", "post", 1000, 100),
        # a served request from host data to host results: forest, EM, results
        _case("solve 2000x150", "solve", 2000, 150, iters=50, tol=1e-8),
        # one quartet-local round over all NNI moves of a tree
        _case("nni round 2000x200", "quartet", 2000, 200, iters=1000, tol=1e-8),
        # many small trees in one forest, sites that fill no wavefront
        _case("em 200 small trees x20", "em", 200, 20, problems=200, leaves_lo=20, iters=20),
        # batched scoring of NNI variants and unrelated trees of ragged sizes
        _case("em scoring 96 trees x200", "em", 2000, 200, problems=32, variants=64, leaves_lo=100, iters=10,
              tol=1e-8),
        # value and gradient of a large tree (gradient-based optimisers)
        _case("gradient 10000x300", "grad", 10000, 300),
        # the headline tree alone, and the headline batch of sixteen
        _case("em 10000x300", "em", 10000, 300, iters=10),
        _case("em 16 trees 10000x300", "em", 10000, 300, problems=16),
        # the largest request of the serving workload
        _case("em 50000x500", "em", 50000, 500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["nll", "em", "em", "em", "batch", "batch", "grad", "post", "solve", "quartet", "ultra"])
    sites = _log_int(rng, 15, 500)
    if kind == "ultra":
        return _case(None, "ultra", _log_int(rng, 30, 400), min(sites, 150), iters=rng.randint(2, 5))
    if kind == "batch":
        hi = _log_int(rng, 60, 5000)
        problems = max(2, min(_log_int(rng, 4, 200), 6_000_000 // (hi * sites)))
        variants = rng.choice([0, 0, problems]) if problems <= 60 else 0
        return _case(None, "em", hi, sites, problems=problems, variants=variants,
                     leaves_lo=rng.choice([max(10, hi // 10), hi]), iters=rng.randint(3, 12), tol=1e-8)
    if kind == "quartet":
        return _case(None, "quartet", _log_int(rng, 100, 2000), min(sites, 300), iters=1000, tol=1e-8)
    if kind in ("post", "solve"):
        return _case(None, kind, _log_int(rng, 100, 5000), min(sites, 250), iters=rng.randint(20, 60), tol=1e-8)
    leaves = min(_log_int(rng, 50, 40000), 15_000_000 // sites)
    if kind in ("nll", "grad"):
        return _case(None, kind, leaves, sites)
    return _case(None, "em", leaves, sites, iters=rng.randint(3, 12))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")


def _random_tree(n, rng):
    """Binary tree of n leaves with uniform split sizes, post-order arrays,
    branch lengths that shrink with the clade; and every node's depth."""
    N = 2 * n - 1
    c0, c1 = np.full(N, -1, np.int64), np.full(N, -1, np.int64)
    parent, length, depth = np.full(N, -1, np.int64), np.full(N, 0.05), np.zeros(N, np.int64)
    m, lo = np.array([n]), np.array([0])  # clade sizes and first post-order ids of one depth
    dep, scale = 0, 1.0 / math.log(n)
    while len(m):
        inner = m > 1
        m, lo = m[inner], lo[inner]
        if not len(m):
            break
        dep += 1
        left = 1 + (rng.random(len(m)) * (m - 1)).astype(np.int64)
        v = lo + 2 * m - 2
        a, b = lo + 2 * left - 2, lo + 2 * m - 3
        c0[v], c1[v] = a, b
        for ch, sz in ((a, left), (b, m - left)):
            parent[ch] = v
            depth[ch] = dep
            length[ch] = (np.log(m / sz) + 0.05) * scale * rng.gamma(2.0, 0.5, len(m))
        m, lo = np.concatenate([left, m - left]), np.concatenate([lo, lo + 2 * left - 1])
    return sim.YuleTree(c0, c1, parent, np.maximum(length, 2 * DMIN), ["c%d" % i for i in range(n)]), depth


def _priors(K, rng):
    sizes = rng.integers(M_LO, M_HI + 1, K)
    out = []
    for m in sizes:
        q = rng.exponential(1.0, int(m))
        q /= q.sum()
        out.append({j + 1: float(x) for j, x in enumerate(q)})
    return out


def _simulate(trees, depths, Qs, seed):
    """Leaf codes of all trees at once (int16, a matrix per tree)."""
    dev = _device()
    K, P = len(Qs[0]), len(trees)
    cum = np.ones((P, K, M_HI))
    for p, Q in enumerate(Qs):
        for k, q in enumerate(Q):
            c = np.cumsum(np.fromiter(q.values(), float, len(q)))
            cum[p, k, :len(q)] = c / c[-1]
    rows = torch.as_tensor(cum.reshape(P * K, M_HI), device=dev)
    flat = (rows + torch.arange(P * K, device=dev)[:, None]).reshape(-1).contiguous()
    base = np.concatenate([[0], np.cumsum([t.n_nodes for t in trees])])
    par = np.concatenate([np.where(t.parent >= 0, t.parent + b, -1) for t, b in zip(trees, base)])
    prob = np.repeat(np.arange(P), np.diff(base))
    dep = np.concatenate(depths)
    order = np.argsort(dep, kind="stable")
    cuts = np.searchsorted(dep[order], np.arange(dep.max() + 2))
    T = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
    length, par_t, prob_t = T(np.concatenate([t.length for t in trees])), T(par), T(prob)
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed))
    state = torch.zeros((int(base[-1]), K), dtype=torch.int16, device=dev)
    for h in range(len(cuts) - 1):
        v = T(order[cuts[h]:cuts[h + 1]])
        pa = par_t[v]
        st = torch.where((pa >= 0)[:, None], state[pa.clamp(min=0)], 0)
        p = torch.exp(-length[v])[:, None]
        pn = p ** TRUE_NU
        u = torch.rand((len(v), K), generator=g, device=dev, dtype=torch.float64)
        u2 = torch.rand((len(v), K), generator=g, device=dev, dtype=torch.float64) * (1 - 1e-9)
        row = prob_t[v][:, None] * K + torch.arange(K, device=dev)
        new = torch.searchsorted(flat, row + u2) - row * M_HI + 1
        zero, keep0, mut = st == 0, p * pn, pn * (1 - p)
        out = torch.where(zero & (u >= keep0), new.clamp(1, M_HI).to(torch.int16), st)
        out = torch.where((zero & (u >= keep0 + mut)) | ((st > 0) & (u >= pn)), -1, out)
        state[v] = out.to(torch.int16)
    res = []
    for t, b in zip(trees, base):
        lf = T(np.nonzero(t.c0 < 0)[0] + b)
        obs = state[lf]
        drop = torch.rand(obs.shape, generator=g, device=dev) < TRUE_PHI
        res.append(torch.where((obs < 0) | drop, -1, obs).to(torch.int16).cpu().numpy())
    sizes = np.concatenate([[len(q) for q in Q] for Q in Qs]).reshape(P, K)
    return [np.minimum(c, sizes[i][None, :]).astype(np.int16) for i, c in enumerate(res)]


def _inputs(case, seed):
    """(trees, codes, Qs): one entry per problem; NNI variants of one tree
    come first and share its characters and priors."""
    rng = np.random.default_rng([int(seed), case["leaves"], case["sites"]])
    n, K = case["leaves"], case["sites"]
    if case["leaves_lo"] and case["leaves_lo"] < n:
        # the sizes belong to the case, the trees to the seed
        of_case = np.random.default_rng([n, K, case["leaves_lo"], case["problems"]])
        sizes = np.exp(of_case.uniform(math.log(case["leaves_lo"]), math.log(n), case["problems"])).astype(int)
    else:
        sizes = [n] * case["problems"]
    if case["variants"]:
        sizes = [n] + list(sizes)
    made = [_random_tree(max(4, int(s)), rng) for s in sizes]
    trees, depths = [t for t, _ in made], [d for _, d in made]
    Qs = [_priors(K, rng) for _ in sizes]
    codes = _simulate(trees, depths, Qs, seed)
    if case["variants"]:
        var = [sim.nni_variant(trees[0], codes[0], rng)[0] for _ in range(case["variants"])]
        trees = var + trees[1:]
        codes = [codes[0]] * len(var) + codes[1:]
        Qs = [Qs[0]] * len(var) + Qs[1:]
    return trees, codes, Qs


def _specs(trees, codes, Qs):
    tables = {}
    for Q in Qs:
        if id(Q) not in tables:
            tables[id(Q)] = SiteTable(Q)
    return [sim.problem_spec(t, Q, c, sites=tables[id(Q)]) for t, c, Q in zip(trees, codes, Qs)]


def _nni_moves(tree):
    """Every NNI move of a tree, post-order ids [moves, 5]: (p, s, A, W, C)
    as the quartet round takes them (p = s = -1 at the root)."""
    u = np.nonzero((tree.c0 >= 0) & (tree.parent >= 0))[0]
    v = tree.parent[u]
    w = np.where(tree.c0[v] == u, tree.c1[v], tree.c0[v])
    p = tree.parent[v]
    s = np.where(p >= 0, np.where(tree.c0[p] == v, tree.c1[p], tree.c0[p]), -1)
    one = np.stack([p, s, tree.c1[u], w, tree.c0[u]], 1)  # first child moves out
    two = np.stack([p, s, tree.c0[u], w, tree.c1[u]], 1)
    return np.concatenate([one, two]), np.concatenate([u, u]), np.concatenate([v, v])


def _quartet_lengths(tree, moves, u, v):
    return np.maximum(2 * DMIN, np.stack([tree.length[moves[:, 2]], tree.length[moves[:, 3]], tree.length[u],
                                          tree.length[moves[:, 4]], tree.length[v]], 1))


def _start(case, trees):
    """Start point: the generating values where a call evaluates given
    parameters, the uniform start where it fits them."""
    if case["kind"] in ("nll", "grad", "post", "quartet"):
        return [t.length for t in trees], TRUE_NU, TRUE_PHI
    return [np.full(t.n_nodes, 0.05) for t in trees], 0.5, 0.5


def prepare(case, seed):
    trees, codes, Qs = _inputs(case, seed)
    specs = _specs(trees, codes, Qs)
    lengths, nu0, phi0 = _start(case, trees)
    kind = case["kind"]
    if kind == "solve":
        return dict(kind=kind, device=torch.cuda.current_device(),
                    req=SolveRequest(specs[0], lengths, nu0, phi0, case["iters"], case["tol"]))
    F = Forest(specs, device=torch.cuda.current_device())
    full = lambda x: torch.full((F.num_problems,), x, dtype=torch.float64, device=F.device)  # noqa: E731
    d_start = F.lengths_to_level(lengths)
    s = dict(kind=kind, F=F, iters=case["iters"], tol=case["tol"], nu0=full(nu0), phi0=full(phi0),
             d0=torch.tensor(d_start, dtype=torch.float64, device=F.device))
    if kind in ("em", "ultra"):
        s.update(d=s["d0"].clone(), nu=s["nu0"].clone(), phi=s["phi0"].clone())
    if kind == "ultra":
        model = HeightModel(F, d_start)
        F.set_ultrametric(model)
        s["heights"] = model.start_heights(d_start, F.free, F.dmin, F.dmax)
    if kind == "grad":
        for x in ("d0", "nu0", "phi0"):
            s[x].requires_grad_(True)
    if kind == "quartet":
        moves, u, v = _nni_moves(trees[0])
        s["qnodes"] = np.where(moves >= 0, F.inv[np.maximum(moves, 0)], -1).astype(np.int32)
        s["len_in"] = _quartet_lengths(trees[0], moves, u, v)
        s["opt"] = np.full(len(moves), 31, np.uint8)
        s["const"] = np.zeros(len(moves))
        F.estep(s["d0"], s["nu0"], s["phi0"])
    return s


def run(s):
    kind = s["kind"]
    if kind == "solve":
        return solve_alone(s["req"], s["device"])
    F = s["F"]
    if kind == "nll":
        return F.nll(s["d0"], s["nu0"], s["phi0"])
    if kind == "grad":
        nll = neg_log_likelihood(F, s["d0"], s["nu0"], s["phi0"])
        gd, gnu, gphi = torch.autograd.grad(nll.sum(), (s["d0"], s["nu0"], s["phi0"]))
        return {"nll": nll, "d": gd, "nu": gnu, "phi": gphi}
    if kind == "post":
        counts, rt, nll = F.estep(s["d0"], s["nu0"], s["phi0"])
        (l0, i0), (lS, iS) = F.posteriors(s["phi0"])
        return {"counts": counts, "rtilde": rt, "nll": nll, "leaf0": l0, "inner0": i0, "leafS": lS, "innerS": iS}
    if kind == "quartet":
        lo, nll, it = F.quartet_em(s["qnodes"], s["len_in"], s["opt"], s["const"], s["nu0"], s["phi0"], s["iters"],
                                   s["tol"])
        return {"lengths": lo, "nll": nll, "iters": it}
    for x in ("d", "nu", "phi"):
        s[x].copy_(s[x + "0"])
    if kind == "ultra":
        F.set_heights(s["heights"])
    nll, it = F.em(s["d"], s["nu"], s["phi"], s["iters"], s["tol"])
    return {"d": s["d"], "nu": s["nu"], "phi": s["phi"], "nll": nll, "iters": it}


def _sizes(case):
    """(leaves, nodes) over all trees of a case, as drawn on average."""
    n, lo = case["leaves"], case["leaves_lo"]
    mean = (n - lo) / math.log(n / lo) if lo and lo < n else n
    leaves = case["problems"] * mean + case["variants"] * n
    return leaves, 2 * leaves - case["problems"] - case["variants"]


def work(case):
    """What one pass cannot do without.  A likelihood reads the leaf codes
    (2 bytes each) and the branch lengths.  A pass that comes back down the
    tree (EM step, gradient, posteriors) also keeps the inside vector of each
    internal node and site, two 64-bit values, written on the way up and read
    on the way down.  Operations per internal node and site: about 20 on the
    way up, 80 on the way down."""
    leaves, nodes = _sizes(case)
    K = case["sites"]
    cells, inner = leaves * K, (nodes - leaves) * K
    kind = case["kind"]
    up = {"bytes": 2 * cells + 8 * nodes, "flops": 20.0 * inner}
    both = {"bytes": 2 * cells + 32 * inner + 16 * nodes, "flops": 100.0 * inner}
    if kind == "nll":
        return up
    if kind == "grad":
        return both
    if kind == "post":
        return {"bytes": both["bytes"] + 16 * (cells + inner) + 40 * nodes, "flops": both["flops"] + 10 * (cells + inner)}
    if kind == "quartet":
        # per move: three subtrees' and the sibling's inside state, the
        # parent's outside state (40 bytes a site and state); about 10 EM steps
        moves = 4 * leaves
        return {"bytes": moves * (K * 5 * 20.0 + 100), "flops": moves * K * 10 * 250.0}
    steps = case["iters"] if case["tol"] == 0 else min(case["iters"], 20)
    out = {x: both[x] * steps for x in both}
    if kind == "ultra":
        out["flops"] += steps * 60.0 * nodes * 100
    return out


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
class _Exact:
    """All trees of a case stacked: node ids are post-order ids plus the
    tree's base; arrays over (node, site)."""

    def __init__(self, trees, codes, Qs):
        self.dev = dev = _device()
        self.K = K = len(Qs[0])
        self.base = np.concatenate([[0], np.cumsum([t.n_nodes for t in trees])])
        N = int(self.base[-1])
        cat = lambda name: np.concatenate(  # noqa: E731
            [np.where(getattr(t, name) >= 0, getattr(t, name) + b, -1) for t, b in zip(trees, self.base)])
        c0, c1 = cat("c0"), cat("c1")
        self.P = len(trees)
        self.prob_np = np.repeat(np.arange(self.P), np.diff(self.base))
        h = np.zeros(N, np.int64)
        inner = np.nonzero(c0 >= 0)[0]
        while True:
            new = 1 + np.maximum(h[c0[inner]], h[c1[inner]])
            if np.array_equal(new, h[inner]):
                break
            h[inner] = new
        self.height = h
        post = np.concatenate([np.arange(t.n_nodes) for t in trees])
        self.level_order = np.lexsort((post, self.prob_np, h))
        T = lambda a, **kw: torch.as_tensor(a, device=dev, **kw)  # noqa: E731
        self.prob = T(self.prob_np)
        self.root = T(self.base[1:] - 1)
        lf = np.nonzero(c0 < 0)[0]
        self.leaf = T(lf)
        lab = torch.zeros((N, K), dtype=torch.int16, device=dev)
        lab[self.leaf] = T(np.concatenate(codes))
        self.levels = []
        for x in range(1, int(h.max()) + 1):
            v = np.nonzero(h == x)[0]
            v, a, b = T(v), T(c0[v]), T(c1[v])
            la, lb = lab[a], lab[b]
            lab[v] = torch.where((la == 0) | (lb == 0), 0,
                                 torch.where(la < 0, lb, torch.where((lb < 0) | (la == lb), la, 0))).to(torch.int16)
            self.levels.append((v, a, b))
        self.lab = lab
        self.nobs = torch.tensor([float((c != -1).sum()) for c in codes], dtype=torch.float64, device=dev)
        self.phimin = torch.tensor([1.0 / (K * c.shape[0]) for c in codes], dtype=torch.float64, device=dev)
        table, seen = [], {}
        for Q in Qs:
            if id(Q) not in seen:
                seen[id(Q)] = len(table)
                t = np.ones((K, M_HI + 1))
                for k, q in enumerate(Q):
                    t[k, 1:len(q) + 1] = list(q.values())
                table.append(t)
        self.table = T(np.stack(table))
        self.table_of = T(np.array([seen[id(Q)] for Q in Qs]))
        self.q = self.weight(lab, self.prob)

    def weight(self, lab, prob):
        k = torch.arange(self.K, device=self.dev)
        return self.table[self.table_of[prob][:, None], k[None, :], lab.long().clamp(min=0)]

    def coef(self, d, nu):
        n = nu[self.prob]
        return torch.exp(-(1 + n) * d), -torch.expm1(-d) * torch.exp(-n * d), torch.exp(-n * d), -torch.expm1(-n * d)

    def edge(self, v, c):
        """Inside values of nodes v over their branches, from below."""
        lab, B0, BA = self.lab[v], self.B0[v], self.BA[v]
        p1n, mut, pn, sil = (x[v][:, None] for x in c)
        S = torch.where(lab < 0, sil, 0.0)
        some = lab != 0
        return p1n * B0 + torch.where(some, mut * self.q[v] * BA, 0.0) + S, torch.where(some, pn * BA, 0.0) + S

    def inside(self, d, nu, phi):
        self.c = c = self.coef(d, nu)
        N, K = self.lab.shape
        zeros = lambda: torch.zeros((N, K), dtype=torch.float64, device=self.dev)  # noqa: E731
        self.B0, self.BA, self.e0, self.eA, self.ls, self.s = (zeros() for _ in range(6))
        lab, ph = self.lab[self.leaf], phi[self.prob[self.leaf]][:, None]
        self.B0[self.leaf] = torch.where(lab == 0, 1 - ph, torch.where(lab < 0, ph, 0.0))
        self.BA[self.leaf] = torch.where(lab > 0, 1 - ph, torch.where(lab < 0, ph, 0.0))
        self.e0[self.leaf], self.eA[self.leaf] = self.edge(self.leaf, c)
        for v, a, b in self.levels:
            lab = self.lab[v]
            B0 = self.e0[a] * self.e0[b]
            BA = torch.where(lab != 0, self.eA[a] * self.eA[b], 0.0)
            s = torch.where(lab < 0, 1.0, torch.maximum(B0, BA))
            self.s[v], self.B0[v], self.BA[v] = s, B0 / s, BA / s
            self.ls[v] = self.ls[a] + self.ls[b] + torch.log(s)
            self.e0[v], self.eA[v] = self.edge(v, c)
        r = self.root
        self.site = torch.log(self.e0[r]) + self.ls[r]
        return self.site.sum(1)

    def outside(self, phi, posteriors=False):
        """Expected counts of every branch and the dropout sums (with the
        state of the last inside())."""
        N, K = self.lab.shape
        self.g0, self.gA = torch.zeros_like(self.B0), torch.zeros_like(self.B0)
        S = torch.zeros((N, 5), dtype=torch.float64, device=self.dev)
        if posteriors:
            self.post0, self.postS = torch.zeros_like(self.B0), torch.zeros_like(self.B0)
        self.g0[self.root] = 1.0 / self.e0[self.root]
        rt = torch.zeros(self.P, dtype=torch.float64, device=self.dev)
        for v, a, b in self.levels[::-1] + [(self.leaf, None, None)]:
            p1n, mut, pn, sil = (x[v][:, None] for x in self.c)
            lab, g0, gA, B0, BA = self.lab[v], self.g0[v], self.gA[v], self.B0[v], self.BA[v]
            mq = mut * self.q[v]
            miss = torch.where(lab < 0, sil, 0.0)
            S[v] = torch.stack([(g0 * p1n * B0).sum(1), (g0 * mq * BA).sum(1), (g0 * miss).sum(1),
                                (gA * pn * BA).sum(1), (gA * miss).sum(1)], 1)
            h0 = g0 * p1n
            hA = torch.where(lab != 0, g0 * mq + gA * pn, 0.0)
            if posteriors:
                own = (g0 + gA) * miss + self.postS[v]  # postS holds the parent's share
                self.post0[v], self.postS[v] = h0 * B0, own
                if a is not None:
                    for x in (a, b):
                        self.postS[x] = torch.where(lab < 0, own, 0.0)
            if a is None:
                r = torch.where(lab < 0, h0 * B0 + hA * BA, 0.0).sum(1)
                rt.index_add_(0, self.prob[v], r)
                break
            s = self.s[v]
            for x, y in ((a, b), (b, a)):
                self.g0[x] = h0 * self.e0[y] / s
                self.gA[x] = hA * self.eA[y] / s
        return S, rt

    def mstep(self, S, rt, d, nu, phi, heights=None):
        s = S.clamp(min=1e-6)
        s = s / s.sum(1, keepdim=True) * self.K
        n = nu[self.prob]
        A, S1 = (n + 1) * s[:, 0] + n * s[:, 1] + n * s[:, 3], s[:, 1]
        B = torch.where(n > 1e-5, s[:, 2] + s[:, 4], 0.0)
        dn = _branch_lengths(A, S1, B, n) if heights is None else heights.solve(A, S1, B, n, self.K)
        phi_n = rt / (self.nobs + rt)
        phi_n = torch.where(phi_n < self.phimin, 0.0, phi_n)
        a, b = s[:, 0] + s[:, 1] + s[:, 3], s[:, 2] + s[:, 4]

        def slope(x):
            xx = x[self.prob]
            out = torch.zeros(self.P, dtype=torch.float64, device=self.dev)
            return out.index_add_(0, self.prob, dn * (b / torch.expm1(xx * dn) - a))

        lo, hi = torch.zeros_like(nu), torch.ones_like(nu)
        top = slope(hi) > 0
        for _ in range(70):
            mid = 0.5 * (lo + hi)
            up = slope(mid) > 0
            lo, hi = torch.where(up, mid, lo), torch.where(up, hi, mid)
        return dn, torch.where(top, 1.0, 0.5 * (lo + hi)), phi_n

    def em(self, d, nu, phi, iters, tol, heights=None):
        done = torch.zeros(self.P, dtype=torch.bool, device=self.dev)
        nll = torch.zeros(self.P, dtype=torch.float64, device=self.dev)
        pre = None
        for step in range(iters + 1):
            llh = self.inside(d, nu, phi)
            nll = torch.where(done, nll, -llh)
            if pre is not None and tol > 0:
                done = done | (((llh - pre) / pre).abs() < tol)
            pre = llh
            if step == iters or bool(done.all()):
                break
            S, rt = self.outside(phi)
            dn, nn, pn = self.mstep(S, rt, d, nu, phi, heights)
            d, nu, phi = torch.where(done[self.prob], d, dn), torch.where(done, nu, nn), torch.where(done, phi, pn)
        return d, nu, phi, nll


def _branch_lengths(A, S1, B, n):
    """argmax over [DMIN, DMAX] of the concave branch objectives."""
    def slope(x):
        return -A + S1 / torch.expm1(x) + torch.where(B > 0, B * n / torch.expm1(n * x), 0.0)

    lo, hi = torch.full_like(A, DMIN), torch.full_like(A, DMAX)
    low, high = ~(slope(lo) > 0), ~(slope(hi) < 0)
    for _ in range(70):
        mid = 0.5 * (lo + hi)
        up = slope(mid) > 0
        lo, hi = torch.where(up, mid, lo), torch.where(up, hi, mid)
    return torch.where(low, DMIN, torch.where(high, DMAX, 0.5 * (lo + hi)))


class _Heights:
    """Branch lengths of one ultrametric tree: node heights above the leaves
    are free (and the stem's top), each branch within its bounds; a barrier
    method with dense Newton steps."""

    def __init__(self, tree, dev):
        N = tree.n_nodes
        self.dev = dev
        inner = np.nonzero(tree.c0 >= 0)[0]
        col = np.full(N + 1, -1, np.int64)
        col[inner] = np.arange(len(inner))
        col[N] = len(inner)
        top = np.where(tree.parent >= 0, tree.parent, N)
        M = np.zeros((N, len(inner) + 1))
        M[np.arange(N), col[top]] += 1.0
        M[inner, col[inner]] -= 1.0
        self.M = torch.as_tensor(M, device=dev)
        t = np.zeros(N + 1)
        for v in inner:
            t[v] = 0.05 + max(t[tree.c0[v]], t[tree.c1[v]])
        t[N] = t[N - 1] + 0.05
        self.start = torch.as_tensor(np.concatenate([t[inner], t[N:]]), device=dev)

    def solve(self, A, S1, B, n, K):
        M, t = self.M, self.start.clone()

        def value(t, mu):
            x = M @ t
            if not bool(((x > DMIN) & (x < DMAX)).all()):
                return -math.inf
            f = -A * x + S1 * torch.log(-torch.expm1(-x)) + torch.where(B > 0, B * torch.log(-torch.expm1(-n * x)), 0.0)
            return float((f + mu * (torch.log(x - DMIN) + torch.log(DMAX - x))).sum())

        mu, end = 1e-2 * K, 1e-13 * K
        while True:
            for _ in range(60):
                x = M @ t
                em, en = torch.expm1(x), torch.expm1(n * x)
                g = -A + S1 / em + torch.where(B > 0, B * n / en, 0.0)
                w = S1 * (em + 1) / em ** 2 + torch.where(B > 0, B * n * n * (en + 1) / en ** 2, 0.0)
                lo, hi = x - DMIN, DMAX - x
                g = g + mu * (1 / lo - 1 / hi)
                w = w + mu * (1 / lo ** 2 + 1 / hi ** 2)
                grad = M.T @ g
                step = torch.linalg.solve(M.T @ (w[:, None] * M), grad)
                lam = float(grad @ step)
                dx = M @ step
                room = torch.where(dx < 0, 0.99 * lo / -dx, torch.where(dx > 0, 0.99 * hi / dx, 1.0))
                a = min(1.0, float(room.min()))
                f0 = value(t, mu)
                if lam > 1e-12 * (1 + abs(f0)):
                    while value(t + a * step, mu) < f0 + 0.25 * a * lam and a > 1e-12:
                        a *= 0.5
                t = t + a * step
                if not lam > 0 or float((a * step).abs().max()) < 1e-15:
                    break
            if mu <= end:
                return M @ t
            mu = max(mu * 0.1, end)


def _exact_quartet(X, tree, nu, phi, iters, tol):
    """The quartet EM of every NNI move: the site likelihood is linear in the
    values that the moved clade's branch hands to its parent."""
    dev, K = X.dev, X.K
    moves, u, v = _nni_moves(tree)
    d = torch.as_tensor(_quartet_lengths(tree, moves, u, v), device=dev)
    A, W, C, v = (torch.as_tensor(x, device=dev) for x in (moves[:, 2], moves[:, 3], moves[:, 4], v))
    n = len(v)
    k0, kA = X.g0[v], X.gA[v]
    rest = 1.0 - k0 * X.e0[v] - kA * X.eA[v]
    rest = torch.where(X.lab[v] < 0, rest, 0.0)  # only a silenced clade leaves a part that is free of it
    scale = torch.exp(X.ls[A] + X.ls[W] + X.ls[C] - X.ls[v])
    k0, kA = k0 * scale, kA * scale
    site0 = X.site[0][None, :]
    prob0 = torch.zeros(n, dtype=torch.long, device=dev)
    la, lw, lc, lv = X.lab[A], X.lab[W], X.lab[C], X.lab[v]
    lu = torch.where((la == 0) | (lw == 0), 0, torch.where(la < 0, lw, torch.where((lw < 0) | (la == lw), la, 0)))
    lab = [la, lw, lu, lc, lv]
    q = [X.weight(x, prob0) for x in lab]
    below = {0: (X.B0[A], X.BA[A]), 1: (X.B0[W], X.BA[W]), 3: (X.B0[C], X.BA[C])}
    done = torch.zeros(n, dtype=torch.bool, device=dev)
    nll = torch.zeros(n, dtype=torch.float64, device=dev)
    pre = None
    for it in range(iters + 1):
        p1n, mut, pn, sil = torch.exp(-(1 + nu) * d), -torch.expm1(-d) * torch.exp(-nu * d), torch.exp(-nu * d), \
            -torch.expm1(-nu * d)

        def edge(j, B):
            S = torch.where(lab[j] < 0, sil[:, j:j + 1], 0.0)
            some = lab[j] != 0
            return (p1n[:, j:j + 1] * B[0] + torch.where(some, mut[:, j:j + 1] * q[j] * B[1], 0.0) + S,
                    torch.where(some, pn[:, j:j + 1] * B[1], 0.0) + S)

        Bs = dict(below)
        e = {j: edge(j, Bs[j]) for j in (0, 1, 3)}
        Bs[2] = (e[0][0] * e[1][0], torch.where(lu != 0, e[0][1] * e[1][1], 0.0))
        e[2] = edge(2, Bs[2])
        Bs[4] = (e[2][0] * e[3][0], torch.where(lv != 0, e[2][1] * e[3][1], 0.0))
        e[4] = edge(4, Bs[4])
        L = rest + k0 * e[4][0] + kA * e[4][1]
        llh = (torch.log(L) + site0).sum(1)
        nll = torch.where(done, nll, -llh)
        if pre is not None:
            done = done | (((llh - pre) / pre).abs() < tol)
        pre = llh
        if it == iters or bool(done.all()):
            break
        g = {4: (k0 / L, kA / L)}

        def down(j):
            g0, gA = g[j]
            return g0 * p1n[:, j:j + 1], torch.where(lab[j] != 0, g0 * mut[:, j:j + 1] * q[j] + gA * pn[:, j:j + 1], 0.0)

        h = down(4)
        g[2], g[3] = (h[0] * e[3][0], h[1] * e[3][1]), (h[0] * e[2][0], h[1] * e[2][1])
        h = down(2)
        g[0], g[1] = (h[0] * e[1][0], h[1] * e[1][1]), (h[0] * e[0][0], h[1] * e[0][1])
        S = torch.zeros((n, 5, 5), dtype=torch.float64, device=dev)
        for j in range(5):
            miss = torch.where(lab[j] < 0, sil[:, j:j + 1], 0.0)
            some = torch.where(lab[j] != 0, Bs[j][1], 0.0)
            S[:, j, 0] = (g[j][0] * p1n[:, j:j + 1] * Bs[j][0]).sum(1)
            S[:, j, 1] = (g[j][0] * mut[:, j:j + 1] * q[j] * some).sum(1)
            S[:, j, 2] = (g[j][0] * miss).sum(1)
            S[:, j, 3] = (g[j][1] * pn[:, j:j + 1] * some).sum(1)
            S[:, j, 4] = (g[j][1] * miss).sum(1)
        s = S.clamp(min=1e-6)
        s = s / s.sum(2, keepdim=True) * K
        dn = _branch_lengths((nu + 1) * s[..., 0] + nu * s[..., 1] + nu * s[..., 3], s[..., 1], s[..., 2] + s[..., 4],
                             torch.full_like(d, nu))
        d = torch.where(done[:, None], d, dn)
    return {"lengths": d, "nll": nll, "iters": None}


def exact(case, seed):
    trees, codes, Qs = _inputs(case, seed)
    X = _Exact(trees, codes, Qs)
    lengths, nu0, phi0 = _start(case, trees)
    d = torch.as_tensor(np.concatenate(lengths), device=X.dev)
    nu = torch.full((X.P,), nu0, dtype=torch.float64, device=X.dev)
    phi = torch.full((X.P,), phi0, dtype=torch.float64, device=X.dev)
    order = torch.as_tensor(X.level_order, device=X.dev)
    kind = case["kind"]
    if kind in ("em", "solve", "ultra"):
        heights = _Heights(trees[0], X.dev) if kind == "ultra" else None
        d, nu, phi, nll = X.em(d, nu, phi, case["iters"], case["tol"], heights)
        if kind == "solve":
            return (float(nll[0]), [d.cpu().numpy()], float(nu[0]), float(phi[0]), None)
        return {"d": d[order], "nu": nu, "phi": phi, "nll": nll, "iters": None}
    nll = -X.inside(d, nu, phi)
    if kind == "nll":
        return nll
    S, rt = X.outside(phi, posteriors=kind == "post")
    if kind == "quartet":
        return _exact_quartet(X, trees[0], nu0, phi0, case["iters"], case["tol"])
    if kind == "post":
        nl = len(X.leaf)
        p0, pS = (x[order].cpu().numpy() for x in (X.post0, X.postS))
        return {"counts": S[order].reshape(-1), "rtilde": rt, "nll": nll, "leaf0": p0[:nl].reshape(-1),
                "inner0": p0[nl:].reshape(-1), "leafS": pS[:nl].reshape(-1), "innerS": pS[nl:].reshape(-1)}
    # gradient: the expected score of the transitions, and of the leaf entries
    x = nu[X.prob]
    gd = -(1 + x) * S[:, 0] + S[:, 1] * (1 / torch.expm1(d) - x) - x * S[:, 3] + (S[:, 2] + S[:, 4]) * x / torch.expm1(x * d)
    gn = d * (-S[:, 0] - S[:, 1] - S[:, 3] + (S[:, 2] + S[:, 4]) / torch.expm1(x * d))
    gnu = torch.zeros_like(nu).index_add_(0, X.prob, gn)
    gphi = -X.nobs / (1 - phi) + rt / phi
    return {"nll": nll, "d": -gd[order], "nu": -gnu, "phi": -gphi}
