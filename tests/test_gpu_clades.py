"""Inside pass over clades: the same bits as level launches (site and problem
likelihoods, and the counts of the outside pass that reads its rows) for trees
of every shape the walk meets -- Yule trees, a caterpillar, a balanced tree,
two leaves, trees of different site counts in one forest -- at clades of one
node, a few, and as many as its pending states allow, with partial chunks and
sites of special patterns, in level and hybrid passes and in the EM loop; and
against the C oracle's likelihoods (1e-9 relative)."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest
from oracle import pmm_ref
from test_gpu_chains import _caterpillar

pytestmark = pytest.mark.gpu


def _balanced(n):
    N = 2 * n - 1
    c0, c1, par = np.full(N, -1), np.full(N, -1), np.full(N, -1)
    it = iter(range(N))

    def build(m):
        if m == 1:
            return next(it)
        a, b = build((m + 1) // 2), build(m // 2)
        v = next(it)
        c0[v], c1[v], par[a], par[b] = a, b, v, v
        return v

    build(n)
    return sim.YuleTree(c0, c1, par, np.random.default_rng(n).uniform(0.01, 0.2, N), ["c%d" % i for i in range(n)])


def _problem(kind, n, K, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    if kind == "yule":
        t, Q, codes, _ = sim.make_problem(n, K, 3, 12, 1.0, 0.1, 0.15, seed)
    else:
        t = _caterpillar(n, rng) if kind == "caterpillar" else _balanced(n)
        Q = sim.random_priors(K, 3, 12, 1.0, rng)
        codes = sim.simulate_codes(t, Q, 0.1, 0.15, rng)
    codes[:, 0] = -1
    codes[: n // 2, 1] = -1
    codes[:, 2] = 1
    codes[::3, 3] = -2
    return t, Q, codes


CASES = [("yule", 200, 150, 1), ("yule", 257, 65, 3), ("caterpillar", 90, 64, 1), ("balanced", 128, 70, 1),
         ("yule", 2, 40, 2), ("yule", 3, 129, 1)]


@pytest.mark.parametrize("kind,n,K,P", CASES)
@pytest.mark.parametrize("cap", [1, 3, 64])
def test_clades_equal_levels(kind, n, K, P, cap, monkeypatch):
    probs = [_problem(kind, n + 37 * i, K - 13 * i, 70 + i) for i in range(P)]
    specs = [sim.problem_spec(*p) for p in probs]
    got = {}
    for clades in (cap, 0):
        monkeypatch.setenv("LAML_CLADES", str(clades))
        F = Forest(specs, device=torch.cuda.current_device())
        d = torch.tensor(F.lengths_to_level([np.maximum(t.length, 0.005) for t, _, _ in probs]),
                         dtype=torch.float64, device=F.device)
        nu = torch.full((P,), 0.2, dtype=torch.float64, device=F.device)
        phi = torch.full((P,), 0.3, dtype=torch.float64, device=F.device)
        for mode in (PASS_HYBRID, PASS_LEVELS):
            F.set_pass_mode(mode)
            print("case", kind, n, K, P, clades, mode, flush=True)
            nll = F.nll(d, nu, phi).cpu().numpy().copy()
            counts, rt, enll = [x.cpu().numpy().copy() for x in F.estep(d, nu, phi)]
            em = [x.clone() for x in (d, nu, phi)]
            F.em(*em, 3, 0.0)
            torch.cuda.synchronize()
            # every outside row again, after an E-step that kept them in registers
            F.estep(d, nu, phi)
            post = [x.copy() for pair in F.posteriors(phi) for x in pair]
            got[clades, mode] = [nll, counts, rt, enll] + [x.cpu().numpy() for x in em] + post
        F.close()
    for mode in (PASS_HYBRID, PASS_LEVELS):
        for a, b in zip(got[cap, mode], got[0, mode]):
            assert np.array_equal(a, b)
    for p, (t, Q, codes) in enumerate(probs):
        r = pmm_ref.RefProblem(t.c0, t.c1, t.parent, codes, Q, None, 1.0 / codes.size)
        np.testing.assert_allclose(got[cap, PASS_HYBRID][0][p], r.estep(np.maximum(t.length, 0.005), 0.2, 0.3)[0],
                                   rtol=1e-9)
