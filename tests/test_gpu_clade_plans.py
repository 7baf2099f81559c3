"""Clade passes where the plan is known to take them: the plan in use is
asserted, so that a comparison with level launches cannot pass on level
launches.  Splits near the root (LAML_TOP_MAX_NODES) give clades as large as
their cap allows: long one-child walks over many batches of leaf codes
(caterpillars), two pending states (Yule and balanced trees), clades that are
whole trees.  Same bits as level launches, in the E-step, EM and posteriors.
And the first call on a forest, whichever it is, takes the plan it lays out."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest
from test_gpu_clades import _problem

pytestmark = pytest.mark.gpu

# kind, leaves and sites of the first tree, trees, and the largest clade at caps 1, 7 and 64
CASES = [("caterpillar", 100, 130, 3, (1, 7, 64)), ("caterpillar", 70, 200, 2, (1, 7, 64)),
         ("yule", 260, 100, 3, None), ("balanced", 256, 70, 2, (1, 7, 8)), ("yule", 2, 70, 4, (1, 1, 1)),
         ("yule", 40, 129, 30, None)]


def _dev(F, x):
    return torch.tensor(np.asarray(x, dtype=np.float64), device=F.device)


@pytest.mark.parametrize("kind,n,K,P,largest", CASES, ids=lambda x: str(x).replace(" ", ""))
@pytest.mark.parametrize("cap", [1, 7, 64])
def test_clades_in_use_equal_levels(kind, n, K, P, largest, cap, monkeypatch):
    monkeypatch.setenv("LAML_TOP_MAX_NODES", "1")
    probs = [_problem(kind, n + (0 if n == 2 else 9 * i), K - 5 * (i % 9), 300 + i) for i in range(P)]
    specs = [sim.problem_spec(*p) for p in probs]
    got = {}
    for clades in (cap, 0):
        monkeypatch.setenv("LAML_CLADES", str(clades))
        F = Forest(specs, device=torch.cuda.current_device())
        d = _dev(F, F.lengths_to_level([np.maximum(t.length, 0.005) for t, _, _ in probs]))
        nu, phi = _dev(F, [0.2] * P), _dev(F, [0.3] * P)
        for mode in (PASS_HYBRID, PASS_LEVELS):
            F.set_pass_mode(mode)
            print("clade plan", kind, n, K, P, clades, mode, flush=True)
            counts, rt, nll = [x.cpu().numpy().copy() for x in F.estep(d, nu, phi)]
            plan = F.pass_plan()
            if clades:
                assert plan["inside_clades"] > 0 and plan["outside_clades"] == plan["inside_clades"], plan
                assert plan["walk_level"] > 1 and plan["blocks"] == 0 and plan["chain_plans"] == 0, plan
                if largest is not None:
                    assert plan["largest_clade"] == largest[(1, 7, 64).index(cap)], plan
                elif cap == 64:
                    assert plan["largest_clade"] > 7, plan
            else:
                assert plan["inside_clades"] == plan["outside_clades"] == 0, plan
            em = [x.clone() for x in (d, nu, phi)]
            F.em(*em, 3, 0.0)
            F.estep(d, nu, phi)
            post = [x.copy() for pair in F.posteriors(phi) for x in pair]
            got[clades, mode] = [nll, counts, rt] + [x.cpu().numpy() for x in em] + post
        F.close()
    for mode in (PASS_HYBRID, PASS_LEVELS):
        for a, b in zip(got[cap, mode], got[0, mode]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("first", ["estep", "nll", "em"])
def test_first_call_takes_the_plan_it_lays_out(first, monkeypatch):
    """7,000 leaves x 300 sites, whose outside pass would run chains without
    clades: no chain plan is laid out when it runs clades."""
    monkeypatch.setenv("LAML_CLADES", "32")
    t, Q, codes, _ = sim.make_problem(7000, 300, 3, 12, 1.0, 0.1, 0.1, 8)
    F = Forest([sim.problem_spec(t, Q, codes)], device=torch.cuda.current_device())
    prm = [_dev(F, F.lengths_to_level([np.maximum(t.length, 0.005)])), _dev(F, [0.2]), _dev(F, [0.1])]
    print("first call", first, flush=True)
    if first == "em":
        F.em(*[x.clone() for x in prm], 1, 0.0)
    elif first == "nll":
        F.nll(*prm)
        F.grad(*prm)
    else:
        F.estep(*prm)
    plan = F.pass_plan()
    assert plan["outside_clades"] > 0 and plan["chain_plans"] == 0, plan
    F.close()


@pytest.mark.parametrize("n,K,P,outside", [(40, 70, 1000, False), (20, 300, 640, False), (300, 300, 60, True)])
def test_outside_clades_only_where_blocks_fill(n, K, P, outside, monkeypatch):
    """Forests of many trees with few clades each keep outside chains; the
    counts are those of level launches either way."""
    base = [_problem("yule", n, K, 500 + i) for i in range(10)]
    specs = [sim.problem_spec(*base[i % 10]) for i in range(P)]
    got = []
    for env in (None, "0"):
        if env is not None:
            monkeypatch.setenv("LAML_CLADES", env)
        F = Forest(specs, device=torch.cuda.current_device())
        d = _dev(F, F.lengths_to_level([np.maximum(base[i % 10][0].length, 0.005) for i in range(P)]))
        nu, phi = _dev(F, [0.2] * P), _dev(F, [0.3] * P)
        assert (F.num_nodes - F.num_leaves) * -(-K // 64) >= 57344
        print("outside clades", n, K, P, env, flush=True)
        counts, rt, nll = F.estep(d, nu, phi)
        plan = F.pass_plan()
        if env is None:
            assert plan["inside_clades"] > 0 and bool(plan["outside_clades"]) == outside, plan
            assert F.chains() == (0 if outside else 1) and plan["chain_plans"] == (0 if outside else 1), plan
        got.append([x.cpu().numpy().copy() for x in (nll, counts, rt)])
        F.close()
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


def test_clades_of_middle_forests_once_they_pay():
    """A forest of 12,288 to 32,768 (node, chunk) pairs lays its clades out when
    its calls would have saved the time, and gives the same bits before and
    after; a call under capture lays out nothing."""
    t, Q, codes = _problem("yule", 4000, 300, 9)
    spec = sim.problem_spec(t, Q, codes)
    F = Forest([spec], device=torch.cuda.current_device())
    assert 12288 <= (F.num_nodes - F.num_leaves) * 5 < 32768
    d, nu, phi = _dev(F, F.lengths_to_level([np.maximum(t.length, 0.005)])), _dev(F, [0.2]), _dev(F, [0.3])

    def likelihood():
        out = F.nll(d, nu, phi, site_llh=True).cpu().numpy().copy()
        return np.concatenate([out, F.site_llh.cpu().numpy()])

    first = likelihood()
    assert F.pass_plan()["inside_clades"] == 0
    counts = [x.cpu().numpy().copy() for x in F.estep(d, nu, phi)]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        for _ in range(12):
            F.nll(d, nu, phi)
    assert F.pass_plan()["inside_clades"] == 0
    for _ in range(12):
        np.testing.assert_array_equal(likelihood(), first)
    assert F.pass_plan()["inside_clades"] > 0
    for a, b in zip(F.estep(d, nu, phi), counts):
        np.testing.assert_array_equal(a.cpu().numpy(), b)
    F.close()
    F = Forest([spec], device=torch.cuda.current_device())
    F.em(d.clone(), nu.clone(), phi.clone(), 3, 0.0)
    assert F.pass_plan()["inside_clades"] > 0
    F.close()
