"""Small problems run whole in one block (forests of one-tree problems of at
most 64 sites whose state fits a CU's LDS, with their launch plan untouched):
NLL, E-step, gradient and EM against the C oracle at the sizes where the
kernel's steps change: two leaves, one narrow level, levels of exactly one
wavefront's cells and one more, levels of several steps, site counts at and
around multiples of 8 and 64, trees deeper than 64 levels, the largest state
that fits and the first that does not (which keeps the general passes),
batches of unequal problems, fixed branches, nu and phi.  Tolerances: the
stated bars (NLL and counts 1e-9 relative, fitted parameters 1e-6)."""
import math

import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd.forest import Forest
from oracle import pmm_ref
from test_gpu_chains import _problem

pytestmark = pytest.mark.gpu

CASES = [
    [("yule", 2, 1)], [("yule", 5, 8)], [("yule", 3, 64)], [("yule", 40, 7)], [("yule", 41, 9)],
    [("yule", 120, 16)], [("yule", 250, 30)], [("yule", 199, 40)], [("yule", 230, 40)], [("yule", 120, 64)],
    [("yule", 119, 63)], [("yule", 700, 3)], [("caterpillar", 130, 20)], [("caterpillar", 64, 33)],
    [("yule", 200, 20), ("caterpillar", 30, 11), ("yule", 2, 5), ("yule", 77, 24)],
    [("yule", 20 + 3 * i, 12) for i in range(20)],
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dx%s-%d-%d" % ((len(c),) + c[0]))
def test_problem_blocks_equal_oracle(case):
    probs = [_problem(kind, n, K, 4000 + 7 * i + n + K) for i, (kind, n, K) in enumerate(case)]
    specs = []
    for i, (t, q, c, _) in enumerate(probs):
        free = np.ones(t.n_nodes, dtype=np.uint8)
        if i % 2:
            free[::3] = 0  # some fixed branches, and (flags 0) fixed nu and phi
        specs.append(sim.problem_spec(t, q, c, free=free, flags=0 if i % 4 == 3 else 3))
    F = Forest(specs, device=torch.cuda.current_device())
    refs = [pmm_ref.RefProblem(t.c0, t.c1, t.parent, c, q, s.trees[0].free, 1.0 / (len(q) * c.shape[0]))
            for (t, q, c, _), s in zip(probs, specs)]
    P, iters = len(probs), 4
    start = [np.maximum(t.length, 0.006) for (t, _, _, _) in probs]
    dev = lambda x: torch.tensor(x, dtype=torch.float64, device=F.device)  # noqa: E731
    d, nu, phi = dev(F.lengths_to_level(start)), dev([0.2] * P), dev([0.1] * P)
    print("case", case, flush=True)
    nll = F.nll(d, nu, phi, site_llh=True).cpu().numpy().copy()
    counts, rt, nll2 = (x.clone() for x in F.estep(d, nu, phi))
    got = np.empty((F.num_nodes, 5))
    got[F.order] = counts.view(-1, 5).cpu().numpy()
    again, rt2 = F.outside(phi)  # over the state of the last call
    np.testing.assert_array_equal(again.view(-1, 5).cpu().numpy(), got[F.order])
    F.nll(d, nu, phi)
    gd, gnu, gphi = (x.cpu().numpy() for x in F.grad(d, nu, phi))
    gd = F.level_to_tree_lengths(gd)
    trace = torch.zeros((iters + 1) * P, dtype=torch.float64, device=F.device)
    de, nue, phie = d.clone(), nu.clone(), phi.clone()
    nll_em, it = F.em(de, nue, phie, iters, 0.0, trace=trace)
    trace = trace.view(iters + 1, P).cpu().numpy()
    fitted = F.level_to_tree_lengths(de.cpu().numpy())
    assert (it.cpu().numpy() == iters + 1).all()
    for p, ref in enumerate(refs):
        rnll, rcounts, R, Rt = ref.estep(start[p], 0.2, 0.1)
        assert math.isclose(nll[p], rnll, rel_tol=1e-9) and math.isclose(nll2[p].item(), rnll, rel_tol=1e-9)
        np.testing.assert_allclose(got[F.tree_base[p]:F.tree_base[p + 1]], rcounts, rtol=1e-9, atol=1e-9)
        assert math.isclose(rt[p].item(), Rt, rel_tol=1e-9, abs_tol=1e-10)
        assert math.isclose(rt2[p].item(), Rt, rel_tol=1e-9, abs_tol=1e-10)
        # the expected score (Fisher identity) on the oracle's counts
        S, x, ln = rcounts, 0.2, start[p]
        terms = [-(1 + x) * S[:, 0], S[:, 1] * (1 / np.expm1(ln) - x), -x * S[:, 3],
                 (S[:, 2] + S[:, 4]) * x / np.expm1(x * ln)]
        np.testing.assert_allclose(gd[p], -sum(terms), rtol=0, atol=1e-9 * max(1.0, max(abs(y).max() for y in terms)))
        dl, n, f = start[p], 0.2, 0.1
        flags = specs[p].flags
        for i in range(iters):
            e, c, R, Rt = ref.estep(dl, n, f)
            assert math.isclose(-trace[i, p], -e, rel_tol=1e-9), (i, trace[i, p], e)
            dl, n, f = ref.mstep(c, R, Rt, dl, n, f, opt_nu=bool(flags & 2), opt_phi=bool(flags & 1))
        np.testing.assert_allclose(fitted[p], dl, rtol=1e-6, atol=1e-9)
        assert abs(nue[p].item() - n) <= 1e-6 and abs(phie[p].item() - f) <= 1e-6
        assert math.isclose(nll_em[p].item(), ref.nll(dl, n, f), rel_tol=1e-9)
    assert F.mstep_status().tolist() == [0] * P
    F.close()
