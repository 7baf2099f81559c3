"""Single calls on forests that run in whole-problem blocks: likelihood, outside
pass and gradient equal those of the general passes (1e-11 relative to the
largest of each output) whatever call came before, for one problem, some, and
more than the blocks take likelihoods of; with fixed branches and 1 to 64
sites."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


def _host(xs):
    return [x.cpu().numpy().copy() for x in xs]


@pytest.mark.parametrize("n,K,P", [(2, 1, 1), (250, 30, 1), (120, 64, 2), (33, 17, 40), (7, 9, 1100)])
def test_calls_equal_general_passes(n, K, P):
    specs, trees = [], []
    for i in range(P):
        t, Q, codes, _ = sim.make_problem(n + i % 5 * (n > 2 and n < 100), K, 3, 9, 1.0, 0.1, 0.15, 700 + i % 12)
        free = np.ones(t.n_nodes, dtype=np.uint8)
        free[::4] = 0
        specs.append(sim.problem_spec(t, Q, codes, free=free))
        trees.append(t)
    out = []
    for general in (False, True):
        F = Forest(specs, device=torch.cuda.current_device())
        assert F.pass_plan()["blocks"] == 1
        if general:
            w, a, b = F.get_chains()
            F.set_chains(w, a, b + 1)  # another plan than the created one
            assert F.pass_plan()["blocks"] == 0
        prm = [torch.tensor(x, dtype=torch.float64, device=F.device)
               for x in (F.lengths_to_level([np.maximum(t.length, 0.01) for t in trees]), [0.2] * P, [0.1] * P)]
        res = []
        for before in ("nll", "estep", "em"):
            print("single calls", n, K, P, general, before, flush=True)
            if before == "em":
                F.em(*prm, 1, 0.0)  # (parameters move)
                F.outside(prm[2])
                F.nll(*prm)
            elif before == "estep":
                res += _host(F.estep(*prm))
            else:
                res += _host([F.nll(*prm, site_llh=True), F.site_llh])
            res += _host(F.outside(prm[2]))
            res += _host(F.grad(*prm))
        out.append(res + _host(prm))
        F.close()
    for a, b in zip(*out):
        np.testing.assert_allclose(a, b, rtol=0, atol=1e-11 * max(1e-3, np.abs(b).max()))
