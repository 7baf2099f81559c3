"""Rows formed again for a reader, after the launch plan was changed since the
call that left none (EM and likelihoods in whole-problem blocks): with inside
chains, whose plan is not built yet, and with fused cherries.  Posteriors and
quartet EM equal those after an E-step at the same parameters (1e-12)."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("change", ["inside chains", "both chains", "fusion", "fusion off again", "tree walk", "none"])
@pytest.mark.parametrize("n,K", [(110, 60), (60, 40), (90, 20)])
@pytest.mark.timeout(60)
def test_readers_after_a_change_of_plan(change, n, K):
    t, Q, codes, _ = sim.make_problem(n, K, 3, 12, 1.0, 0.1, 0.15, 12)
    spec = sim.problem_spec(t, Q, codes)
    F = Forest([spec], device=torch.cuda.current_device())
    d = torch.tensor(F.lengths_to_level([np.maximum(t.length, 0.01)]), dtype=torch.float64, device=F.device)
    nu = torch.full((1,), 0.2, dtype=torch.float64, device=F.device)
    phi = torch.full((1,), 0.1, dtype=torch.float64, device=F.device)
    u = int(F.num_nodes - 2)
    v, p = int(F.parent[u]), -1
    q = np.asarray([[p, -1, F.child0[u], F.child0[v] if F.child1[v] == u else F.child1[v], F.child1[u]]])
    args = (q, np.full((1, 5), 0.05), np.full(1, 31), np.zeros(1), nu, phi, 5, 0.0)
    F.estep(d, nu, phi)
    want = [x.copy() for pair in F.posteriors(phi) for x in pair] + [x.cpu().numpy() for x in F.quartet_em(*args)[:2]]
    # other rows, then a likelihood (in a block) at the parameters above
    F.estep(0.5 * d, nu, phi)
    F.nll(d, nu, phi)
    if change.endswith("chains"):
        F.set_chains(2 if change.startswith("inside") else 3, 0, 0)
    elif change.startswith("fusion"):
        F.set_pass_mode(PASS_LEVELS)
        F.set_fusion(True)
        if change.endswith("again"):
            F.set_fusion(False)
    elif change == "tree walk":
        F.set_pass_mode(1)
    for reader in ("posteriors", "quartet"):
        print("rows again", change, n, K, reader, flush=True)
        if reader == "posteriors":
            got = [x.copy() for pair in F.posteriors(phi) for x in pair]
            ref = want[:4]
        else:
            got = [x.cpu().numpy() for x in F.quartet_em(*args)[:2]]
            ref = want[4:]
        for a, b in zip(got, ref):
            np.testing.assert_allclose(a, b, rtol=1e-12, atol=1e-13)
    # the passes of the changed plan still run
    F.nll(d, nu, phi)
    F.set_pass_mode(PASS_HYBRID)
    F.close()
