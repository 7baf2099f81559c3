"""The level from which the hybrid passes walk: reported for the current pass
mode, taken as set, and the created plan again when its own level is set."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.autotune import current_plan
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K,P", [(600, 70, 1), (300, 130, 12), (90, 30, 1), (300, 20, 12)])
def test_walk_level(n, K, P):
    specs, trees = [], []
    for i in range(P):
        t, Q, codes, _ = sim.make_problem(n, K, 3, 9, 1.0, 0.1, 0.15, 40 + i)
        specs.append(sim.problem_spec(t, Q, codes))
        trees.append(t)
    F = Forest(specs, device=torch.cuda.current_device())
    d = torch.tensor(F.lengths_to_level([np.maximum(t.length, 0.005) for t in trees]), dtype=torch.float64,
                     device=F.device)
    nu = torch.full((P,), 0.2, dtype=torch.float64, device=F.device)
    phi = torch.full((P,), 0.3, dtype=torch.float64, device=F.device)
    created, walk = F.pass_plan(), F.get_shapes()[2]
    assert F.pass_mode() == PASS_HYBRID and walk == created["walk_level"]
    F.set_pass_mode(PASS_LEVELS)
    fused = F.get_shapes()[2]
    assert F.pass_plan()["walk_level"] == fused
    F.set_pass_mode(PASS_HYBRID)
    want = [x.cpu().numpy().copy() for x in F.estep(d, nu, phi)]
    for top in sorted({1, 2, fused, walk, max(1, walk - 1), min(walk + 1, F.num_levels), F.num_levels}):
        F.set_shapes(top_level=top)
        assert F.get_shapes()[2] == top and F.pass_plan()["walk_level"] == top
        assert F.pass_plan()["blocks"] == (created["blocks"] if top == walk else 0)
        print("walk level", n, K, P, top, flush=True)
        for a, b in zip(F.estep(d, nu, phi), want):
            np.testing.assert_allclose(a.cpu().numpy(), b, rtol=1e-12, atol=1e-12)
    F.set_shapes(top_level=walk)
    assert F.pass_plan()["blocks"] == created["blocks"]
    for a, b in zip(F.estep(d, nu, phi), want):
        np.testing.assert_array_equal(a.cpu().numpy(), b)
    # the created plan, noted and applied
    plan = current_plan(F)
    assert plan.top_level == walk
    plan.apply(F)
    assert F.pass_plan()["walk_level"] == walk and F.pass_plan()["blocks"] == created["blocks"]
    F.close()


def test_reported_chains_follow_the_outside_pass(monkeypatch):
    t, Q, codes, _ = sim.make_problem(7000, 300, 3, 12, 1.0, 0.1, 0.1, 8)
    for clades, chains in (("32", 0), ("0", 1)):
        monkeypatch.setenv("LAML_CLADES", clades)
        F = Forest([sim.problem_spec(t, Q, codes)], device=torch.cuda.current_device())
        assert F.chains() == chains and F.get_chains()[0] == 1
        F.set_chains(1, 0, 0)  # other chains than the created plan's run as chains
        assert F.chains() == 1
        F.close()
