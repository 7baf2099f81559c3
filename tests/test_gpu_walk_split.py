"""The level where the hybrid passes' walk takes over depends on the number of
trees and site chunks: likelihoods equal to level launches' bit for bit, counts
and dropout sums to 1e-12 (another order of sums over chunks)."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,n,K", [(1, 60, 70), (1, 300, 20), (3, 200, 65), (9, 30, 40), (40, 25, 33), (30, 40, 16),
                                   (520, 4, 70)])
def test_walk_split_equals_levels(T, n, K):
    specs, trees = [], []
    for i in range(T):
        t, Q, codes, _ = sim.make_problem(n + i % 7, K - i % 3, 3, 9, 1.0, 0.1, 0.15, 40 + i)
        specs.append(sim.problem_spec(t, Q, codes))
        trees.append(t)
    F = Forest(specs, device=torch.cuda.current_device())
    d = torch.tensor(F.lengths_to_level([np.maximum(t.length, 0.005) for t in trees]), dtype=torch.float64,
                     device=F.device)
    nu = torch.full((T,), 0.2, dtype=torch.float64, device=F.device)
    phi = torch.full((T,), 0.3, dtype=torch.float64, device=F.device)
    out = []
    for mode in (PASS_HYBRID, PASS_LEVELS):
        F.set_pass_mode(mode)
        F.set_chains(1 if mode == PASS_HYBRID else 0)  # (a plan of its own: no whole-problem blocks)
        counts, rt, nll = [x.cpu().numpy().copy() for x in F.estep(d, nu, phi)]
        out.append((nll, counts, rt))
    F.close()
    assert np.array_equal(out[0][0], out[1][0])
    np.testing.assert_allclose(out[0][1], out[1][1], rtol=1e-12, atol=1e-12)
    np.testing.assert_allclose(out[0][2], out[1][2], rtol=1e-12, atol=1e-12)
