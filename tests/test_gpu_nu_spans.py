"""M-step nu solve where a problem's branches cross the spans of 256 that the
blocks of an evaluation take, started near the optimum (one or two
evaluations) and far from it (more): nu (1e-9 relative) and branch lengths
(1e-9) of the oracle's bisections, and the same bits for a problem alone as in
a forest of nine."""
import math

import numpy as np
import pytest
import torch
from test_gpu_mstep_edges import _oracle, _rows_for

from laml_amd import sim
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


def _spec(n):
    tree, Q, codes, _ = sim.make_problem(n, 4, 3, 5, 1.0, 0.1, 0.1, 7)
    return sim.problem_spec(tree, Q, codes)


def _mstep(sizes, seed, nu0):
    F = Forest([_spec(n) for n in sizes], device=0)
    node_prob = F.tree_prob[F.tree_of]
    counts = np.zeros((F.num_nodes, 5))
    rows = [_rows_for("generic", int((node_prob == p).sum()), 4, np.random.default_rng([seed, p]))
            for p in range(len(sizes))]
    for p in range(len(sizes)):
        counts[node_prob == p] = rows[p]
    P, dev = len(sizes), F.device
    d = torch.full((F.num_nodes,), 0.05, dtype=torch.float64, device=dev)
    nu = torch.full((P,), nu0, dtype=torch.float64, device=dev)
    phi = torch.full((P,), 0.1, dtype=torch.float64, device=dev)
    F.mstep(d, nu, phi, counts=torch.tensor(counts.reshape(-1), dtype=torch.float64, device=dev),
            rtilde=torch.full((P,), 3.0, dtype=torch.float64, device=dev))
    torch.cuda.synchronize()
    assert (F.mstep_status() == 0).all()
    dh, nuh = d.cpu().numpy(), nu.cpu().numpy()
    F.close()
    return rows, [dh[node_prob == p] for p in range(P)], nuh


@pytest.mark.parametrize("n", [2, 127, 128, 129, 256, 257])
@pytest.mark.parametrize("nu0", [0.25, 1e-4])
def test_nu_over_span_edges(n, nu0):
    sizes = [n, 3, 40, 128, 129, 5, 200, 11, 60]
    _, d1, nu1 = _mstep(sizes[:1], n, nu0)
    rows, d9, nu9 = _mstep(sizes, n, nu0)
    assert nu1[0] == nu9[0] and np.array_equal(d1[0], d9[0])
    for p in range(len(sizes)):
        wd, wnu = _oracle(rows[p], 4, nu0)
        np.testing.assert_allclose(d9[p], wd, rtol=1e-9)
        assert math.isclose(nu9[p], wnu, rel_tol=1e-9), (p, nu9[p], wnu)
