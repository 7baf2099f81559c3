"""EM steps in whole-problem blocks report failures and set phi as the general
passes do: a branch without a finite length (an unbounded box, entered from its
lower bound) fails the branch solve and leaves phi alone; a dropout sum that is
not a number makes phi one and fails no branch.  The other problems of the
forest are untouched."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("failure", ["branch", "dropout"])
@pytest.mark.parametrize("flags", [3, 1, 2])
def test_status_and_phi_as_in_the_general_passes(failure, flags):
    specs, trees = [], []
    for i in range(3):
        t, Q, codes, _ = sim.make_problem(40 + 9 * i, 20, 3, 9, 1.0, 0.1, 0.15, 140 + i)
        specs.append(sim.problem_spec(t, Q, codes, flags=flags))
        trees.append(t)
    out = []
    for mode in (PASS_HYBRID, PASS_LEVELS):
        F = Forest(specs, device=torch.cuda.current_device(), dmin=0.005,
                   dmax=float("inf") if failure == "branch" else 10.0)
        lengths = [np.maximum(t.length, 0.01) for t in trees]
        phi0 = [0.3, 0.3, 0.3]
        if failure == "branch":
            lengths[1][:] = 0.005  # (every branch that the data want longer)
        else:
            phi0[1] = float("nan")
        d = torch.tensor(F.lengths_to_level(lengths), dtype=torch.float64, device=F.device)
        nu = torch.full((3,), 0.2, dtype=torch.float64, device=F.device)
        phi = torch.tensor(phi0, dtype=torch.float64, device=F.device)
        F.set_pass_mode(mode)
        assert F.pass_plan()["blocks"] == (mode == PASS_HYBRID)
        print("problem status", failure, flags, mode, flush=True)
        F.em(d, nu, phi, 1, 0.0)
        out.append((F.mstep_status(), phi.cpu().numpy(), nu.cpu().numpy(), d.cpu().numpy()))
        F.close()
    print(out[0][:3], out[1][:3], flush=True)
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_allclose(out[0][1], out[1][1], rtol=1e-9)  # (NaN equals NaN)
    sound = [0, 2]
    assert (out[0][0][sound] == 0).all()
    np.testing.assert_allclose(out[0][2][sound], out[1][2][sound], rtol=1e-9)
    if failure == "branch":
        assert out[0][0][1] & 1 and np.isfinite(out[0][1]).all()
        np.testing.assert_allclose(out[0][3], out[1][3], rtol=1e-8)
    else:
        assert not out[0][0][1] & 1
