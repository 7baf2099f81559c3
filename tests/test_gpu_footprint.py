"""The admission estimate plus the per-forest allowance bounds the device memory
of forests that run in whole-problem blocks, whose tables pad every level of a
tree to a wavefront's cells: batches of Yule trees, and of caterpillars, whose
levels hold one node each."""
import pytest
import torch

from laml_amd import sim
from laml_amd.forest import Forest
from laml_amd.serving import FOREST_FIXED_BYTES, estimate_forest_bytes
from test_gpu_chains import _problem

pytestmark = pytest.mark.gpu


def _used(specs):
    dev = torch.cuda.current_device()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info(dev)
    F = Forest(specs, device=dev)
    assert F.pass_plan()["blocks"] == 1
    d = torch.full((F.num_nodes,), 0.05, dtype=torch.float64, device=F.device)
    nu = torch.full((F.num_problems,), 0.5, dtype=torch.float64, device=F.device)
    phi = nu.clone()
    F.em(d, nu, phi, 3, 1e-8)
    F.estep(d, nu, phi)
    F.nll(d, nu, phi)
    F.grad(d, nu, phi)
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info(dev)[0]
    F.close()
    return used


@pytest.mark.parametrize("kind,n,K,P", [("caterpillar", 900, 8, 16), ("caterpillar", 900, 8, 100),
                                        ("caterpillar", 250, 30, 100), ("yule", 120, 64, 400), ("yule", 250, 30, 400),
                                        ("yule", 8, 8, 2000), ("yule", 700, 8, 16)])
def test_estimate_bounds_block_forests(kind, n, K, P):
    base = [_problem(kind, n, K, 3 + i) for i in range(min(P, 4))]
    specs = [sim.problem_spec(*base[i % len(base)][:3]) for i in range(P)]
    _used(specs[:1])  # (the first calls load code and the kernels' scratch memory)
    used = _used(specs)
    est = estimate_forest_bytes(specs) + FOREST_FIXED_BYTES
    print("footprint", kind, n, K, P, est, used, flush=True)
    assert est >= used
