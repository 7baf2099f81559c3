"""Outside states kept conditional on the data (a0, aX) at the site patterns
where they differ in kind: every leaf missing, one state everywhere (no node
is 'z', the root included), one half of the tree missing, explicit -1
entries, one unedited leaf, random.  Expected counts, dropout sums and the
gradient against the C oracle, posteriors against the Python oracle, in level
launches, hybrid and tree-walk passes and with outside chains, at nu = 0 (a
missing clade's inside values then shrink to phi^leaves) and nu = 0.25.
Tolerance: 1e-9 relative (the stated bar for counts), 1e-9 absolute for
posteriors."""
import math

import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import CHAINS_OUTSIDE, PASS_HYBRID, PASS_LEVELS, PASS_TREES
from laml_amd.forest import Forest
from oracle import pmm_ref
from oracle.em_oracle import OracleEM, postorder

pytestmark = pytest.mark.gpu


def _problem(n, K):
    tree, Q, codes, _ = sim.make_problem(n, K, 2, 6, 1.0, 0.2, 0.2, 900 + K)
    half = n // 2
    codes[:, 0] = -1
    codes[:, 1] = 1
    codes[:half, 2] = -1
    codes[half:, 2] = 2
    codes[:, 3] = np.where(np.arange(n) % 3 == 0, -2, 1)
    codes[:, 4] = 1
    codes[n - 1, 4] = 0
    codes[:half, 5] = -1
    return tree, Q, codes


@pytest.mark.parametrize("nu", [0.0, 0.25])
@pytest.mark.parametrize("n,K", [(70, 8), (70, 20), (300, 70)])
def test_counts_and_posteriors_at_special_sites(n, K, nu):
    tree, Q, codes = _problem(n, K)
    phi = 0.3
    if nu == 0.0:
        codes = np.where(codes == -2, -1, codes).astype(np.int16)  # silencing is impossible
    d = np.maximum(tree.length, 0.005)
    p = pmm_ref.RefProblem(tree.c0, tree.c1, tree.parent, codes, Q, None, 1.0 / (K * n))
    rnll, rcounts, _, Rt = p.estep(d, nu, phi)
    msa = {c: [{-1: "?", -2: -1}.get(int(x), int(x)) for x in codes[i]] for i, c in enumerate(tree.leaf_names)}
    o = OracleEM([tree.newick()], msa, Q, nu=nu, phi=phi)
    for v, x in zip(postorder(o.trees[0]), d):
        v.edge_length = float(x)
    o.az_partition()
    o.estep()
    want0 = np.exp([v.a["post0"] for v in postorder(o.trees[0])])
    wantS = np.exp([v.a["post1"] for v in postorder(o.trees[0])])
    dev = torch.cuda.current_device()
    for mode in (PASS_LEVELS, PASS_HYBRID, PASS_TREES):
        for chains in (0, CHAINS_OUTSIDE):
            print("case", n, K, nu, mode, chains, flush=True)
            F = Forest([sim.problem_spec(tree, Q, codes)], device=dev)
            F.set_pass_mode(mode)
            F.set_chains(chains, 0, 0)
            dt = torch.tensor(F.lengths_to_level([d]), dtype=torch.float64, device=F.device)
            nut, phit = (torch.tensor([x], dtype=torch.float64, device=F.device) for x in (nu, phi))
            counts, rt, nll = F.estep(dt, nut, phit)
            got = np.empty((F.num_nodes, 5))
            got[F.order] = counts.view(-1, 5).cpu().numpy()
            np.testing.assert_allclose(got, rcounts, rtol=1e-9, atol=1e-9)
            assert math.isclose(rt.item(), Rt, rel_tol=1e-9, abs_tol=1e-10)
            assert math.isclose(nll.item(), rnll, rel_tol=1e-9)
            (l0, i0), (lS, iS) = F.posteriors(phit)
            for (leaf, inner), want in (((l0, i0), want0), ((lS, iS), wantS)):
                post = np.empty((F.num_nodes, K))
                post[F.order] = np.concatenate([leaf, inner]).reshape(-1, K)
                np.testing.assert_allclose(post, want, rtol=0, atol=1e-9)
            F.close()
