"""Quartet EM at the site counts where the block's width changes (one
wavefront per 64 sites up to eight, more in turns): NLL (1e-9 relative),
branch lengths (1e-6) and EM iteration counts of the CPU oracle's EM of the
same candidates."""
import math
import random

import pytest
from test_gpu_quartet import _search_state

from laml_amd.quartet import QuartetScorer, _clade_index
from laml_amd.solvers import DEFAULT_STRATEGY, EM_solver
from laml_amd.topology_search import _nni_swap, _nni_unswap
from oracle.em_oracle import OracleEM, postorder
from oracle.pmm_ref import RefProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1030])
def test_quartet_em_over_block_widths(K):
    ts, msa, Q = _search_state(10, K, 5)
    random.seed(1)
    sel = ts._list_moves()[::5][:3]
    scorer = QuartetScorer(ts, DEFAULT_STRATEGY, EM_solver)
    res = scorer.score(sel)
    iters = scorer.iters.copy()
    below = _clade_index(ts.treeList_obj[0])[1]
    for i, (mv, (score, lazy)) in enumerate(zip(sel, res)):
        u, v, uc, w = mv
        st = ts._local_strategy(u, DEFAULT_STRATEGY)
        _nni_swap(u, v, uc, w)
        nwks = [t.newick() for t in ts.treeList_obj]
        _nni_unswap(u, v, uc, w)
        o = OracleEM(nwks, msa, Q)
        o.mark_fixed(st["fixed_brlen"])
        x0 = o.ini_all(random.Random(1234), fixed_phi=st["fixed_phi"], fixed_nu=st["fixed_nu"])
        o.x2params(x0, fixed_phi=st["fixed_phi"], fixed_nu=st["fixed_nu"])
        rp, d0 = RefProblem.from_oracle(o)
        nll, it, od, _, _ = rp.em(d0, o.nu, o.phi, opt_nu=False, opt_phi=False)
        assert math.isclose(-score, nll, rel_tol=1e-9), (i, -score, nll)
        assert int(iters[i]) == it, (i, int(iters[i]), it)
        blow, length = {}, {}
        for nd, x in zip([nd for r in o.trees for nd in postorder(r)], od):
            cl = frozenset([nd.label]) if not nd.children else frozenset().union(*[blow[id(c)] for c in nd.children])
            blow[id(nd)] = cl
            length[cl] = x
        A = next(x for x in u.child_nodes() if x is not uc)
        cA, cW, cC = below[id(A)], below[id(w)], below[id(uc)]
        for j, cl in enumerate([cA, cW, cA | cW, cC, cA | cW | cC]):
            assert abs(lazy.lengths[j] - length[cl]) <= 1e-6 * max(1.0, length[cl]), (i, j, lazy.lengths[j], length[cl])
    scorer.close()
