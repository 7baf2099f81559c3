"""M-steps in branch-length boxes whose upper bound lies past the lengths at
which expm1 overflows (709.8): the fastEM model's [1e-6, 1000] and one above,
from lengths at both bounds and inside, against bisection in long double on the
same expected counts (lengths and nu to 1e-9 relative, the M-step's stated
bar) -- the M-step entry, one EM step of forests that run in whole-problem
blocks and in the general passes, quartet-local EM, and fastEM from branches of
length zero."""
import numpy as np
import pytest
import torch

import mstep_reference as ref
from laml_amd import sim
from laml_amd.fastem import EMOptimizer
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu


def _dev(F, x):
    return torch.tensor(np.asarray(x, dtype=np.float64), dtype=torch.float64, device=F.device)


def _starts(n, dmin, dmax):
    x = np.full(n, 0.05)
    x[0::4], x[1::4], x[2::8] = dmin, dmax, 0.0
    return x


@pytest.mark.parametrize("dmin,dmax", [(1e-6, 1e3), (1e-3, 1e4)])
@pytest.mark.parametrize("nprob,nu0", [(1, 0.3), (3, 1e-4), (9, 0.3)])
def test_mstep(dmin, dmax, nprob, nu0):
    K = 30
    specs = []
    for p in range(nprob):
        t, Q, codes, _ = sim.make_problem(40 + 200 * (p == 1), K, 5, 20, 1.0, 0.1, 0.1, 60 + p)
        specs.append(sim.problem_spec(t, Q, codes))
    F = Forest(specs, device=torch.cuda.current_device(), dmin=dmin, dmax=dmax)
    rng = np.random.default_rng(4)
    counts = np.exp(rng.uniform(np.log(1e-5), np.log(K), (F.num_nodes, 5)))
    counts[::5, [0, 1, 3]] = 0.0  # silenced for certain: at a small nu these branches end at dmax
    d = _dev(F, _starts(F.num_nodes, dmin, dmax))
    nu, phi = _dev(F, [nu0] * nprob), _dev(F, [0.1] * nprob)
    print("wide box", dmin, dmax, nprob, nu0, flush=True)
    F.mstep(d, nu, phi, counts=_dev(F, counts.reshape(-1)), rtilde=_dev(F, [3.0] * nprob))
    torch.cuda.synchronize()
    assert F.mstep_status().tolist() == [0] * nprob
    node_prob = F.tree_prob[F.tree_of]
    for p in range(nprob):
        sel = node_prob == p
        wd, wnu = ref.mstep(counts[sel], K, nu0, dmin, dmax)
        np.testing.assert_allclose(d.cpu().numpy()[sel], wd, rtol=1e-9)
        np.testing.assert_allclose(nu[p].item(), wnu, rtol=1e-9)


@pytest.mark.parametrize("n,K", [(90, 24), (300, 70)])
def test_em_step(n, K):
    t, Q, codes, _ = sim.make_problem(n, K, 5, 20, 1.0, 0.1, 0.1, 70)
    F = Forest([sim.problem_spec(t, Q, codes)], device=torch.cuda.current_device(), dmin=1e-6, dmax=1e3)
    x = np.maximum(t.length, 0.01)
    x[::3] = 1e-6
    d, nu, phi = _dev(F, F.lengths_to_level([x])), _dev(F, [0.2]), _dev(F, [0.1])
    counts = F.estep(d, nu, phi)[0].view(-1, 5).cpu().numpy().copy()
    print("wide box EM", n, K, flush=True)
    F.em(d, nu, phi, 1, 0.0)
    wd, wnu = ref.mstep(counts, K, 0.2, 1e-6, 1e3)
    assert (wd < 100).all()
    np.testing.assert_allclose(d.cpu().numpy(), wd, rtol=1e-8)  # (counts of two kernels: to 1e-9)
    np.testing.assert_allclose(nu.item(), wnu, rtol=1e-8)


def test_quartet_em_from_the_lower_bound():
    t, Q, codes, _ = sim.make_problem(60, 40, 5, 20, 1.0, 0.1, 0.1, 80)
    F = Forest([sim.problem_spec(t, Q, codes)], device=torch.cuda.current_device(), dmin=1e-6, dmax=1e3)
    d, nu, phi = _dev(F, F.lengths_to_level([np.maximum(t.length, 0.01)])), _dev(F, [0.2]), _dev(F, [0.1])
    cand = []
    for u in range(F.num_leaves, F.num_nodes):
        v = F.parent[u]
        if v < 0:
            continue
        p = F.parent[v]
        s = -1 if p < 0 else (F.child0[p] if F.child1[p] == v else F.child1[p])
        C = F.child0[v] if F.child1[v] == u else F.child1[v]
        cand.append((p, s, F.child0[u], C, F.child1[u]))
    m = len(cand)
    F.estep(d, nu, phi)
    out = []
    for x in (1e-6, 1e-6 * (1 + 1e-9)):  # at the bound, just inside
        print("wide box quartet", x, flush=True)
        out.append(F.quartet_em(np.asarray(cand), np.full((m, 5), x), np.full(m, 31), np.zeros(m), nu, phi, 1, 0.0))
    assert (out[0][0] < 100).all() and (out[0][0] > 1e-3).any()
    # (the start differs by 1e-9, which the counts carry to the lengths)
    np.testing.assert_allclose(out[0][0].cpu().numpy(), out[1][0].cpu().numpy(), rtol=1e-6)
    np.testing.assert_allclose(out[0][1].cpu().numpy(), out[1][1].cpu().numpy(), rtol=1e-9)


def test_fastem_from_branches_of_length_zero():
    t, Q, codes, _ = sim.make_problem(100, 30, 3, 15, 1.0, 0.1, 0.1, 90)
    children = [[] if a < 0 else [int(a), int(b)] for a, b in zip(t.c0, t.c1)]
    order = [v for v in range(t.n_nodes) if not children[v]] + [v for v in range(t.n_nodes) if children[v]]
    new = {v: i for i, v in enumerate(order)}
    children = [[new[c] for c in children[v]] for v in order]
    q = np.zeros((len(Q), max(len(x) for x in Q)))
    for k, x in enumerate(Q):
        for j, pr in x.items():
            q[k, j - 1] = pr
    opt = EMOptimizer(q, np.maximum(codes, -1).astype(np.int64))
    mask = np.ones(len(children), dtype=bool)
    bl = np.full(len(children), 0.05)
    print("fastEM from zero", flush=True)
    want = opt.optimize({"children": children}, bl, 0.3, 0.3, mask)
    bl[::2] = 0.0
    got = opt.optimize({"children": children}, bl, 0.3, 0.3, mask)
    assert got["branch_lengths"].max() < 100 and want["branch_lengths"].max() < 100
    # (both stop where a step gains less than 1e-5 of the likelihood)
    assert abs(got["nllh"] - want["nllh"]) < 1e-2 * want["nllh"]
