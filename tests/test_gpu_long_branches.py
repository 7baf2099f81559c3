"""Branches so long or short that likelihoods leave the range of a double:
cherries whose two branches hold lengths of 297 (with unedited leaves the
product of the two edges is about 1e-310, whose reciprocal no double holds),
single branches of length 300 and of 1e-300.  Posteriors, counts and
likelihoods against the model in long double (1e-9: a product of 1e-310 keeps
some 13 decimals), in whole-problem blocks, level launches and walk, outside
chains and clades; and an EM step stays finite."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd.forest import Forest
from long_double_model import evaluate

pytestmark = pytest.mark.gpu

KINDS = {"block32": (40, 20, {}), "block64": (40, 45, {}), "general": (90, 70, {}),
         "chains": (120, 66, {"LAML_CHAINS": "1", "LAML_TOP_MAX_NODES": "4"}),
         "clades": (120, 66, {"LAML_CLADES": "16", "LAML_TOP_MAX_NODES": "4"})}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("shape", ["cherries", "single", "short"])
def test_long_and_short_branches(kind, shape, monkeypatch):
    n, K, env = KINDS[kind]
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    t, Q, codes, _ = sim.make_problem(n, K, 3, 12, 1.0, 0.1, 0.15, 5)
    codes[:, 0], codes[:, 1], codes[::3, 2] = 0, 1, -2
    N = t.n_nodes
    x = np.maximum(t.length, 0.01)
    cherries = [v for v in range(N) if t.c0[v] >= 0 and t.c0[t.c0[v]] < 0 and t.c0[t.c1[v]] < 0]
    if shape == "cherries":
        for v in cherries[::3]:
            x[[t.c0[v], t.c1[v]]] = 297.0
    else:
        x[np.random.default_rng(2).integers(0, N - 1, n // 12)] = 300.0 if shape == "single" else 1e-300
    F = Forest([sim.problem_spec(t, Q, codes)], device=torch.cuda.current_device())
    prm = [torch.tensor(y, dtype=torch.float64, device=F.device) for y in (F.lengths_to_level([x]), [0.2], [0.1])]
    print("long branches", kind, shape, flush=True)
    counts = F.estep(*prm)[0].view(-1, 5).cpu().numpy().copy()
    post = [np.concatenate(pair).reshape(N, K) for pair in F.posteriors(prm[2])]
    F.nll(*prm, site_llh=True)
    site = F.site_llh.cpu().numpy().copy()
    outside = F.outside(prm[2])[0].view(-1, 5).cpu().numpy().copy()
    F.em(*prm, 1, 0.0)
    em = [y.cpu().numpy() for y in prm]
    p0, pS, want, llh = evaluate(t, Q, codes, x, 0.2, 0.1)
    got = np.empty((4, N, max(K, 5)))
    for i, y in enumerate((counts, outside, *post)):
        got[i, F.order, :y.shape[1]] = y
    np.testing.assert_allclose(site, llh.astype(float), rtol=1e-9)
    np.testing.assert_allclose(got[0, :, :5], want.astype(float), rtol=0, atol=1e-9 * K)
    np.testing.assert_allclose(got[1, :, :5], want.astype(float), rtol=0, atol=1e-9 * K)
    np.testing.assert_allclose(got[2, :, :K], p0.astype(float), rtol=0, atol=1e-9)
    np.testing.assert_allclose(got[3, :, :K], pS.astype(float), rtol=0, atol=1e-9)
    assert all(np.isfinite(y).all() for y in em)
    F.close()
