"""Calls captured into a HIP graph by the caller and replayed with other
parameters in the same buffers, between eager calls that read the state they
leave: posteriors, quartet EM, outside pass and gradient after a replay equal
those of a fresh forest that ran the same calls eagerly (1e-12: whole-problem
blocks and general passes may both be in play).  Forests: in whole-problem
blocks (32 and 64 lanes a row), in level launches and walk alone, with outside
chains, with clades."""
import numpy as np
import pytest
import torch

from laml_amd import sim
from laml_amd._lib import PASS_HYBRID, PASS_LEVELS
from laml_amd.forest import Forest

pytestmark = pytest.mark.gpu

KINDS = {"block32": (90, 24, {}), "block64": (100, 40, {}), "levels": (300, 70, {}),
         "chains": (300, 130, {"LAML_CHAINS": "1"}), "clades": (400, 130, {"LAML_CLADES": "16"})}
CLOSE = dict(rtol=1e-12, atol=1e-13)


class Case:
    def __init__(self, kind, monkeypatch):
        n, K, env = KINDS[kind]
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        t, Q, codes, _ = sim.make_problem(n, K, 3, 12, 1.0, 0.1, 0.15, 31)
        self.spec = sim.problem_spec(t, Q, codes)
        self.F = self.forest()
        base = self.F.lengths_to_level([np.maximum(t.length, 0.01)])
        rng = np.random.default_rng(5)
        self.points = [(base * rng.uniform(0.5, 2.0, len(base)), 0.1 + 0.1 * i, 0.3 - 0.05 * i) for i in range(4)]
        self.d, self.nu, self.phi = (torch.zeros(m, dtype=torch.float64, device=self.F.device)
                                     for m in (len(base), 1, 1))

    def forest(self):
        return Forest([self.spec], device=torch.cuda.current_device())

    def set(self, i):
        x = self.points[i]
        self.d.copy_(torch.tensor(x[0]))
        self.nu.fill_(x[1])
        self.phi.fill_(x[2])
        return self.d, self.nu, self.phi

    def candidates(self):
        F = self.F
        out = []
        for u in range(F.num_leaves, F.num_nodes, 5):
            v = F.parent[u]
            if v < 0:
                continue
            p = F.parent[v]
            s = -1 if p < 0 else (F.child0[p] if F.child1[p] == v else F.child1[p])
            out.append((p, s, F.child0[u], F.child0[v] if F.child1[v] == u else F.child1[v], F.child1[u]))
        m = len(out)
        return np.asarray(out), np.full((m, 5), 0.05), np.full(m, 31), np.zeros(m)


def _capture(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    return g


def _post(F, phi):
    return [x.copy() for pair in F.posteriors(phi) for x in pair]


def _host(xs):
    return [x.cpu().numpy().copy() for x in xs]


def _same(got, want):
    for a, b in zip(got, want):
        np.testing.assert_allclose(a, b, **CLOSE)


@pytest.mark.parametrize("kind", list(KINDS))
def test_readers_after_a_replayed_estep(kind, monkeypatch):
    c = Case(kind, monkeypatch)
    q = c.candidates()
    prm = c.set(0)
    g = _capture(lambda: c.F.estep(*prm))
    for i in (3, 1, 0):  # (nothing but posteriors between the replays)
        c.set(i)
        g.replay()
        got = _post(c.F, c.phi)
        E = c.forest()
        E.estep(*prm)
        want = _post(E, c.phi)
        E.close()
        _same(got, want)
    for i in (0, 1, 2):
        c.set(i)
        print("replayed estep", kind, i, flush=True)
        g.replay()
        got = [c.F.counts.cpu().numpy().copy()]
        got += _post(c.F, c.phi)
        got += _host(c.F.quartet_em(*q, c.nu, c.phi, 5, 0.0))[:2]
        got += _host(c.F.outside(c.phi))
        got += _host(c.F.grad(*prm))
        E = c.forest()
        want = [E.estep(*prm)[0].cpu().numpy().copy()]
        want += _post(E, c.phi)
        E.estep(*prm)
        want += _host(E.quartet_em(*q, c.nu, c.phi, 5, 0.0))[:2]
        E.nll(*prm)
        want += _host(E.outside(c.phi))
        want += _host(E.grad(*prm))
        E.close()
        _same(got, want)
    c.F.close()


@pytest.mark.parametrize("kind", list(KINDS))
def test_readers_after_a_replayed_likelihood(kind, monkeypatch):
    """Between the replays, an E-step and posteriors at other parameters."""
    c = Case(kind, monkeypatch)
    prm = c.set(0)
    g = _capture(lambda: c.F.nll(*prm))
    other = tuple(x.clone() for x in c.set(3))
    for i in (0, 1):
        c.set(i)
        c.F.estep(*other)
        _post(c.F, other[2])
        print("replayed likelihood", kind, i, flush=True)
        g.replay()
        got = _host(c.F.outside(c.phi)) + _host(c.F.grad(*prm))
        E = c.forest()
        E.nll(*prm)
        want = _host(E.outside(c.phi)) + _host(E.grad(*prm))
        E.close()
        _same(got, want)
    c.F.close()


@pytest.mark.parametrize("kind", list(KINDS))
def test_replayed_quartet_round_after_new_esteps(kind, monkeypatch):
    c = Case(kind, monkeypatch)
    q = c.candidates()
    dev = [torch.as_tensor(np.ascontiguousarray(x, dtype=t), device=c.F.device)
           for x, t in zip(q, (np.int32, np.float64, np.uint8, np.float64))]
    m = len(q[0])
    out = torch.empty((m, 5), dtype=torch.float64, device=c.F.device)
    nll = torch.empty(m, dtype=torch.float64, device=c.F.device)
    it = torch.empty(m, dtype=torch.int32, device=c.F.device)
    from laml_amd import _lib

    def quartet():
        _lib.check(c.F._lib.laml_quartet_em(c.F.handle, m, *[_lib.ptr(x) for x in dev], _lib.ptr(c.nu),
                                            _lib.ptr(c.phi), 5, 0.0, _lib.ptr(out), _lib.ptr(nll), _lib.ptr(it),
                                            c.F.stream()))

    prm = c.set(0)
    c.F.estep(*prm)
    _post(c.F, c.phi)
    g = _capture(quartet)
    for i in (1, 2):
        c.set(i)
        print("replayed quartet round", kind, i, flush=True)
        c.F.estep(*prm)
        g.replay()
        E = c.forest()
        E.estep(*prm)
        want = _host(E.quartet_em(*q, c.nu, c.phi, 5, 0.0))[:2]
        E.close()
        _same(_host((out, nll)), want)
    c.F.close()


@pytest.mark.parametrize("kind", ["block32", "block64"])
def test_outside_after_a_replay_in_another_plan(kind, monkeypatch):
    """An E-step captured in level launches, replayed after an eager
    likelihood of other parameters in whole-problem blocks."""
    c = Case(kind, monkeypatch)
    prm = c.set(0)
    c.F.set_pass_mode(PASS_LEVELS)
    g = _capture(lambda: c.F.estep(*prm))
    c.F.set_pass_mode(PASS_HYBRID)
    other = tuple(x.clone() for x in c.set(3))
    c.set(1)
    c.F.nll(*other)
    print("replayed in another plan", kind, flush=True)
    g.replay()
    got = _host(c.F.outside(c.phi)) + _host(c.F.grad(*prm))
    E = c.forest()
    E.nll(*prm)
    want = _host(E.outside(c.phi)) + _host(E.grad(*prm))
    E.close()
    _same(got, want)
    # and a likelihood captured in blocks, read in level launches
    g = _capture(lambda: c.F.nll(*prm))
    c.F.set_pass_mode(PASS_LEVELS)
    c.F.nll(*other)
    c.set(2)
    g.replay()
    got = _host(c.F.outside(c.phi)) + _host(c.F.grad(*prm))
    E = c.forest()
    E.nll(*prm)
    want = _host(E.outside(c.phi)) + _host(E.grad(*prm))
    E.close()
    _same(got, want)
    c.F.close()


@pytest.mark.parametrize("call", ["estep", "em"])
def test_readers_after_a_replay_with_fused_cherries(call, monkeypatch):
    """An E-step, or an EM of no steps (a likelihood), captured with fused
    cherries (whose rows it does not write) and replayed after an eager E-step
    without."""
    c = Case("levels", monkeypatch)
    prm = c.set(0)
    c.F.set_pass_mode(PASS_LEVELS)
    c.F.set_fusion(True)
    assert c.F.fusion()
    g = _capture(lambda: c.F.estep(*prm) if call == "estep" else c.F.em(*prm, 0, 0.0))
    c.F.set_fusion(False)
    other = tuple(x.clone() for x in c.set(3))
    c.set(1)
    c.F.estep(*other)
    g.replay()
    got = _post(c.F, c.phi) if call == "estep" else []
    got += _host(c.F.outside(c.phi)) + _host(c.F.grad(*prm))
    E = c.forest()
    E.set_pass_mode(PASS_LEVELS)
    E.estep(*prm)
    want = _post(E, c.phi) if call == "estep" else []
    want += _host(E.outside(c.phi)) + _host(E.grad(*prm))
    E.close()
    _same(got, want)
    c.F.close()
