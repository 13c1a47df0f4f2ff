"""
The linear reverse pass (Jacobians of a range of steps together, then only
the products step by step) against the kernels that apply the cell VJP step
by step: tiles of one cell to several with a short last one, segments longer
and shorter than a range of steps and than an exchange, fields, uncoupled
cells, Rush-Larsen and a second model. The two differ by the order of a few
additions per step.
"""
import numpy as np
import pytest

import myokit_amd as myokit
from myokit_amd.adjoint import TissueAdjoint
from tests.helpers import Scenario

pytestmark = pytest.mark.gpu


def _both(sc, fields, probes, dur, K):
    res = []
    for linear in (1, 0):
        s = sc.product(myokit.DOUBLE_PRECISION)
        for name, v in fields.items():
            s.set_field(name, v)
        s.set_engine_option('adj_linear', linear)
        adj = TissueAdjoint(s, probes, checkpoint_every=K)
        n = adj.n_steps(dur)
        target = -60.0 + 30 * np.sin(np.arange(n * len(probes))).reshape(
            n, len(probes))
        loss, g, dgx, dgy = adj.loss_and_gradient(dur, target)
        kind = adj.reverse_kernel()[0]
        assert (kind == 'linear') == bool(linear), kind
        assert dgy == 0
        res.append((loss, dgx, {k: np.array(v) for k, v in g.items()}))
    (l1, x1, g1), (l2, x2, g2) = res
    assert l1 == pytest.approx(l2, rel=1e-13)
    # a step's products round at 2^-53 of its largest terms, a few terms per
    # step: 1e-12 of the largest gradient over some hundred steps
    for k in g1:
        np.testing.assert_allclose(g1[k], g2[k], rtol=1e-9,
                                   atol=1e-12 * np.max(np.abs(g2[k])))
    # the conductance's gradient cancels over the cells
    assert x1 == pytest.approx(x2, rel=1e-7, abs=1e-9)


@pytest.mark.parametrize('n,rl,K', [
    (1, False, 1000), (2, True, 37), (64, False, 16), (65, False, 17),
    (161, True, 1000), (200, False, 1), (513, False, 300)])
def test_cable(n, rl, K):
    rng = np.random.default_rng(n)
    sc = Scenario('lr1991', n, rl=rl, dt=0.005, gx=9.5, paced=(4, 1, 0, 0))
    fields = {'ina.gNa': 16 * rng.uniform(0.8, 1.2, n),
              'ica.gCa': 0.09 * rng.uniform(0.8, 1.2, n)}
    _both(sc, fields, sorted({0, n // 2, n - 1}), 2.6, K)


def test_conductance_field_uncoupled_and_other_model():
    rng = np.random.default_rng(4)
    sc = Scenario('lr1991', 130, dt=0.005, paced=(4, 1, 0, 0),
                  conductance_field=(rng.uniform(2, 12, 129), None))
    _both(sc, {'ina.gNa': 16 * rng.uniform(0.8, 1.2, 130)}, [3, 129], 2.0, 90)
    sc = Scenario('lr1991', 100, dt=0.005, diffusion=False,
                  events=((1, 0, 0.5, 1000, 0),))
    _both(sc, {'ina.gNa': 16 * rng.uniform(0.8, 1.2, 100)}, [0, 99], 2.0, 90)
    sc = Scenario('br1977', 70, dt=0.005, gx=9.5, paced=(4, 1, 0, 0))
    _both(sc, {}, [0, 69], 2.0, 90)


# below the shortest segments whose gain outweighs their cooperative launches
# a gradient takes the kernels without those, and on small sheets with a
# conductance field wherever segments are recomputed
@pytest.mark.parametrize('shape,prec,field,kinds', [
    (40, 64, False, {2: 'block', 3: 'linear'}),
    (200, 64, False, {9: 'block', 10: 'linear'}),
    (1000, 64, True, {9: 'step-overlap', 10: 'linear'}),
    (1000, 32, False, {15: 'step-overlap', 16: 'step'}),
    ((40, 20), 32, False, {19: 'step-overlap', 20: 'sheet'}),
    ((40, 20), 64, False, {47: 'step-overlap', 48: 'sheet'}),
    ((40, 20), 64, True, {64: 'step-overlap', 300: 'step'}),
    ((300, 130), 64, True, {15: 'step', 16: 'step'}),
])
def test_segment_lengths(shape, prec, field, kinds):
    rng = np.random.default_rng(3)
    n = int(np.prod(shape))
    if not field:
        g = None
    elif isinstance(shape, tuple):
        g = (rng.uniform(2, 12, (shape[1], shape[0] - 1)),
             rng.uniform(2, 12, (shape[1] - 1, shape[0])))
    else:
        g = (rng.uniform(2, 12, n - 1), None)
    res = []
    for K, kind in list(kinds.items()) + [(7, None)]:
        s = Scenario('lr1991', shape, dt=0.005, gx=9.5, gy=6.0,
                     paced=(4, 20, 0, 0), conductance_field=g).product(prec)
        s.set_field('ina.gNa', 16 * np.linspace(0.8, 1.2, n).reshape(
            shape[::-1] if isinstance(shape, tuple) else (n,)))
        if kind is None:
            s.set_tuning(driver='grid')
            s.set_engine_option('adj_linear', 0)
        probe = [(0, 0)] if isinstance(shape, tuple) else [0]
        adj = TissueAdjoint(s, probe, checkpoint_every=K)
        target = np.full((adj.n_steps(1.0), 1), -60.0)
        loss, grad, dgx, dgy = adj.loss_and_gradient(1.0, target)
        if kind is not None:
            assert adj.reverse_kernel()[0] == kind
        res.append((loss, dgx, dgy, np.array(grad['ina.gNa'])))
    # against the one-step kernels on the grid driver: sums in another order
    # (single precision: states and adjoints of 200 steps, rounded at 6e-8)
    rel = 1e-9 if prec == 64 else 1e-4
    for l, x, y, g in res[:-1]:
        l0, x0, y0, g0 = res[-1]
        assert l == pytest.approx(l0, rel=rel)
        np.testing.assert_allclose(g, g0, rtol=0,
                                   atol=rel * np.max(np.abs(g0)))
        # (the conductances' gradients cancel over the cells)
        assert x == pytest.approx(x0, rel=100 * rel, abs=1e-9)
        assert y == pytest.approx(y0, rel=100 * rel, abs=1e-9)
