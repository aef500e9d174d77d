"""Captured phases of a step hold the addresses of the context's scratch.
Scratch that has to grow after the capture moves, and the next steps must not
replay the graphs of its old place: the fields are those of a run without
graphs, bit for bit, and allocations made after the growth (which may take the
old place) keep their values."""
import numpy as np
import pytest

from dcm_amd import hip as H
from dcm_amd import workloads as W
from helpers import field

pytestmark = pytest.mark.gpu


class _Guards:
    """Small device arrays of known values, of about the scratch's sizes."""

    def __init__(self, ctx):
        self.a = [H.DeviceArray(ctx, (n,)).set(np.full(n, 7.25))
                  for n in (128, 160, 272, 376, 576, 704) for _ in range(6)]

    def check(self):
        for a in self.a:
            np.testing.assert_array_equal(a.get(), 7.25)
            a.free()


def _snapshot(case, m):
    out = [m.get(f) for f in (H.F_U, H.F_V, H.F_W, H.F_TH, H.F_P)]
    return out + [m.get(H.F_Q, n) for n in range(case.nq)]


def _compare(run):
    for a, b in zip(run(True), run(False)):
        np.testing.assert_array_equal(a, b)


def _single(case, precision, grow):
    """Steps to the capture of both time levels' graphs, the growth, steps."""
    def run(graphs):
        with H.Context(case.dom) as c:
            m = H.Model(c, case, precision)
            try:
                m.set_graphs(graphs)
                grow(c, m, 0)
                m.step(7)
                for phase in (1, 2):
                    grow(c, m, phase)
                    g = _Guards(c)
                    m.step(6)
                    g.check()
                return _snapshot(case, m)
            finally:
                m.close()
    _compare(run)


def test_multigrid_switched_off():
    """The solve by groups of sweeps needs more partial sums than the V-cycle's."""
    def grow(c, m, phase):
        c.set_precond_multigrid(phase == 0)
    _single(W.warm_bubble(1, 64, 64, steps=19), H.FP64, grow)


def test_sum_order_switched():
    def grow(c, m, phase):
        c.set_sum_order(H.SUM_TREE if phase == 1 else H.SUM_SEQUENTIAL)
    _single(W.warm_bubble(1, 101, 120, steps=19), H.FP64, grow)


@pytest.mark.parametrize("shape", [(32, 32, 32), (1, 101, 120)])
@pytest.mark.parametrize("vertical", [True, False])
def test_category_of_many_fields_on_the_models_context(shape, vertical):
    case = W.warm_bubble(*shape, steps=19)

    def grow(c, m, phase):
        if phase == 0:
            return
        nf = 8 if phase == 1 else 32
        dom = case.dom
        psi = c.array(np.stack([field(dom, 40 + n, 0.0, 1.0) for n in range(nf)]))
        w = c.array(0.1 * field(dom, 39))
        if vertical:
            c.mpdata_vec_vert3d(0.5, w, psi, nf)
        else:
            c.mpdata_vec3d(0.5, w, w, w, psi, nf)
        psi.free()
        w.free()
    _single(case, H.FP64, grow)


def test_second_mixed_model_on_the_context():
    """The batched FP32 MPDATA's fields and partial sums grow with the second
    model's number of fields."""
    dom = dict(delta=50.0, dt=0.5, steps=19)
    case, more = (W.moist_bubble(20, 12, 33, ntracer=n, seed=5, **dom) for n in (1, 6))

    def grow(c, m, phase):
        if phase == 1:
            b = H.Model(c, more, H.MIXED)
            b.step(2)
            b.close()
    _single(case, H.MIXED, grow)


def test_calls_on_an_ensemble_members_context():
    cases = [W.warm_bubble(1, 64, 64, steps=19, seed=3),
             W.warm_bubble(12, 10, 24, steps=19, seed=4)]
    dom = cases[0].dom

    def run(graphs):
        ctxs = [H.Context(k.dom) for k in cases]
        models = [H.Model(c, k, H.FP64) for c, k in zip(ctxs, cases)]
        try:
            for m in models:
                m.set_graphs(graphs)
            with H.Ensemble(models) as e:
                e.set_graphs(graphs)
                e.step(7)
                for nf in (8, 32):
                    psi = ctxs[0].array(np.stack([field(dom, 40 + n, 0.0, 1.0)
                                                  for n in range(nf)]))
                    w = ctxs[0].array(0.1 * field(dom, 39))
                    ctxs[0].mpdata_vec_vert3d(0.5, w, psi, nf)
                    g = _Guards(ctxs[0])
                    e.step(6)
                    g.check()
            return [f for k, m in zip(cases, models) for f in _snapshot(k, m)]
        finally:
            for m in models:
                m.close()
            for c in ctxs:
                c.close()
    _compare(run)
