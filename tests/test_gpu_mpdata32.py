"""The limiter and last donor pass of the mixed path's FP32 MPDATA at the edges
of its tiles: a last tile of one row, one or two i planes, chunks of 16 planes
with one left over, columns that fill or just pass a wavefront, 256 levels."""
import numpy as np
import pytest

from dcm_amd import hip as H
from dcm_amd import workloads as W
from helpers import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 9, 40), (2, 1, 33), (17, 8, 32), (16, 17, 64), (5, 5, 256),
                                   (33, 4, 65), (18, 3, 200)])
def test_limited_pass_tracks_the_fp64_path(shape):
    """Five steps of two advected fields of different categories; each step
    rounds a field to FP32 some ten times (6e-8 each), and the limiter's
    factors are quotients of sums of such roundings: 1e-6 of the field."""
    case = W.moist_bubble(*shape, delta=50.0, dt=0.5, steps=5, ntracer=1, seed=17)
    out = {}
    for prec in (H.FP64, H.MIXED):
        with H.Context(case.dom) as c:
            m = H.Model(c, case, prec)
            try:
                m.step(5)
                out[prec] = {"th": m.get(H.F_TH), "q0": m.get(H.F_Q, 0), "q1": m.get(H.F_Q, 1)}
            finally:
                m.close()
    for f in out[H.FP64]:
        assert np.isfinite(out[H.MIXED][f]).all(), f
        assert rel_l2(out[H.FP64][f], out[H.MIXED][f]) < 1e-6, f
