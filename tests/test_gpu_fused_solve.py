"""The small-system solve: groups of sweeps per launch (``k_sweeps``), whose
iterates and sums are those of the one-pass-per-launch kernels bit for bit.
Per-kernel timing (``Model.profile``) runs the latter."""
import numpy as np
import pytest

from dcm_amd import hip as H
from dcm_amd import workloads as W
from helpers import field, interior, small_domain

pytestmark = pytest.mark.gpu


def _solves(dom, mixed, cheb, iters):
    """The solve of one right-hand side in both forms: statuses, iteration
    counts, residuals and the pressure."""
    b = np.zeros(dom.shape)
    interior(b)[...] = interior(field(dom, 5))
    interior(b)[...] -= interior(b).mean()
    zero = np.zeros(dom.shape)
    case = W.Case("c", dom, 0.5, 1, u=zero, v=zero, w=zero, th=zero)
    out = []
    with H.Context(dom) as c:
        m = H.Model(c, case)
        if cheb is not None:
            c.set_precond_chebyshev(*cheb)
        for profiled in (False, True):
            m.profile(profiled)
            x, sw, db = c.array(field(dom, 6)), c.zeros(), c.array(b)
            if mixed:
                st = c.bicgstab_mixed(sw, x, db, 1e-10)
            else:
                st = c.bicgstab(sw, x, db, 1e-10, itmax=iters, check=False)
            out.append((st, x.get()))
        m.profile(False)
        m.close()
    return out


# one column or a closed axis (at most 8 x 4 or 8 x 8 columns), ragged last
# tiles, boxes that wrap onto themselves, one and several k tiles of 64 and of
# 32 lanes, two positions a thread; the last two exceed the FP64 box and run
# fused in FP32 only
SHAPES = [(1, 101, 120), (1, 40, 95), (2, 3, 40), (8, 4, 64), (9, 5, 33), (9, 9, 32),
          (12, 11, 48), (24, 17, 64), (40, 33, 20), (19, 21, 70), (10, 18, 96)]


@pytest.mark.parametrize("iters", [1, 4, 9])
@pytest.mark.parametrize("shape", SHAPES)
def test_fused_fp64_sweeps_match_the_passes(shape, iters):
    # (stretched in y and z, uniform in x as the fused kernels require; such
    # an operator has no symmetric null space: a few iterations, converged or
    # not)
    dom = small_domain(*shape, stretched=True)
    dom.dx, dom.dxn = np.full_like(dom.dx, 50.0), np.full_like(dom.dxn, 50.0)
    a, b = _solves(dom, False, None, iters)
    assert a[0] == b[0] and a[0][1] == iters
    np.testing.assert_array_equal(a[1], b[1])


@pytest.mark.parametrize("cheb", [None, (0.0, 4), (0.01, 5), (0.002, 8)])
@pytest.mark.parametrize("shape", SHAPES)
def test_fused_fp32_sweeps_match_the_passes(shape, cheb):
    a, b = _solves(small_domain(*shape), True, cheb, 0)
    assert a[0] == b[0] and a[0][0] > 4
    np.testing.assert_array_equal(a[1], b[1])
