"""The FP64 MPDATA passes as marching kernels (dcm_mpdata64.hip), taken on
grids uniform along x, bit for bit against the oracle: edges of the launch
tiles, short marches, kord 1 to 3, and numerators outside the range in which
a quotient comes from a reciprocal."""
import numpy as np
import pytest

import oracle as O
from dcm_amd import hip as H
from helpers import field, small_domain

pytestmark = pytest.mark.gpu


def _dom(shape, moderate=True):
    """Stretched in y and z, varying density, uniform along x."""
    dom = small_domain(*shape, stretched=True, varying_theta=True)
    dom.dx, dom.dxn = np.full_like(dom.dx, 47.0), np.full_like(dom.dxn, 47.0)
    if not moderate:  # outside the fast kernels' range: the per-cell kernels
        dom.dy = dom.dy.copy()
        dom.dy[0] = 1e13
    return dom


def _compare(dom, psi, scale=1.0, kord=2, monotone=True, neumann=0, nq=None, lbc=0.0, ubc=0.0):
    g = O.Grid(dom)
    vel = [scale * 0.25 * 45.0 * field(dom, s) for s in (3, 4, 5)]
    for a in vel:
        O.fill_full(g, a, 0.0, 0.0)
    with H.Context(dom) as c:
        d = [c.array(a) for a in vel]
        dpsi = c.array(psi)
        if nq is None:
            ex, lb, ub = c.mpdata3d(1.0, *d, dpsi, lbc, ubc, kord, monotone, neumann)
            r, olb, oub = O.mpdata3d(g, 1.0, *vel, psi, lbc, ubc, kord, monotone, neumann)
            assert (lb, ub) == (olb, oub)
        else:
            ex, _, _ = c.mpdata_vec3d(1.0, *d, dpsi, nq, None, None, kord, monotone, neumann)
            r, _, _ = O.mpdata_vec3d(g, 1.0, *vel, psi, None, None, kord, monotone, neumann)
        assert ex == r
        np.testing.assert_array_equal(dpsi.get(), psi)


SHAPES = [(1, 1, 2), (1, 9, 40), (3, 2, 16), (2, 5, 33), (5, 4, 64), (17, 9, 31), (33, 6, 65),
          (4, 17, 130)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kord,monotone,neumann", [(1, True, 0), (2, True, 0), (2, False, 1),
                                                   (3, True, 2), (3, False, 0)])
def test_marching_passes_bitwise(shape, kord, monotone, neumann):
    dom = _dom(shape)
    psi = field(dom, 7, -1.0, 3.0)
    O.fill_full(O.Grid(dom), psi, 0.25, 0.5)
    _compare(dom, psi, kord=kord, monotone=monotone, neumann=neumann, lbc=0.25, ubc=0.5)


@pytest.mark.parametrize("shape", [(5, 7, 20), (18, 5, 66)])
@pytest.mark.parametrize("kord", [2, 3])
def test_marching_category_bitwise(shape, kord):
    dom = _dom(shape)
    g = O.Grid(dom)
    q = np.stack([field(dom, 20 + n, 0.0, 1.0 + n) for n in range(3)])
    q[1][:, :, :5] = 0.0
    for n in range(3):
        O.fill_full(g, q[n], 0.0, 0.0)
    _compare(dom, q, kord=kord, nq=3)


# fields and winds so small that residuals of the reciprocal quotients would
# underflow, zero regions, and spacings beyond the fast range
@pytest.mark.parametrize("amp,scale", [(1e-285, 1.0), (1e-300, 1.0), (1.0, 1e-280), (1e-310, 1.0),
                                       (1e280, 1.0)])
def test_marching_passes_at_the_ends_of_the_range(amp, scale):
    dom = _dom((9, 8, 34))
    psi = amp * field(dom, 9, 0.0, 1.0)
    psi[3:6] = 0.0
    O.fill_full(O.Grid(dom), psi, 0.0, 0.0)
    _compare(dom, psi, scale=scale)


def test_spacings_outside_the_range_take_the_per_cell_kernels():
    dom = _dom((7, 6, 18), moderate=False)
    psi = field(dom, 11, 0.0, 1.0)
    O.fill_full(O.Grid(dom), psi, 0.0, 0.0)
    _compare(dom, psi)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_non_finite_cells_as_the_per_cell_kernels(bad):
    """One bad cell: the same cells as the oracle's are not finite, the others
    the same bits."""
    dom = _dom((9, 8, 34))
    g = O.Grid(dom)
    vel = [0.25 * 45.0 * field(dom, s) for s in (3, 4, 5)]
    for a in vel:
        O.fill_full(g, a, 0.0, 0.0)
    vel[0][5, 4, 17] = bad
    psi = field(dom, 12, 0.0, 1.0)
    O.fill_full(g, psi, 0.0, 0.0)
    with H.Context(dom) as c:
        d = [c.array(a) for a in vel]
        dpsi = c.array(psi)
        c.mpdata3d(1.0, *d, dpsi)
        O.mpdata3d(g, 1.0, *vel, psi)
        np.testing.assert_array_equal(dpsi.get(), psi)
