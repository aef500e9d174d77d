"""The transform preconditioner of the mixed path's FP32 inner solve
(dcm_spectral.hip), taken with dcm_set_precond_multigrid on grids uniform
along every axis whose line lengths have the factors 2, 3, 5 and 7 and halve
together on every multigrid level, to two cells or more on the coarsest."""
import numpy as np
import pytest

from dcm_amd import hip as H
from helpers import rel_l2, small_domain

pytestmark = pytest.mark.gpu


def _solve(dom, mg, precision_tol=1e-10, seed=5):
    r = np.random.default_rng(seed)
    b = np.zeros(dom.shape)
    b[1:-1, 1:-1, 1:-1] = r.standard_normal((dom.ip, dom.jp, dom.kp))
    # orthogonal to the left null vector, dz of the level below
    wt = np.broadcast_to(dom.dz[:-2], (dom.ip, dom.jp, dom.kp))
    b[1:-1, 1:-1, 1:-1] -= (wt * b[1:-1, 1:-1, 1:-1]).sum() / wt.sum()
    with H.Context(dom) as c:
        if mg:
            c.set_precond_multigrid(mg)
        x = c.array(np.zeros(dom.shape))
        it, outer, err = c.bicgstab_mixed(c.array(np.zeros(dom.shape)), x, c.array(b),
                                          tol=precision_tol)
        return it, outer, err, x.get()[1:-1, 1:-1, 1:-1]


# every radix and their mixtures, short and long lines, tiles with a remainder
# of columns
@pytest.mark.parametrize("shape", [(16, 16, 16), (10, 14, 10), (12, 12, 12), (20, 28, 36),
                                   (48, 80, 32), (112, 32, 32), (32, 112, 48), (60, 28, 20),
                                   (288, 96, 64), (96, 64, 288), (320, 192, 128)])
def test_the_transforms_invert_the_operator(shape):
    """In exact arithmetic M is the operator's inverse: after the first half
    of an iteration the residual is rounding, so each refinement takes one
    iteration; the solution is the plain sweeps' to the tolerance of both."""
    dom = small_domain(*shape)
    it, outer, err, x = _solve(dom, 1)
    assert err < 1e-10 and it == outer, (it, outer, err)
    _, _, err0, x0 = _solve(dom, 0)
    assert err0 < 1e-10
    assert rel_l2(x0 - x0.mean(), x - x.mean()) < 1e-7


@pytest.mark.parametrize("shape", [(1024, 128, 128), (128, 768, 128), (128, 128, 1024)])
def test_long_lines(shape):
    """Lines of up to 1024 values: each refinement takes one iteration, or two
    where FP32 rounding times the condition number, (2 n / pi)^2 / 2 times 6e-8
    along a line of n = 768 or more, nears the inner tolerance.  Both solutions
    leave a residual of 1e-10 of b, which may all lie in the smoothest mode,
    1/sqrt(cells) of b and most of the solution: 2e-10 sqrt(cells) apart."""
    dom = small_domain(*shape, delta=10.0)
    it, outer, err, x = _solve(dom, 1)
    assert err < 1e-10 and outer <= it <= 2 * outer, (it, outer, err)
    _, _, err0, x0 = _solve(dom, 0)
    assert err0 < 1e-10
    assert rel_l2(x0 - x0.mean(), x - x.mean()) < 2e-10 * np.sqrt(x.size)


def _stretched(*shape):
    dom = small_domain(*shape)
    f = 1.0 + 0.2 * np.random.default_rng(3).random((2, dom.kp + 2))
    dom.dz, dom.dzn = dom.dz * f[0], dom.dzn * f[1]
    return dom


def test_grids_it_does_not_take_keep_the_v_cycle():
    """A stretched axis (the shapes whose V-cycle is all fused kernels, and one
    with per-pass levels), a line length with a factor above 7, and
    semi-coarsened hierarchies and one that ends at a single cell along x: several V-cycles per refinement, and the same
    bits from the fused kernels and from one launch per pass."""
    for dom in (_stretched(64, 64, 32), _stretched(256, 128, 64), small_domain(88, 48, 32),
                small_domain(128, 4, 64), small_domain(96, 4, 16),
                small_domain(32, 96, 96)):
        one, two = _solve(dom, 1), _solve(dom, 2)
        assert one[2] < 1e-10 and one[0] > one[1], (dom.ip, one[:3])
        assert one[:3] == two[:3]
        np.testing.assert_array_equal(one[3], two[3])
