"""The limited parabola (slopes) on the host, from the headers the kernels are
built from: against the limiter written with its conditions, as the scheme
states it, on finite means, and on means that are not numbers.

A parabola over a cell mean that is not a number is not a number either, so that
a broken state spreads through the stencil as it does in the scheme, instead of
being limited to a finite slope beside the broken cell.
"""
import ctypes

import numpy as np
import pytest

from penguin_amd.build import ADJCHECK

W = np.array([-1 / 12, 7 / 12, 0.0, 0.0, 7 / 12, -1 / 12])


@pytest.fixture(scope="module", params=[np.float64, np.float32])
def slopes(request):
    L = ctypes.CDLL(ADJCHECK)
    dp, fp = ctypes.POINTER(ctypes.c_double), ctypes.POINTER(ctypes.c_float)

    def f(a, w, flat):
        x = np.ascontiguousarray(np.concatenate([a, w, [flat]]), dtype=request.param)
        y = np.zeros(2, request.param)
        if request.param is np.float32:
            L.adjc_slopes_f32(x.ctypes.data_as(fp), y.ctypes.data_as(fp))
        else:
            ly, lx = np.zeros(2), np.zeros(12)
            assert L.adjc_eval(2, *(v.ctypes.data_as(dp) for v in (x, ly, y, lx))) == 0
        return y
    f.dtype = request.param
    return f


def _limiter(a, w, flat):
    """4th-order slopes, limited to the neighbours' differences, flattened,
    then the monotonicity correction of the parabola."""
    d = np.diff(a)
    l = w[0] * d[0] + w[1] * d[1] + w[2] * d[2]
    r = w[3] * d[1] + w[4] * d[2] + w[5] * d[3]
    l = np.copysign(np.fmin(abs(l), abs(d[1])), d[1])
    r = np.copysign(np.fmin(abs(r), abs(d[2])), d[2])
    if r * l <= 0:
        l = r = 0.0
    l, r = l * (1 - flat), r * (1 - flat)
    t2, t1 = (l + r) ** 2, 3 * (l + r) * (l - r)
    if t2 < t1:
        l = 2 * r
    elif t2 < -t1:
        r = 2 * l
    return np.array([l, r])


def test_finite_means(slopes):
    rng = np.random.default_rng(7)
    kinds = np.zeros(4, int)
    for n in range(4000):
        a = np.cumsum(rng.normal(0, 1, 5) * 10.0 ** rng.uniform(-3, 0, 5)) + rng.choice([0.0, 1.0])
        a = a.astype(slopes.dtype).astype(float)
        if n % 7 == 0:
            a[rng.integers(1, 5)] = a[0]          # equal neighbours
        flat = rng.choice([0.0, rng.uniform(0, 0.5)])
        want, got = _limiter(a, W, flat), slopes(a, W, flat)
        kinds[0 if not want.any() else 1 if want[0] == 2 * want[1] else 2 if want[1] == 2 * want[0] else 3] += 1
        # differences of means of order one, three products and their sum
        assert np.abs(got - want).max() <= 8 * np.finfo(slopes.dtype).eps * max(1.0, np.abs(a).max()), (n, a, flat)
    assert kinds.min() > 100, kinds


@pytest.mark.parametrize("cell", range(5))
@pytest.mark.parametrize("a", [[1.0, 1.1, 1.3, 1.4, 1.45], [1.0, 0.7, 0.6, 0.2, 0.1], [1.0, 1.2, 0.9, 1.3, 1.1]])
def test_a_mean_that_is_not_a_number(slopes, a, cell):
    a = np.array(a)
    a[cell] = np.nan
    with np.errstate(invalid="ignore"):
        want = _limiter(a, W, 0.0)
    got = slopes(a, W, 0.0)
    # the cell itself or one beside it: no parabola; one cell further: the
    # neighbours' differences still bound it
    assert np.isnan(want).any() == (1 <= cell <= 3)
    assert np.isnan(got).any() == (1 <= cell <= 3), (want, got)
    assert np.isnan(got[np.isnan(want)]).all(), (want, got)


def test_flattening_that_is_not_a_number(slopes):
    assert np.isnan(slopes(np.array([1.0, 1.1, 1.3, 1.4, 1.45]), W, np.nan)).all()
