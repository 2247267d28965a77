"""States that are not finite, through the sweeps and the step.

A cell that is not a number makes its neighbours along a sweep so on both sides
(their parabolas take its mean), and no state with a value that is not finite is
advanced for long: an infinite or undefined velocity is refused by the step that
reads it, a density by the step after it, by the CFL rate.
"""
import numpy as np
import pytest

from penguin_amd import Disk, disk2d
from penguin_amd.disk import PenguinError

pytestmark = pytest.mark.gpu

J, I = 30, 20


def _broken(prec, fluid, field, value):
    p = disk2d(40, 64, precision=prec, dust_flag=1)
    d = Disk(p)
    s = d.get_state()
    s[fluid][field, J, I] = value
    d.set_state(*s)
    return d


@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("field", [0, 2, 3])
@pytest.mark.parametrize("sweep", ["sweep_x", "sweep_y", "orbital_advection"])
def test_spreads_to_both_neighbours(prec, field, sweep):
    d = _broken(prec, 0, field, np.nan)
    getattr(d, sweep)(1e-4)
    bad = np.isnan(d.get_state()[0]).any(axis=0)
    dj, di = (0, 1) if sweep == "sweep_x" else (1, 0)
    for k in (-1, 0, 1):
        assert bad[J + k * dj, I + k * di], k
    # and no further than the stencil: two cells and the flux between
    j, i = np.nonzero(bad)
    assert np.abs(j - J).max() <= 3 * dj and np.abs(i - I).max() <= 3 * di
    d.close()


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("prec", [4, 8])
@pytest.mark.parametrize("fluid, field", [(0, 0), (0, 2), (0, 3), (1, 0), (1, 1), (1, 2)])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_is_refused(prec, fluid, field, value, graph):
    d = _broken(prec, fluid, field, value)
    velocity = field > 0
    if velocity:
        with pytest.raises(PenguinError, match="rate is inf"):
            d.global_dt(1.0)
    with pytest.raises(PenguinError, match="before step %d is inf" % (0 if velocity else 1)):
        d.run(6, use_graph=graph)
    d.close()
