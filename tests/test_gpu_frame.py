"""Reading a state back in pieces by several host threads (pg_get_state):
frames below and above one thread's share, of one piece and of several, with
a ragged last piece, and of one row a piece, give back the values that
were set, and a read after steps equals a second read of the same state."""
import numpy as np
import pytest

from penguin_amd import Disk, disk2d, disk3d

pytestmark = pytest.mark.gpu


# cells: 4 k and 131 k (one thread), 2.1 M (pieces of 3 MB, the last ragged)
@pytest.mark.parametrize("nr, nphi", [(40, 101), (257, 510), (701, 3001)])
@pytest.mark.parametrize("dust", [0, 1])
def test_frame_2d(nr, nphi, dust):
    d = Disk(disk2d(nr, nphi, precision=8, dust_flag=dust))
    rng = np.random.default_rng(4)
    g, dd = d.get_state()
    g[[0, 2, 3]] *= 1.0 + 1e-3 * rng.standard_normal((3, nphi, nr))
    cs2 = g[1] / d.get_state()[0][0]
    g[1] = cs2 * g[0]
    if dust:
        dd[:3] *= 1.0 + 1e-3 * rng.standard_normal((3, nphi, nr))
    d.set_state(g, dd)
    a, b = d.get_state()
    # the device holds deviations from a background of order one: one rounding each way
    assert np.abs(a - g).max() <= 4 * np.finfo(float).eps * np.abs(g).max()
    if dust:
        assert np.abs(b - dd).max() <= 4 * np.finfo(float).eps * np.abs(dd).max()
    d.run(2)
    for x, y in zip(d.get_state(), d.get_state()):
        assert x is y or np.array_equal(x, y)
    d.close()


# the second: rows of 6 MB, one a piece
@pytest.mark.parametrize("nr, nphi, nth", [(97, 131, 67), (300000, 4, 4)])
def test_frame_3d(nr, nphi, nth):
    d = Disk(disk3d(nr, nphi, nth, precision=4))
    g = np.random.default_rng(5).uniform(0.5, 1.5, (5, nth, nphi, nr)).astype(np.float32).astype(np.float64)
    v = d.get_state()[0][3]           # the azimuthal velocity is held as a deviation: set the background's own
    g[3] = v
    d.set_state(g)
    assert np.array_equal(d.get_state()[0], g)
    d.close()
