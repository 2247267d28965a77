"""Reading a 2D state back in FP32: frames of one (pageable) piece, of several
pinned ones by one thread and of several by several.  Every read gives the values
that were set, rounded once as a deviation from the background, and the same bits
as the first."""
import numpy as np
import pytest

from penguin_amd import Batch, Disk, disk2d

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float32).eps


# 0.15 (one piece), 3, 9 and 25 MB a fluid
@pytest.mark.parametrize("nr, nphi", [(41, 301), (257, 1023), (600, 1300), (701, 3001)])
@pytest.mark.parametrize("dust", [0, 1])
def test_frame_2d_fp32(nr, nphi, dust):
    d = Disk(disk2d(nr, nphi, precision=4, dust_flag=dust))
    rng = np.random.default_rng(6)
    g0, q0 = d.get_state()
    g, q = g0.copy(), None if q0 is None else q0.copy()
    dev = 1e-3 * rng.standard_normal((3, nphi, nr))
    g[[0, 2, 3]] += dev
    g[1] = g0[1] / g0[0] * g[0]
    if dust:
        q[:3] *= 1.0 + dev
    d.set_state(g, q)
    a, b = d.get_state()
    # the background itself (of order one) is FP64; density, u and v are stored
    # as deviations or as small values, the dust's density and u as they are
    for k, f in enumerate((0, 2, 3)):
        held = g[f] if f == 2 else dev[k] + (g0[f] - _background(g0, f))
        assert np.abs(a[f] - g[f]).max() <= EPS * np.abs(held).max() + 4 * np.finfo(float).eps * np.abs(g[f]).max(), f
    assert np.abs(a[1] - g[1]).max() <= EPS * np.abs(g[1]).max()
    assert not a[4].any()
    if dust:
        for f in (0, 1, 2):
            assert np.abs(b[f] - q[f]).max() <= EPS * np.abs(q[f]).max(), f
        assert not b[3].any()
    for _ in range(4):
        a2, b2 = d.get_state()
        assert np.array_equal(a2, a) and (b is None or np.array_equal(b2, b))
    d.close()


def _background(g, f):
    return g[f].mean(axis=0, keepdims=True)


def test_disks_of_a_batch_share_the_pieces():
    sizes = [(41, 301), (701, 1301), (64, 128), (512, 1024)]
    ps = [disk2d(nr, nphi, precision=4, seed=k, noise_rho=1e-3) for k, (nr, nphi) in enumerate(sizes)]
    want = []
    for p in ps:
        with Disk(p) as d:
            want.append(d.get_state()[0])
    with Batch(ps) as b:
        for _ in range(3):
            for k in (2, 0, 3, 1, 0):
                assert np.array_equal(b.get_state(k)[0], want[k]), k
