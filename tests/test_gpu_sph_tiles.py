"""The radial sweep's tiles (several rows of a segment of radii per block):
grids whose rows cross polar layers within a block, whose last block holds
fewer rows, whose row is cut into unequal segments, and the smallest grid,
against the oracle in FP64 at the module test's tolerances."""
import numpy as np
import pytest

import oracle
from penguin_amd import Disk, disk3d

pytestmark = pytest.mark.gpu


# rows per block: 5 (of 102 slots; 5187 rows, so the last block holds 2, and
# rows of 57 cross layers within a block), 7 (of segments of 67, 67 and 66
# radii), 1, 1, 1
@pytest.mark.parametrize("nx, ny, nz", [(96, 57, 91), (200, 73, 37), (41, 37, 9), (259, 6, 5), (4, 4, 4)])
def test_radial_sweep_tiles(nx, ny, nz):
    p = disk3d(nx, ny, nz, precision=8, noise_rho=1e-2, noise_vr=1e-2, ramp_time=0.0)
    o, d = oracle.Oracle(p), Disk(p)
    g, _ = o.get_state()
    K, J, I = np.meshgrid(*(np.arange(n) for n in g.shape[1:]), indexing="ij")
    g[0] *= 1 + 0.1 * np.cos(2 * np.pi * J / ny - 6.0 * I / nx + 2.0 * K / nz)
    g[2] += 0.05 * np.sqrt(g[1] / g[0]) * np.sin(2 * np.pi * J / ny + 2.0 * I / nx - K / nz)
    o.set_state(g)
    d.set_state(g)
    dt = 0.5 * o.global_dt(1.0)
    d.sweep_x(dt)
    o.sweepx(dt)
    a, b = d.get_state()[0], o.get_state()[0]
    for k in range(5):
        assert np.abs(a[k] - b[k]).sum() <= 1e-10 * np.abs(b[k]).sum(), k
        assert np.abs(a[k] - b[k]).max() <= 1e-6 * np.abs(b[k]).max(), k
    d.close()
