"""The azimuthal pass's tiles (pg_batch_set_schedule's ring_b) at their edges:
rings shorter than a tile and its halo (read around more than once), one row
short of, equal to and past a tile's rows, radii that do not fill a tile's
strip; gas and dust, both precisions.  Every tile gives the same bits, and a
new disk's own choice of tile among them."""
import numpy as np
import pytest

from penguin_amd import Batch, Disk, config_c2

pytestmark = pytest.mark.gpu

SIZES = [(8, 8), (9, 19), (17, 20), (16, 21), (23, 51), (8, 52), (15, 53), (9, 127), (24, 128), (10, 129)]


@pytest.mark.parametrize("prec", [4, 8])
def test_ring_tiles_give_the_same_bits(prec):
    ps = [config_c2(precision=prec, xres=nr, yres=nphi, seed=k, noise_rho=1e-3, ramp_time=1e-9)
          for k, (nr, nphi) in enumerate(SIZES)]
    out = {}
    for ring in (256, 512, 1024):
        b = Batch(ps)
        tile, _, order, rows = b.schedule()
        b.set_schedule(tile, ring, order, rows)
        b.run(6)
        out[ring] = [b.get_state(k) for k in range(len(ps))]
        b.close()
    for k, p in enumerate(ps):
        d = Disk(p)
        d.run(6, use_graph=True)
        own = d.get_state()
        d.close()
        for ring, got in out.items():
            for f in (0, 1):
                assert np.array_equal(got[k][f], own[f]), (SIZES[k], ring, f)
