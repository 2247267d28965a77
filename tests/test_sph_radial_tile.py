"""The rule for the 3D radial sweep's tile (pg_sph.h) over all the rows it can
meet: every radius in one segment, a thread per slot, LDS within what a launch
takes without asking, and the slot's row by multiplication exact."""
import ctypes

import pytest

from penguin_amd.build import ADJCHECK

PAD, FIELDS = 3, 15


def radial_tile(nx, rows, es):
    out = (ctypes.c_int * 3)()
    ctypes.CDLL(ADJCHECK).hostcheck_radial_tile(nx, ctypes.c_long(rows), es, out)
    return tuple(out)


@pytest.mark.parametrize("es, threads", [(4, 512), (8, 256)])
def test_radial_tile(es, threads):
    tiles = set()
    for nx in list(range(4, 1100)) + [2000, 4097, 30001, 300000]:
        for rows in (16, 640, 2047, 2048, 9999, 98304):
            tx, xr, xm = radial_tile(nx, rows, es)
            slots = tx + 2 * PAD
            nseg = -(-nx // tx)
            assert tx >= 1 and xr >= 1 and xr * slots <= threads, (nx, rows)
            assert (nseg - 1) * tx < nx <= nseg * tx and nseg <= nx, (nx, rows)
            assert FIELDS * xr * slots * es <= 65536, (nx, rows)
            # a thread for every slot, and at least one block a CU where there are rows enough
            assert xr == 1 or nseg * -(-rows // xr) >= 2048, (nx, rows)
            tiles.add((slots, xm))
    for slots, xm in tiles:
        for t in range(512):
            assert (t * xm) >> 20 == t // slots, (t, slots)


@pytest.mark.parametrize("nx, rows, es, want", [(384, 1536 * 64, 4, (96, 5)), (96, 384 * 64, 4, (96, 5)),
                                                (40, 64 * 16, 8, (40, 1)), (101, 190 * 33, 4, (101, 3))])
def test_the_tiles_that_were_measured(nx, rows, es, want):
    assert radial_tile(nx, rows, es)[:2] == want
