"""Azimuthal, advection and viscosity adjoints at the edges of their tiles (46,
44 and 7 rows in FP64; 8 and 64 radii): one row less than whole tiles, whole
tiles, one more, and rings shorter than a tile.

These passes do not know where on the ring they are: turning the state and the
output weights by some rows must turn the adjoint by as many, wherever the tiles
then cut the ring.  (That the adjoint is right is held to finite differences in
test_gpu_adjoint_passes.py.)  Each cell's arithmetic is the same at every place
of a tile up to the contraction of products, so the two may differ by rounding:
some 100 terms no larger than the largest adjoint, carried through differences
of neighbours that cancel at most three digits, 100 x 1e3 x 1.1e-16.
"""
import numpy as np
import pytest

from penguin_amd import Disk, config_c5

pytestmark = pytest.mark.gpu

SIZES = [(65, 45), (64, 46), (72, 47), (71, 43), (70, 44), (127, 92), (129, 93), (24, 13), (63, 88)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", ["sweep_y", "orbital_advection", "viscosity"])
def test_adjoint_turns_with_the_ring(name, size):
    d = Disk(config_c5(precision=8, xres=size[0], yres=size[1]).replace(noise_rho=0.0))
    g, _ = d.get_state()
    rng = np.random.default_rng(11)
    cs = np.sqrt(g[1] / g[0])
    wobble = rng.uniform(-1, 1, (3, *g[0].shape))
    g[0] *= 1.0 + 0.02 * wobble[0]
    g[1] *= 1.0 + 0.02 * wobble[0]
    g[2] += 0.02 * cs * wobble[1]
    g[3] += 0.02 * cs * wobble[2]
    d.set_state(g)
    dt = 0.4 * d.global_dt(1.0)
    lam = rng.uniform(-1, 1, (2 if name == "viscosity" else 3, d.ny, d.nx))
    want, _ = d.adjoint_pass(name, 0.0, dt, lam)
    want = np.array(want)
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    for turn in (1, 7, d.ny // 2):
        d.set_state(np.roll(g, turn, axis=1))
        got, _ = d.adjoint_pass(name, 0.0, dt, np.roll(lam, turn, axis=1))
        diff = np.abs(np.roll(np.asarray(got), -turn, axis=1) - want)
        for k in range(3):
            assert diff[k].max() <= 1.1e-11 * np.abs(want[k]).max(), (turn, k)
    d.close()
