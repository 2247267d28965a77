"""Radial tiles of several rows (the 3D radial sweep): alone, against the oracle,
and as it begins a step with the first half kick in it, against the step taken
module by module, whose kick is a pass of its own over the cells in memory order.
Rows of one segment and of several, equal and unequal, blocks that cross polar
layers and a last block that is not full; each case names the tile that it is
there for (cells of a segment, rows of a block).

(test_gpu_sph_tiles.py's grids, at FP64's 256 threads, take one or two rows of
one segment, or one row of several.)

Against the oracle FP64 is held to the module tests' tolerances; the step's two
forms differ by contraction and by the round trip of the azimuthal velocity
through the background's, some 100 roundings of 1.1e-16 on values that cancel to
a hundredth.  FP32: a value of order one carries some 40 roundings of 6e-8; the
radial and polar velocities are a thirtieth of the sound speed, so theirs weigh
thirty times as much.  A row or layer taken for another would differ by the
state's own structure, a tenth of each field.
"""
import numpy as np
import pytest

import oracle
from penguin_amd import Disk, disk3d
from tests.test_sph_radial_tile import radial_tile

pytestmark = pytest.mark.gpu

CASES = [
    # precision, grid, tile
    (8, (37, 128, 97), (37, 5)),     # 128 rows a layer: blocks cross layers; the last holds 1 row
    (8, (130, 91, 48), (44, 5)),     # segments of 44, 44 and 42; the last block holds 3 rows
    (8, (300, 97, 40), (75, 3)),     # four segments; the last block holds 1 row
    (4, (37, 128, 97), (37, 6)),     # the last block holds 2 rows
    (4, (259, 90, 40), (65, 7)),     # segments of 65, 65, 65 and 64; the last block holds 2 rows
    (4, (96, 109, 97), (96, 5)),     # the 384- and 96-radius disks' tile; the last block holds 3 rows
]
NAMES = ("rho", "p", "u", "v", "w")


def _pair(prec, grid):
    kw = dict(noise_rho=1e-2, noise_vr=1e-2, ramp_time=0.0)
    o = oracle.Oracle(disk3d(*grid, precision=8, **kw))
    g, _ = o.get_state()
    K, J, I = np.meshgrid(*(np.arange(n) for n in g.shape[1:]), indexing="ij")
    phi, lr, th = 2 * np.pi * (J + 0.5) / g.shape[2], I / g.shape[3] * np.log(2.5 / 0.4), (K + 0.5) / g.shape[1]
    cs = np.sqrt(g[1] / g[0])
    # neighbouring rows and layers differ too
    wave = 1 + 0.1 * np.cos(2 * phi - 6 * lr + 2 * th) + 0.02 * np.cos(np.pi * (J + 2 * K) / 3)
    g[0] *= wave
    g[1] *= wave * (1 + 0.05 * np.sin(phi + 3 * th))
    g[2] += 0.05 * cs * np.sin(phi + 2 * lr - th)
    g[3] += 0.05 * cs * np.cos(3 * phi - lr + th)
    g[4] += 0.05 * cs * np.sin(2 * phi + lr) * np.sin(np.pi * th)
    g = g.astype(np.float32).astype(np.float64)      # both sides start from the same numbers
    o.set_state(g)
    d = Disk(disk3d(*grid, precision=prec, **kw))
    d.set_state(g)
    return d, o


def _compare(a, b, prec, fp64, what):
    for k, name in enumerate(NAMES):
        err = np.abs(a[k] - b[k]).sum() / np.abs(b[k]).sum()
        mx = np.abs(a[k] - b[k]).max() / np.abs(b[k]).max()
        print(f"{what} {name}: rel L1 {err:.2e} max {mx:.2e}", flush=True)
        l1, pt = fp64 if prec == 8 else (1e-4 if name in "uw" else 1e-5, 1e-2)
        assert err <= l1 and mx <= pt, (what, name, err, mx)


@pytest.mark.parametrize("prec, grid, tile", CASES)
def test_tile_is_the_one_named(prec, grid, tile):
    assert radial_tile(grid[0], grid[1] * grid[2], prec)[:2] == tile


@pytest.mark.parametrize("prec, grid, tile", CASES)
def test_radial_sweep(prec, grid, tile):
    d, o = _pair(prec, grid)
    dt = 0.5 * o.global_dt(1.0)
    d.sweep_x(dt)
    o.sweepx(dt)
    _compare(d.get_state()[0], o.get_state()[0], prec, (1e-10, 1e-6), "sweep")
    d.close()


@pytest.mark.parametrize("prec, grid, tile", CASES)
def test_step_is_its_modules(prec, grid, tile):
    d, o = _pair(prec, grid)
    g = d.get_state()[0]
    dt = 0.5 * d.global_dt(1.0)
    d.solve(0.0, dt)
    fused = d.get_state()[0]
    d.close()
    d = Disk(d.p)
    d.set_state(g)
    d.viscosity()
    d.sources(0.0, 0.0, 0.5 * dt)
    for module in (d.sweep_x, d.sweep_y, d.sweep_z, d.orbital_advection):
        module(dt)
    swept = d.get_state()[0]
    # the predicted state, by the forces at the step's start, for its own viscous forces
    d.sources(dt, 0.5 * dt, 0.5 * dt, inplace=False)
    d.viscosity()
    d.set_state(swept)
    d.sources(dt, 0.5 * dt, 0.5 * dt)
    _compare(fused, d.get_state()[0], prec, (1e-12, 1e-9), "step")
    assert np.abs(fused - g).max() > 1e-4
    d.close()
