"""The frame reader (pg_frame.h) on the CPU, over a stand-in for the HIP calls
it makes whose copies land at the earliest or at the latest moment a stream may
choose: every cell arrives once whatever the shape, a second and third read
through the same buffers too, and a read that fails ends, reports and leaves
nothing behind."""
import ctypes

import numpy as np
import pytest

from penguin_amd.build import ADJCHECK

OUT_OF_MEMORY, INVALID_VALUE = 2, 1      # hipError_t


@pytest.fixture(scope="module")
def lib():
    return ctypes.CDLL(ADJCHECK)


def _read(lib, rows, nx, nf, reads=1, late=0, refuse=0, fail=-1):
    src = np.random.default_rng(rows + nx).standard_normal((nf, rows, nx)).astype(np.float32)
    dst = np.zeros((nf, rows, nx))
    stats = (ctypes.c_long * 8)()
    err = lib.hostcheck_frame(ctypes.c_long(rows), ctypes.c_long(nx), nf, reads, late, refuse, fail,
                              src.ctypes.data_as(ctypes.c_void_p), dst.ctypes.data_as(ctypes.c_void_p), stats)
    return err, src, dst, dict(zip(("copies", "allocs", "most", "pinned", "events", "threads", "given", "block"),
                                     stats))


# one piece by one thread, several pieces by one, several pieces by several
# threads with a ragged last piece, rows longer than a piece
SHAPES = [(7, 5, 3), (300, 260, 3), (301, 4001, 3), (3001, 701, 5), (3, 700001, 5)]


@pytest.mark.parametrize("rows, nx, nf", SHAPES)
@pytest.mark.parametrize("late", [0, 1])
def test_every_cell_once(lib, rows, nx, nf, late):
    err, src, dst, st = _read(lib, rows, nx, nf, reads=3, late=late)
    assert err == 0
    assert np.array_equal(dst, 3 * src.astype(np.float64))
    assert st["pinned"] == 0 and st["events"] == 0, st


@pytest.mark.parametrize("rows, nx, nf", SHAPES)
@pytest.mark.parametrize("late", [0, 1])
@pytest.mark.parametrize("refuse", [1, 2])        # none at all; none after the first
def test_without_pinned_memory(lib, rows, nx, nf, late, refuse):
    err, src, dst, st = _read(lib, rows, nx, nf, reads=2, late=late, refuse=refuse)
    assert err == 0 and st["allocs"] < refuse and st["pinned"] == 0
    assert np.array_equal(dst, 2 * src.astype(np.float64))


@pytest.mark.parametrize("rows, nx, nf", SHAPES)
@pytest.mark.parametrize("late", [0, 1])
def test_a_copy_that_fails(lib, rows, nx, nf, late):
    copies = _read(lib, rows, nx, nf)[3]["copies"]
    for fail in sorted({0, copies // 2, copies - 1}):
        err, _, _, st = _read(lib, rows, nx, nf, reads=2, late=late, fail=fail)
        assert err == INVALID_VALUE, fail
        assert st["pinned"] == 0 and st["events"] == 0, st


@pytest.mark.parametrize("rows, nx, nf", [(7, 5, 3), (128, 64, 3), (330, 260, 3)])
def test_a_small_frame_is_one_copy_without_pinned_memory(lib, rows, nx, nf):
    err, src, dst, st = _read(lib, rows, nx, nf, reads=2)
    assert err == 0 and np.array_equal(dst, 2 * src.astype(np.float64))
    assert st["copies"] == 1 and st["allocs"] == 0 and st["threads"] == 1, st


# 1.2 MB in two pieces; 2.4, 7 and 14 MB in three buffers; 42 MB
@pytest.mark.parametrize("rows, nx, nf, pieces", [(500, 201, 3, 2), (500, 401, 3, 3), (301, 2001, 3, 3), (301, 4001, 3, 3),
                                                  (3001, 701, 5, 3)])
def test_a_piece_is_an_allocation_of_its_own(lib, rows, nx, nf, pieces):
    err, src, dst, st = _read(lib, rows, nx, nf, reads=3, late=1)
    assert err == 0 and np.array_equal(dst, 3 * src.astype(np.float64))
    frame = 4 * rows * nx * nf
    assert st["allocs"] == pieces and st["block"] <= max(1 << 20, frame // 16), st


# rows of 14, 0.6 and 0.014 MB: a piece holds 1, 4 and 187 of them
@pytest.mark.parametrize("rows, nx, nf, per", [(6, 700001, 5, 1), (74, 30001, 5, 4), (3001, 701, 5, 187)])
def test_threads_and_pieces_follow_the_rows(lib, rows, nx, nf, per):
    err, src, dst, st = _read(lib, rows, nx, nf, reads=2, late=1)
    assert err == 0 and np.array_equal(dst, 2 * src.astype(np.float64))
    assert 1 <= st["threads"] <= st["given"] <= min(8, per), st
    row = 4 * nx * nf
    assert st["copies"] == nf * -(-rows // per), st
    assert st["most"] == 3 * per * row and per * row <= max(8 << 20, row), st
