"""Runs of the captured step in graphs of several lengths: counts that take
each length, and their remainders, in sequence on one handle with reads in
between, against the same steps launched one by one, bit for bit; gas and dust
with wave killing, an inviscid gas disk, and with the time average on."""
import numpy as np
import pytest

from penguin_amd import Disk, config_c1, config_c2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg, kw, ave", [(config_c2, {}, False), (config_c1, {"visc_flag": 0}, False),
                                          (config_c1, {}, True)])
def test_graph_lengths(cfg, kw, ave):
    p = cfg(xres=40, yres=96).replace(ramp_time=1e-3, **kw)
    a, b = Disk(p), Disk(p)
    if ave:
        a.average_begin(1.0)
        b.average_begin(1.0)
    for n in (1, 3, 4, 5, 16, 21, 37):
        da, db = a.run(n, use_graph=True), b.run(n, use_graph=False)
        assert np.array_equal(da, db) and a.t == b.t, n
        for x, y in zip(a.get_state(), b.get_state()):
            assert x is None or np.array_equal(x, y), n
    if ave:
        assert np.array_equal(a.average(), b.average())
    a.close()
    b.close()
