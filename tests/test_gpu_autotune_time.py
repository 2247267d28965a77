"""What pg_batch_autotune reports is device time of captured steps: never more
than a whole call of as many steps takes, launches, copies and all, on the
schedule it chose, once that call's graphs are there.  (A disk whose step takes
some 20 us shows it: recording and instantiating the graphs of 20 steps takes
about as long as running them.  A tenth is allowed for one timing against the
best of twenty.)"""
import time

import pytest

from penguin_amd import Batch, disk2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [4, 5])
def test_reported_time_is_of_replays(steps):
    with Batch([disk2d(64, 128)]) as b:
        best = b.autotune(steps)
        n = 4 * steps                      # what the finalists are timed over
        calls = []
        for _ in range(20):
            t0 = time.perf_counter()
            b.run(n)
            calls.append(1e3 * (time.perf_counter() - t0) / n)
        print(f"autotune {best:.4f} ms per step, a call of {n} steps {min(calls):.4f}", flush=True)
        assert 0.0 < best <= 1.1 * min(calls)
