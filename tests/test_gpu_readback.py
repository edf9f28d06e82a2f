"""Coordinates read back through pinned host memory: what was written is read
at every buffer parity and on both sides of the staging size, with blocks
still running in front of the read, and several jobs in turn."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 1023, 1025, 16384, 16385])
def test_read_after_running_blocks(n):
    print("case: %d beads" % n, flush=True)
    sysm = S.synth_chain(n, seed=81)
    kw = c0_params(seed=82, pairs_freq=5, possiblepairs_freq=50, nav=50)
    with S.Engine(0, 8 << 30) as e:
        a, b = (e.add_job(S.make_params(**kw), sysm, 4000) for _ in range(2))
        seen = []
        for blocks in (1, 1, 60):  # 5 steps, 10 steps, a long run not waited for
            e.run_blocks(blocks)
            x, y = e.coords(a), e.coords(b)
            np.testing.assert_array_equal(x, y)
            e.synchronize()
            np.testing.assert_array_equal(x, e.coords(a))
            seen.append(x)
        assert not np.array_equal(seen[0], seen[1]) and not np.array_equal(seen[1], seen[2])
        new = x + np.float32(1.0)
        e.set_coords(b, new)
        np.testing.assert_array_equal(e.coords(b), new)
        np.testing.assert_array_equal(e.coords(a), x)
