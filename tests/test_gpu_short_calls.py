"""Calls of fewer blocks than a graph holds: from 50 steps on they are replayed
from a graph of their own, and the host's share of a call falls with it;
shorter ones and odd remainders, after captures and among longer calls, give
the trajectories of direct launches, to the bit."""
import time

import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _engine(graph, sizes):
    e = S.Engine(0, 8 << 30)
    e.set_tuning(0, graph)
    ids = [e.add_job(S.make_params(**c0_params(seed=81 + k, temperature=0.6, nav=50)), S.synth_chain(n, seed=80 + k),
                     10 ** 6) for k, n in enumerate(sizes)]
    return e, ids


@pytest.mark.parametrize("sizes", [[300, 40], [22] * 3], ids=["step-launches", "block-launches"])
@pytest.mark.parametrize("calls", [[5] * 44, [7, 5, 13, 1, 26, 9] * 14, [3] * 30 + [5] * 30], ids=str)
def test_short_calls_equal_direct_launches(sizes, calls):
    print("case: %r, %d calls %r .." % (sizes, len(calls), calls[:6]), flush=True)
    out = []
    for graph in (True, False):
        e, ids = _engine(graph, sizes)
        got = []
        for k, blocks in enumerate(calls):
            e.run_blocks(blocks)
            if k % 11 == 0:
                got += [e.coords(j) for j in ids]
        out.append(got + [x for j in ids for x in (e.coords(j), e.rng(j), e.temperature(j), np.array(e.status(j)))])
        e.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


def test_repeated_calls_of_five_blocks_are_replayed():
    """A replay takes the host a fraction of the calls' 65 launches (20 us
    and 200): half is the line."""
    host = []
    for graph in (True, False):
        e, _ = _engine(graph, [1000])
        for _ in range(60):  # every phase of the lists has come more than four times
            e.run_blocks(5)
        e.synchronize()
        best = 1e9
        for _ in range(5):
            t = 0.0
            for _ in range(8):
                a = time.perf_counter()
                e.run_blocks(5)
                t += time.perf_counter() - a
            e.synchronize()
            best = min(best, t / 8)
        host.append(best)
        e.close()
    print("case: host's share of a call %.0f us with graphs, %.0f without" % (host[0] * 1e6, host[1] * 1e6), flush=True)
    assert host[0] < 0.5 * host[1]
