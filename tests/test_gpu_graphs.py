"""Blocks replayed several at a time from captured graphs: the trajectories are
those of direct launches, to the bit, over calls that begin anywhere in the
lists' periods, with reads, a written coordinate and a new job between them,
jobs that end on the way, and exact hydrodynamics (one block a graph)."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _run(graph, jobs, calls, late):
    with S.Engine(0, 8 << 30) as e:
        e.set_tuning(0, graph)
        ids = [e.add_job(S.make_params(**kw), sysm, steps) for sysm, kw, steps in jobs]
        out = []
        for k, blocks in enumerate(calls):
            e.run_blocks(blocks)
            out += [e.coords(j) for j in ids]
            if k == 2:
                e.set_coords(ids[0], out[-len(ids)] * np.float32(1.0001))
            if k == 3 and late:
                sysm, kw, steps = late
                ids.append(e.add_job(S.make_params(**kw), sysm, steps))
        return out + [x for j in ids for x in (e.rng(j), e.temperature(j), np.array(e.status(j)))]


def _job(n, seed, steps=10 ** 6, **kw):
    base = dict(seed=seed, temperature=0.6, nav=50)
    base.update(kw)
    return S.synth_chain(n, seed=seed), c0_params(**base), steps


@pytest.mark.parametrize("jobs,calls,late", [
    ([_job(300, 61), _job(40, 62)], [7, 120, 3, 95, 130, 1, 90], None),
    ([_job(22, 63)] * 3, [120, 30, 1, 60, 130], _job(25, 64)),
    ([_job(300, 65, steps=700), _job(22, 66, steps=1545)], [60, 60, 60], None),
    ([_job(40, 67, hi_on=1, hi_exact=1, hi_a=1.9, hi_chol_freq=3)], [9, 14, 3, 12], None),
], ids=["two-sizes", "late-job", "ends", "exact-hi"])
def test_graphs_equal_direct_launches(jobs, calls, late):
    print("case: %d jobs, calls %r" % (len(jobs), calls), flush=True)
    for a, b in zip(_run(True, jobs, calls, late), _run(False, jobs, calls, late)):
        np.testing.assert_array_equal(a, b)
