"""A block of steps in one launch, for small jobs: coordinates, generators,
temperatures and the forces after it are those of one launch per step, to the
bit -- for the smallest jobs and the largest it takes, jobs of several sizes
in one launch, ends inside a block, lists that overflow, heating, blocks longer than one launch, a tip and
a plane, minimization, and one job of the batch run by itself."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _job(n, seed, **kw):
    sysm = S.synth_chain(n, seed=seed)
    sysm.fixed = np.array([0], np.int32)
    sysm.pulled = np.array([n - 1], np.int32)
    base = dict(seed=seed + 1, pulling=1, fixedEnd=0, pulledEnd=n - 1, deltax=0.02, pullFreq=50, nav=50,
                outputtiming=50, dcdfreq=50, temperature=0.6)
    base.update(kw)
    return sysm, c0_params(**base)


def _compare(jobs, steps, blocks, alone=False):
    out = []
    for shape in (None, dict(split_rows=0, split_global=0)):
        with S.Engine(0, 8 << 30) as e:
            if shape is not None:
                e.set_shape(**shape)
            ids = [e.add_job(S.make_params(**kw), sysm, steps) for sysm, kw in jobs]
            if alone:
                e.run_job(ids[-1])
            else:
                e.run_blocks(blocks)
            out.append([x for j in ids
                        for x in (e.coords(j), e.rng(j), e.temperature(j), e.forces(j), np.array(e.status(j)))])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)


# eight rows per wavefront (up to 128 beads), sixteen above
@pytest.mark.parametrize("sizes", [[2], [32, 9, 2], [22] * 30, [33] * 101, [128] * 100 + [5], [256] * 100 + [17, 2]],
                         ids=["2", "32-9-2", "22x30", "33x101", "128x100", "256x100"])
def test_sizes(sizes):
    print("case: %d jobs up to %d beads" % (len(sizes), max(sizes)), flush=True)
    _compare([_job(n, 2000 + k) for k, n in enumerate(sizes)], 1000, 6)


@pytest.mark.parametrize("steps,blocks,kw", [
    (27, 5, {}), (1000, 3, dict(pairs_freq=300, possiblepairs_freq=300, nav=300, pullFreq=300, outputtiming=300,
                                dcdfreq=300)),
    (100, 6, dict(minimization=1)),
    (100, 6, dict(pulling=0, indentation=1, indTip=(0.0, 0.0, 80.0), indChip=(0.0, 0.0, 80.0),
                  indDirection=(0.0, 0.0, -1.0), indSurfR0=(0.0, 0.0, -60.0), indSurfN=(0.0, 0.0, 1.0), indTipR=20.0,
                  indKs=0.07, indDeltaX=0.01, indTipZeta=5000.0, indTipA=0.0, indTipB=1.0)),
    (100, 6, dict(max_pairs=4)),
    (100, 9, dict(heating=1, initialT=0.3, deltaT=0.05, tempFreq=20)),
], ids=["end-inside", "long-block", "minimization", "tip", "overflow", "heating"])
def test_forms(steps, blocks, kw):
    print("case: %r" % (kw,), flush=True)
    _compare([_job(n, 2100 + n, **kw) for n in (30, 22, 7)], steps, blocks)


def test_one_job_of_a_batch():
    print("case: run_job", flush=True)
    _compare([_job(n, 2200 + n) for n in (300, 22)], 95, 0, alone=True)
