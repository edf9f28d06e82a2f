"""Timing the steps: the events count every step and leave the trajectories
as they are, also for jobs that take a block of steps in one launch (whose
updaters and Verlet lists are then built before the timed launch), with a
block longer than one launch."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,freq", [([22] * 5, 10), ([30, 7], 300), ([300], 10)],
                         ids=["block", "long-block", "step-launches"])
def test_profiled_steps(sizes, freq):
    out = []
    for profile in (True, False):
        with S.Engine(0, 1 << 30) as e:
            ids = []
            for k, n in enumerate(sizes):
                sysm = S.synth_chain(n, seed=50 + k)
                sysm.fixed = np.array([0], np.int32)
                sysm.pulled = np.array([n - 1], np.int32)
                ids.append(e.add_job(S.make_params(**c0_params(
                    seed=51 + k, temperature=0.6, pulling=1, fixedEnd=0, pulledEnd=n - 1, deltax=0.02, pullFreq=freq,
                    pairs_freq=freq, possiblepairs_freq=freq, nav=freq, outputtiming=freq, dcdfreq=freq,
                    heating=1, initialT=0.3, deltaT=0.05, tempFreq=freq)), sysm, 10 ** 6))
            e.profile(profile)
            print("case: %r, profile %s" % (sizes[:3], profile), flush=True)
            e.run_blocks(12)
            if profile:
                launches, ms = e.profile_read()
                assert launches == 12 * e.block_steps() and ms > 0.0
            out.append([x for j in ids for x in (e.coords(j), e.rng(j), e.temperature(j), e.ext(j), e.list(j, 2)[0])])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
