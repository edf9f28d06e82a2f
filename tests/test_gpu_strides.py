"""Small jobs of different strides in one batch: a block is the strides'
common divisor, so most blocks begin in the middle of a stride of some job --
no updater, no list and no cleared temperature of that job there -- and the
jobs end at different blocks.  The steps in one launch give the bits of one
launch per step and of each job alone, and the oracle's."""
import numpy as np
import pytest

import oracle as O
import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _job(n, stride, seed, **kw):
    sysm = S.synth_chain(n, seed=seed)
    sysm.fixed = np.array([0], np.int32)
    sysm.pulled = np.array([n - 1], np.int32)
    return sysm, c0_params(seed=seed + 1, temperature=0.6, pulling=1, fixedEnd=0, pulledEnd=n - 1, deltax=0.02,
                           pullFreq=stride, pairs_freq=stride, possiblepairs_freq=3 * stride, nav=2 * stride,
                           outputtiming=2 * stride, dcdfreq=2 * stride, **kw)


HEAT = dict(heating=1, initialT=0.3, deltaT=0.05)


# block lengths 5, 1 and (longer than one launch) 300
@pytest.mark.parametrize("jobs,L", [
    ([(22, 10, 100, dict(HEAT, tempFreq=20)), (30, 15, 200, {}), (7, 10, 60, {}),
      (25, 35, 280, dict(HEAT, tempFreq=35))], 5),
    ([(22, 7, 70, dict(HEAT, tempFreq=14)), (9, 10, 120, {})], 1),
    ([(22, 300, 900, {}), (12, 600, 1200, dict(HEAT, tempFreq=600))], 300),
], ids=["5", "1", "300"])
def test_strides(jobs, L):
    steps = max(j[2] for j in jobs)
    made = [_job(n, stride, 600 + k, **kw) + (end,) for k, (n, stride, end, kw) in enumerate(jobs)]
    out = []
    for shape in (dict(split_rows=-1), dict(split_rows=0, split_global=0)):
        with S.Engine(0, 1 << 30) as e:
            e.set_shape(**shape)
            ids = [e.add_job(S.make_params(**kw), sysm, end - 1) for sysm, kw, end in made]
            assert e.block_steps() == L
            got = []
            print("case: strides, blocks of %d, %r" % (L, shape), flush=True)
            for _ in range(3):  # in uneven parts
                e.run_blocks(max(1, steps // (2 * L) - 1))
                got += [x for j in ids for x in (e.coords(j), np.array(e.status(j)))]
            e.run_blocks(steps // L)
            got += [x for j in ids for x in (e.coords(j), e.rng(j), e.temperature(j), e.ext(j), np.array(e.status(j)),
                                             e.list(j, 2)[0], e.list(j, 3)[0])]
            out.append(got)
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    for q, (sysm, kw, end) in enumerate(made):
        with S.Engine(0, 1 << 30) as e:
            j = e.add_job(S.make_params(**kw), sysm, end - 1)
            e.run_job(j)
            alone = e.coords(j), e.rng(j), e.temperature(j)
        ref = O.Sim(O.make_params(**kw), sysm)
        ref.run(end - 1)
        together = out[0][-7 * len(made) + 7 * q:][:3]
        for a, b, c in zip(together, alone, (ref.coords(), ref.rng(), ref.temperature())):
            np.testing.assert_array_equal(a, b)
            np.testing.assert_array_equal(a, c)
