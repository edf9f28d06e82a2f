"""The spread step as the engine chooses it when no shape is set: two, four,
eight or sixteen rows per wavefront by the beads of the launch.  Every choice
gives the one-bead-per-lane step's bits, at the smallest jobs (fewer rows
than a wavefront takes, lists shorter than its positions), at remainders
and for beads almost on top of each other (the general division)."""
import numpy as np
import pytest

import oracle as O
import sopgpu as S
from helpers import c0_params, numpy_chain

pytestmark = pytest.mark.gpu

ONE_LANE = dict(split_rows=0, split_global=0)


def _run(jobs, shape, blocks, lds=True):
    with S.Engine(0, 8 << 30) as e:
        if shape is not None:
            e.set_shape(**shape)
        e.set_lds_step(lds)
        ids = [e.add_job(S.make_params(**kw), sysm, 10 * blocks - 10) for sysm, kw in jobs]
        e.run_blocks(blocks)
        return [x for j in ids for x in (e.coords(j), e.rng(j), e.temperature(j), e.forces(j))]


def _job(n, seed, **kw):
    sysm = S.synth_chain(n, seed=seed)
    sysm.fixed = np.array([0], np.int32)
    sysm.pulled = np.array([n - 1], np.int32)
    return sysm, c0_params(seed=seed + 1, pulling=1, fixedEnd=0, pulledEnd=n - 1, deltax=0.02, pullFreq=50, nav=50,
                           outputtiming=50, dcdfreq=50, **kw)


# 2 rows (a launch of few rows), 8 rows (short lists), 4, 8 and 16 rows
@pytest.mark.parametrize("sizes", [[2], [3, 65, 130], [22] * 40 + [5], [1000] * 8 + [33], [4000] * 5 + [6001],
                                   [5000] * 8 + [71]], ids=["2", "3-65-130", "22x40", "1000x8", "4000x5", "5000x8"])
@pytest.mark.parametrize("lds", [True, False], ids=["lds", "global"])
def test_chosen_step_equals_one_lane_step(sizes, lds):
    jobs = [_job(n, 1100 + k) for k, n in enumerate(sizes)]
    print("case: rows %d in %d jobs" % (sum(sizes), len(sizes)), flush=True)
    for a, b in zip(_run(jobs, None, 12, lds), _run(jobs, ONE_LANE, 12, lds)):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("gap", [0.0, 1e-12, 1e-9])
def test_coincident_beads_take_the_general_division(gap):
    """Two far ends of a chain moved onto each other: d^2 below 2^-64 (and
    zero), where the quotient overflows; forces equal the oracle's."""
    n = 90
    sysm = numpy_chain(n, seed=1200)
    sysm.coords[n - 1, :3] = sysm.coords[0, :3]
    sysm.coords[n - 1, 0] = sysm.coords[0, 0] = 0.0
    sysm.coords[n - 1, 0] = gap
    keep = ~((sysm.natives[:, 0] == 0) & (sysm.natives[:, 1] == n - 1))
    sysm.natives, sysm.nat_r0, sysm.nat_eh = sysm.natives[keep], sysm.nat_r0[keep], sysm.nat_eh[keep]
    kw = c0_params()
    with S.Engine(0, 1 << 30) as e:
        j = e.add_job(S.make_params(**kw), sysm, 0)
        e.rebuild(j, 3)
        f = e.forces(j)
    ref = O.Sim(O.make_params(**kw), sysm)
    ref.build_possible()
    ref.build_verlet()
    np.testing.assert_array_equal(f, ref.forces32())


# a launch of one job takes its record as an argument, and so does one job of
# a batch run by itself; beside another job of its kind it reads the table
@pytest.mark.parametrize("n", [63, 65, 1000, 5121])
@pytest.mark.parametrize("rows", [4, 8, 16])
def test_one_job_equals_the_same_job_in_a_batch(n, rows):
    print("case: %d beads alone and in a batch, %d rows" % (n, rows), flush=True)
    job, other = _job(n, 1300), _job(130, 1301)
    shape = dict(split_rows=rows, split_global=rows)
    alone, batch = _run([job], shape, 6), _run([job, other], shape, 6)[:4]
    with S.Engine(0, 8 << 30) as e:
        e.set_shape(**shape)
        ids = [e.add_job(S.make_params(**kw), sysm, 50) for sysm, kw in (other, job)]
        e.run_job(ids[1])
        single = [e.coords(ids[1]), e.rng(ids[1]), e.temperature(ids[1]), e.forces(ids[1])]
    for a, b, c in zip(alone, batch, single):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a, c)
