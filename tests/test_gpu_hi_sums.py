"""The all-pairs hydrodynamic sums at each workgroup shape that the bead
count of a launch chooses (4, 8 or 16 beads, chunks of 256 or 128
partners), with pairs outside the short evaluation's range (separations
with a zero or tiny component, radii near zero or huge), and epsilon's
parallel sum beside its one-by-one fallback: the oracle's bits."""
import numpy as np
import pytest

import oracle as O
import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _kw(n, **kw):
    d = c0_params(hi_on=1, hi_a=1.9, hi_epsilon_freq=10, hi_capricious=0, hi_unlisted=1, pulling=1, fixedEnd=0,
                  pulledEnd=n - 1, fconst=1.4, nav=100, outputtiming=100, dcdfreq=100)
    d.update(kw)
    return d


def _chain(n, seed):
    sysm = S.synth_chain(n, seed=seed)
    sysm.fixed = np.array([0], np.int32)
    sysm.pulled = np.array([n - 1], np.int32)
    return sysm


def _equal_to_oracle(sysm, kw, steps):
    with S.Engine(0, 2 << 30) as e:
        j = e.add_job(S.make_params(**kw), sysm, steps)
        e.run_job(j)
        got = e.coords(j), e.rng(j), e.hi(j)
    ref = O.Sim(O.make_params(**kw), sysm)
    ref.run(steps)
    np.testing.assert_array_equal(got[0], ref.coords())
    np.testing.assert_array_equal(got[1], ref.rng())
    eps, beta = ref.hi_tea()
    np.testing.assert_array_equal(got[2][0], eps[0])
    np.testing.assert_array_equal(got[2][1], beta[0])


# workgroups of 4, 8 and 16 beads; last beads alone in their workgroup, and
# partner counts around a chunk
@pytest.mark.parametrize("n", [1, 2, 65, 257, 1025, 2049])
def test_tea_sums_equal_the_oracle(n):
    print("case: TEA n=%d" % n, flush=True)
    kw = _kw(n) if n > 1 else _kw(n, pulling=0)
    _equal_to_oracle(_chain(n, 1300 + n), kw, 10)


def test_tea_sums_of_many_jobs_equal_each_alone():
    """More than 4,096 beads in the launch: workgroups of 8 beads, chunks of 128."""
    jobs = [(_chain(n, 1400 + k), _kw(n, seed=1410 + k)) for k, n in enumerate([1000, 1500, 129, 1700])]
    with S.Engine(0, 4 << 30) as e:
        ids = [e.add_job(S.make_params(**kw), s, 20) for s, kw in jobs]
        e.run_blocks(3)
        together = [e.coords(j) for j in ids]
    for (s, kw), c in zip(jobs, together):
        with S.Engine(0, 4 << 30) as e:
            j = e.add_job(S.make_params(**kw), s, 20)
            e.run_job(j)
            np.testing.assert_array_equal(e.coords(j), c)


@pytest.mark.parametrize("a", [1.9, 3.8, 1e-9, 3e7])
def test_pairs_outside_the_short_range_equal_the_oracle(a):
    """Beads that share a coordinate, almost share one, or lie 1e12 A away;
    hydrodynamic radii outside the short evaluation's range."""
    n = 130
    sysm = _chain(n, 1500)
    free = np.arange(n) >= 100       # beads 100 .. are not bonded to anything
    for name, r0 in (("bonds", "bond_r0"), ("natives", "nat_r0")):
        ij = getattr(sysm, name)
        keep = ~free[ij].any(axis=1)
        setattr(sysm, name, ij[keep])
        setattr(sysm, r0, getattr(sysm, r0)[keep])
        if name == "natives":
            sysm.nat_eh = sysm.nat_eh[keep]
    sysm.coords[100:110, 0] = sysm.coords[5, 0]
    sysm.coords[110:115, 1] = 0.0
    sysm.coords[112, 1] = 1e-14
    sysm.coords[100:120, 2] += 60.0
    sysm.coords[120, :3] = (1e12, 3.0, -4.0)
    print("case: pairs outside the short range, a=%g" % a, flush=True)
    _equal_to_oracle(sysm, _kw(n, hi_a=a), 0)


def test_epsilon_of_values_far_apart_is_added_in_order():
    """One bead so far away that its epsilon lies 2^22 below the others': the
    sum is not exact in any order, and is formed bead by bead."""
    n = 90
    sysm = _chain(n, 1600)
    far = n - 2
    keep = ~(sysm.bonds == far).any(axis=1)
    sysm.bonds, sysm.bond_r0 = sysm.bonds[keep], sysm.bond_r0[keep]
    keep = ~(sysm.natives == far).any(axis=1)
    sysm.natives, sysm.nat_r0, sysm.nat_eh = sysm.natives[keep], sysm.nat_r0[keep], sysm.nat_eh[keep]
    sysm.coords[far, :3] = (4e9, 1e9, 2e9)
    _equal_to_oracle(sysm, _kw(n), 0)
