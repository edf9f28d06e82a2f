"""Possible pairs by the boxes of 64-bead tiles (the list itself:
src/Updaters/possiblepairlist_kernel.cu:18-71): entries, order, counts and
the overflow flag are those of the all-pairs scan, exactly -- at the edges of
the tiles and of a wavefront's beads, for beads in no order along the chain
(every tile near: the collected tiles are worked off in parts), for more
exclusions than lanes, a row that overflows and coordinates that are not
finite."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _both(sysm, **kw):
    out = []
    for boxes in (True, False):
        with S.Engine(0, 8 << 30) as e:
            e.set_cells(min_beads=1, enabled=boxes)
            e.set_lds_step(False)
            j = e.add_job(S.make_params(**c0_params(pairs_threshold=32.0, **kw)), sysm, 0)
            e.rebuild(j, 3)
            cnt, ent = e.list(j, 3)
            out.append((e.status(j)[2], cnt, np.where(np.arange(ent.shape[0])[:, None] < cnt[None, :], ent, -1)))
    (fa, ca, ea), (fb, cb, eb) = out
    assert fa == fb
    np.testing.assert_array_equal(ca, cb)
    np.testing.assert_array_equal(ea, eb)
    return fa, ca


@pytest.mark.parametrize("n", [2, 5, 63, 64, 65, 130, 4097])
def test_edges(n):
    print("case: chain of %d" % n, flush=True)
    _, cnt = _both(S.synth_chain(n, seed=70 + n), max_possiblePairs=1024)
    assert n < 64 or cnt.max() > 0


def test_beads_in_no_order():
    sysm = S.synth_shell(40, 500, seed=5, radius=80.0)
    sysm.coords = np.ascontiguousarray(sysm.coords[np.random.default_rng(3).permutation(sysm.n)])
    print("case: 20,000 beads shuffled", flush=True)
    _, cnt = _both(sysm, max_possiblePairs=1024)
    assert cnt.max() > 256


def test_many_exclusions_and_overflow():
    sysm = S.synth_chain(700, seed=71)
    hub = np.array([(5, j) for j in range(100, 240)], np.int32)
    keep = ~(((sysm.natives == 5).any(1)) & ((sysm.natives >= 100).any(1)))
    sysm.natives = np.concatenate([sysm.natives[keep], hub])
    sysm.nat_r0 = np.concatenate([sysm.nat_r0[keep], np.full(len(hub), 6.0, np.float32)])
    sysm.nat_eh = np.concatenate([sysm.nat_eh[keep], np.full(len(hub), 1.0, np.float32)])
    print("case: 140 natives of one bead", flush=True)
    assert _both(sysm, max_possiblePairs=1024, max_native=256)[0] == 0
    print("case: rows that overflow", flush=True)
    assert _both(sysm, max_possiblePairs=64, max_native=256)[0] & 1


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_coordinates_not_finite(value):
    sysm = S.synth_chain(300, seed=72)
    sysm.coords[70, 0] = value
    sysm.coords[128:192, 1] = value
    print("case: coordinates of %r" % value, flush=True)
    _both(sysm, max_possiblePairs=1024)
