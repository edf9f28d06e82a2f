"""Per-bead energies from terms spread over a wavefront, added in list order:
the oracle's bits at row counts around a wavefront's and a workgroup's rows,
and for a bead with more natives than a chunk holds."""
import numpy as np
import pytest

import oracle as O
import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _check(sysm, **kw):
    kw = c0_params(**kw)
    ref = O.Sim(O.make_params(**kw), sysm)
    ref.build_possible()
    ref.build_verlet()
    with S.Engine(0, 4 << 30) as e:
        j = e.add_job(S.make_params(**kw), sysm, 0)
        e.rebuild(j, 3)
        per, sums = e.energies(j)
    np.testing.assert_array_equal(per, ref.energies32())
    np.testing.assert_array_equal(sums, ref.sum_energies()[:, 0])


@pytest.mark.parametrize("n", [2, 3, 4, 5, 15, 17, 65, 700])
def test_sizes(n):
    print("case: chain of %d" % n, flush=True)
    sysm = S.synth_chain(n, seed=90 + n)
    sysm.coords[:, :3] += np.random.default_rng(n).normal(0.0, 0.1, (n, 3)).astype(np.float32)
    _check(sysm)


def test_many_natives():
    sysm = S.synth_chain(300, seed=91)
    keep = ~((sysm.natives == 5).any(1) & (sysm.natives >= 100).any(1))
    hub = np.array([(5, j) for j in range(100, 240)], np.int32)
    sysm.natives = np.concatenate([sysm.natives[keep], hub])
    sysm.nat_r0 = np.concatenate([sysm.nat_r0[keep], np.full(len(hub), 6.0, np.float32)])
    sysm.nat_eh = np.concatenate([sysm.nat_eh[keep], np.full(len(hub), 1.3, np.float32)])
    print("case: 140 natives of one bead", flush=True)
    _check(sysm, max_native=256)
