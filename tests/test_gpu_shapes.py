"""The launch shape says what runs: an engine that was not asked for rows per
wavefront reports -1 (chosen by the beads of the launch) and keeps it when
another field is set or the reported shape is set again; the autotuner
returns the shape it left set, also for jobs that take a block of steps in
one launch, and another engine takes it.  With one bead per lane asked for,
the fields of that step give the same bits."""
import numpy as np
import pytest

import sopgpu as S
from helpers import c0_params

pytestmark = pytest.mark.gpu


def _add(e, sizes, steps=10 ** 6):
    return [e.add_job(S.make_params(**c0_params(seed=31 + k, temperature=0.6, nav=100)),
                      S.synth_chain(n, seed=30 + k), steps) for k, n in enumerate(sizes)]


def test_the_choice_by_beads_is_kept():
    with S.Engine(0, 1 << 30) as e:
        assert e.shape()["split_rows"] == -1 and e.shape()["split_global"] == -1
        first = e.shape()
        e.set_shape(**first)
        assert e.shape() == first
        e.set_shape(sort_every=10)
        assert e.shape() == dict(first, sort_every=10)
        e.set_shape(split_rows=8)
        assert e.shape() == dict(first, sort_every=10, split_rows=8)
        e.set_shape(split_rows=-1)
        assert e.shape() == dict(first, sort_every=10)
        for bad in (-2, 1, 2, 3):
            for field in ("split_rows", "split_global"):
                with pytest.raises(S.SopError):
                    e.set_shape(**{field: bad})


@pytest.mark.parametrize("sizes", [[22] * 30, [300, 6000], [30, 7, 6000]], ids=["block", "spread", "mixed"])
def test_autotune_returns_the_shape_it_left(sizes):
    print("case: autotune on %d jobs up to %d beads" % (len(sizes), max(sizes)), flush=True)
    with S.Engine(0, 4 << 30) as e:
        ids = _add(e, sizes)
        e.run_blocks(3)
        rep = e.autotune()
        assert e.shape() == rep["shape"] and rep["ms_per_step_best"] <= rep["ms_per_step_start"]
        e.run_blocks(9)
        tuned = [e.coords(j) for j in ids]
    with S.Engine(0, 4 << 30) as e:
        e.set_shape(**rep["shape"])
        assert e.shape() == rep["shape"]
        ids = _add(e, sizes)
        e.run_blocks(12)
        for j, c in zip(ids, tuned):
            np.testing.assert_array_equal(e.coords(j), c)


@pytest.mark.parametrize("shape", [
    dict(unit_rows=512, shared_units=0, pair_batch=8, verlet_chunk=4, sort_every=10, max_blocks=256),
    dict(unit_rows=128, shared_units=1, pair_batch=4, verlet_chunk=8, sort_every=40),
])
def test_fields_of_the_one_lane_step(shape):
    sizes, got = [300, 1100, 2049, 6000], []
    for sh in (dict(), dict(split_rows=0, split_global=0, **shape)):
        with S.Engine(0, 4 << 30) as e:
            e.set_shape(**sh)
            ids = _add(e, sizes, 490)
            print("case: shape %r" % (sh,), flush=True)
            e.run_blocks(50)
            got.append([e.coords(j) for j in ids])
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)
