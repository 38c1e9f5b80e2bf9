"""The number of spawn bins when the previous iteration's spawning rate says
nothing about the next one: an iteration with a time step too small to spawn,
and a large upload after iterations of a few walkers.  The iteration that
follows spawns about 1.5e5 records; it must be the oracle's, and its merge must
not search one bin for all of them.

Bound on the merge's time: at least one spawn in 64 attempts is expected, so a
bin of 44 expected records holds at most 64 * 44 = 2816, which a wave merges in
at most 22 rounds of 44 steps; at a microsecond a step that is 1 ms.  10 ms
leaves a factor of ten; one bin of all records takes 2.3e3 steps in each of
some 900 rounds.
"""
import numpy as np
import pytest

from common import hubbard_spec
from test_gpu_parity import assert_stats
from test_gpu_spawn_capacity import _dets

pytestmark = pytest.mark.gpu
TAU = 0.05
MERGE_STAGE = 6


@pytest.mark.parametrize("before", ["no_spawns", "few_walkers"])
def test_bins_after_an_iteration_that_spawned_nothing(before):
    from neci_stable_amd.engine import Engine
    from oracle_ctypes import Oracle
    spec = hubbard_spec(18, 18, 4.0, init_walkers=200_000, max_spawned=400_000, max_walkers=400_000,
                        n_hash_buckets=200_000, seed=5)
    tiny = 1e-9
    d = _dets(spec, 20_000, np.random.default_rng(23))
    sg = np.full((len(d), 1), 10.0)
    fl = np.zeros(len(d), dtype=np.uint32)
    eng = Engine(spec)
    orc, orc_tiny = Oracle(spec, TAU), Oracle(spec, tiny)
    few = slice(0, 2)
    if before == "no_spawns":
        eng.upload(eng.rows(d, sg))
        a = eng.iterate(1, tiny, 0.0)
        orc_tiny.add_walkers_bulk(d, sg, fl)
        assert_stats(a, orc_tiny.iterate(1, 0.0), 1)
        assert a["n_spawned"] == 0
        w = orc_tiny.walkers()
        orc.add_walkers_bulk(w[0], w[1], w[2])
    else:
        eng.upload(eng.rows(d[few], sg[few]))
        a = eng.iterate(1, tiny, 0.0)
        orc_tiny.add_walkers_bulk(d[few], sg[few], fl[few])
        assert_stats(a, orc_tiny.iterate(1, 0.0), 1)
        assert a["n_spawned"] == 0
        w = orc_tiny.walkers()
        orc.add_walkers_bulk(w[0], w[1], w[2])
        rest = slice(2, None)
        eng.upload(eng.rows(d[rest], sg[rest]))
        orc.add_walkers_bulk(d[rest], sg[rest], fl[rest])
    eng.set_profiling(1 << MERGE_STAGE)
    a, b = eng.iterate(2, TAU, 20.0), orc.iterate(2, 20.0)
    assert b["rc"] == 0 and b["n_unique"] > 50_000
    assert_stats(a, b, 1)
    ms, n = eng.stage_times()
    assert n == 1 and ms[MERGE_STAGE] < 10.0
    eng.close()
