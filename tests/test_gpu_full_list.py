"""Spawned lists close to their capacity with many records per determinant (a
10-site chain's determinants with some 700 walkers each, a few with most of
them): most records find their bin full.  The iteration is that of an engine
with room, and the merge's time grows with the list, not with its square: four
times the list takes less than eight times as long (and half a millisecond), in
the first iteration, whose number of determinants is not known beforehand, and
in the next.  (With the records of full bins searched by every bin's wave it
took 15 times as long.)"""
from itertools import combinations

import numpy as np
import pytest

from common import hubbard_spec, sort_walkers

pytestmark = pytest.mark.gpu
TAU = 0.01
MERGE_STAGE = 6
EXACT = ["nborn", "ndied", "nannihil", "naborted", "nremoved", "tot_parts", "norm_sq", "inst_no_at_hf"]


def _spec(max_spawned):
    return hubbard_spec(10, 10, 4.0, init_walkers=1_000_000, max_spawned=max_spawned, max_walkers=100_000,
                        n_hash_buckets=100_000, seed=3)


def _dets(n):
    """n of the chain's 252^2 determinants."""
    half = [sum(1 << (2 * s) for s in c) for c in combinations(range(10), 5)]
    d = (np.array(half, dtype=np.int64)[:, None] | (np.array(half, dtype=np.int64)[None, :] << 1)).reshape(-1)
    return np.random.default_rng(37).permutation(d)[:n, None]


def _full_list(ndets):
    """Merge times (ms) of two iterations with a list that they fill, checked against an engine with room."""
    from neci_stable_amd.engine import Engine
    d = _dets(ndets)
    sg = np.ceil(100 * np.random.default_rng(41).lognormal(0.0, 2.0, (ndets, 1)))  # a few hold most
    room = Engine(_spec(16_000_000))
    room.upload(room.rows(d, sg))
    want = [room.iterate(it, TAU, 0.0) for it in (1, 2)]
    full = Engine(_spec(max(w["n_spawned"] for w in want) + 10))
    full.upload(full.rows(d, sg))
    ms = []
    for it in (1, 2):
        full.set_profiling(1 << MERGE_STAGE)
        got = full.iterate(it, TAU, 0.0)
        ms.append(full.stage_times()[0][MERGE_STAGE])
        for f in EXACT:
            np.testing.assert_array_equal(got[f], want[it - 1][f], err_msg=f)
        for f in ("n_spawned", "n_unique", "n_new", "tot_walkers"):
            assert got[f] == want[it - 1][f]
    for x, y in zip(sort_walkers(*full.download()[:3]), sort_walkers(*room.download()[:3])):
        np.testing.assert_array_equal(x, y)
    room.close()
    full.close()
    return ms, want[0]["n_spawned"]


def test_time_grows_with_the_list():
    _full_list(1000)  # the kernels' first launches
    small, n_small = _full_list(15_000)
    big, n_big = _full_list(60_000)
    print(f"merge {small} ms at {n_small} spawns, {big} ms at {n_big}", flush=True)
    assert 3.5 * n_small < n_big < 4.5 * n_small
    for a, b in zip(small, big):
        assert b < 8 * a + 0.5
