"""Statistics of an iteration that cannot place its new determinants: whole-
number runs sum them in the prepass and the merge, before the insertion
refuses the list (MaxWalkers would be passed) or single determinants of it
(the walker hash is full).  TotParts, the norm, the walkers on the reference
and the number of occupied determinants that the failing call leaves are those
of the walker list that is kept, in the iteration's block and in the cycle's
sums; alone and in a batch."""
import numpy as np
import pytest

from common import hubbard_spec, mol_spec
from test_gpu_spawn_capacity import _dets

pytestmark = pytest.mark.gpu
TAU = 0.01
FULL = dict(walkers=2, hash=6)


def _spec(system, nrep, limit):
    kw = dict(init_walkers=2000, max_spawned=60_000, n_replicas=nrep, seed=5)
    if limit == "walkers":
        kw.update(max_walkers=1200, n_hash_buckets=4000)
    else:  # 1200 entries: 840 live ones are below the 80 % that is an error by itself
        kw.update(max_walkers=60_000, n_hash_buckets=300)
    return hubbard_spec(18, 18, 4.0, **kw) if system == "one" else mol_spec(33, 8, rank=4, **kw)


def _start(spec):
    from neci_stable_amd.engine import Engine
    eng = Engine(spec)
    d = _dets(spec, 840, np.random.default_rng(29))
    d[0] = eng.ref
    d = np.unique(d, axis=0)
    eng.upload(eng.rows(d, np.full((len(d), spec.S), 40.0)))
    return eng


def _kept(eng, st, S):
    d, sg = eng.download()[:2]
    live = np.abs(sg).sum(axis=1) > 0
    assert st["tot_walkers"] == live.sum()
    np.testing.assert_array_equal(st["tot_parts"][:S], np.abs(sg).sum(axis=0))
    np.testing.assert_array_equal(st["norm_sq"][:S], (sg * sg).sum(axis=0))
    np.testing.assert_array_equal(st["inst_no_at_hf"][:S], sg[(d == eng.ref).all(axis=1)].sum(axis=0))


CASES = [("one", 1), ("one", 2), ("one", 3), ("two", 1)]


@pytest.mark.parametrize("limit", ["walkers", "hash"])
@pytest.mark.parametrize("system,nrep", CASES)
def test_statistics_are_the_kept_lists(system, nrep, limit):
    from neci_stable_amd._lib import NgpuError
    spec = _spec(system, nrep, limit)
    eng = _start(spec)
    with pytest.raises(NgpuError) as e:
        eng.iterate(1, TAU, 0.0)
    assert e.value.code == FULL[limit]
    st = eng._out.to_dict(spec.S)
    assert st["n_new"] > 1000
    _kept(eng, st, spec.S)
    with pytest.raises(NgpuError):
        eng.cycle_stats()
    _kept(eng, eng._out.to_dict(spec.S), spec.S)
    eng.close()


@pytest.mark.parametrize("limit", ["walkers", "hash"])
def test_in_a_batch(limit):
    from neci_stable_amd._lib import NgpuError
    from neci_stable_amd.engine import Batch
    spec = _spec("one", 1, limit)
    engines = [_start(spec), _start(spec)]
    batch = Batch(engines)
    batch.iterate([1, 1], [TAU, TAU], [0.0, 0.0])
    for e in engines:
        with pytest.raises(NgpuError) as err:
            e.stats()
        assert err.value.code == FULL[limit]
        _kept(e, e._out.to_dict(1), 1)
    batch.close()
    for e in engines:
        e.close()
