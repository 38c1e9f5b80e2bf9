"""A spawned list past MaxSpawned whose determinants alone would pass every
list of the engine: max_walkers == max_spawned, and one iteration spawns many
times as many distinct determinants as either.  checkValidSpawnedList
(fcimc_helper.F90:483-510) stops the run between spawning and annihilation:
the call returns NGPU_ERR_SPAWN_FULL at the oracle's iteration, the engine
keeps the walkers of that point (parents after death, no spawn merged), and
nothing is left behind for a later engine.  One- and two-word determinants,
one, two and three replicas, FP64 and FP32 records, alone and in a batch.

The new list's bound: the merge takes a list only when it is no longer than
max_spawned, each merged determinant has at least one record, and the new
list has max(max_spawned, max_walkers) rows.
"""
import numpy as np
import pytest

from common import hubbard_spec, mol_spec, sort_walkers

pytestmark = pytest.mark.gpu
TAU = 0.01
CAP = 1500


def _dets(spec, n, rng):
    """n distinct random determinants with the reference's spin counts."""
    nsp = spec.nbasis // 2
    out = np.zeros((2 * n, spec.W), dtype=np.uint64)
    for spin in (1, 0):
        k = sum(1 for o in spec.ref_orbs if o % 2 == spin)
        occ = np.argpartition(rng.random((2 * n, nsp)), k - 1, axis=1)[:, :k]
        bit = 2 * occ + (0 if spin else 1)
        for j in range(k):
            np.bitwise_or.at(out, (np.arange(2 * n), bit[:, j] >> 6),
                             np.uint64(1) << (bit[:, j] & 63).astype(np.uint64))
    out = np.unique(out, axis=0)
    assert len(out) >= n
    return out[rng.permutation(len(out))[:n]].view(np.int64)


def _spec(system, nrep, fp32):
    kw = dict(init_walkers=CAP, max_spawned=CAP, max_walkers=CAP, n_hash_buckets=4000, n_replicas=nrep, seed=5,
              spawn_fp32=fp32)
    return hubbard_spec(18, 18, 4.0, **kw) if system == "one" else mol_spec(33, 8, rank=4, **kw)


def _start(spec):
    from neci_stable_amd.engine import Engine
    from oracle_ctypes import Oracle
    eng, orc = Engine(spec), Oracle(spec, TAU)
    d = _dets(spec, 1000, np.random.default_rng(17))
    sg = np.full((len(d), spec.S), 40.0)
    eng.upload(eng.rows(d, sg))
    orc.add_walkers(d, sg, np.zeros(len(d), dtype=np.uint32))
    return eng, orc


def _kept(eng, orc):
    a = sort_walkers(*eng.download()[:2])
    w = orc.walkers()
    b = sort_walkers(w[0], w[1])
    live = np.abs(b[1]).sum(axis=1) > 0
    np.testing.assert_array_equal(a[0], b[0][live])
    np.testing.assert_array_equal(a[1], b[1][live])


CASES = [("one", 1, False), ("one", 1, True), ("one", 2, False), ("one", 3, False), ("two", 1, False),
         ("two", 3, False)]


@pytest.mark.parametrize("system,nrep,fp32", CASES)
def test_more_new_determinants_than_the_lists_hold(system, nrep, fp32):
    from neci_stable_amd._lib import NgpuError
    spec = _spec(system, nrep, fp32)
    wide = _spec(system, nrep, fp32)
    # the same iteration with room: how many determinants it spawns
    from oracle_ctypes import Oracle
    big = Oracle(wide, TAU, max_walkers=400_000, max_spawned=400_000)
    d = _dets(spec, 1000, np.random.default_rng(17))
    big.add_walkers(d, np.full((len(d), nrep), 40.0), np.zeros(len(d), dtype=np.uint32))
    b = big.iterate(1, 0.0)
    assert b["rc"] == 0 and b["n_unique"] > 2 * CAP and b["n_new"] > 2 * CAP
    big.close()
    for _ in range(2):  # a second engine takes the memory the first one had
        eng, orc = _start(spec)
        assert orc.iterate(1, 0.0)["rc"] == 1
        with pytest.raises(NgpuError) as e:
            eng.iterate(1, TAU, 0.0)
        assert e.value.code == 1 and eng.error() == (1, 1)
        _kept(eng, orc)
        with pytest.raises(NgpuError):
            eng.iterate(2, TAU, 0.0)
        _kept(eng, orc)
        eng.close()
        orc.close()


def test_in_a_batch():
    from neci_stable_amd._lib import NgpuError
    from neci_stable_amd.engine import Batch, Engine
    spec = _spec("one", 1, False)
    full, orc = _start(spec)
    roomy = hubbard_spec(18, 18, 4.0, init_walkers=CAP, max_spawned=200_000, max_walkers=200_000, n_hash_buckets=60_000,
                         seed=5)
    ok, alone = Engine(roomy), Engine(roomy)
    d = _dets(spec, 1000, np.random.default_rng(17))
    for e in (ok, alone):
        e.upload(e.rows(d, np.full((len(d), 1), 40.0)))
    batch = Batch([full, ok])
    assert batch.groups()[1] == 1
    for it in (1, 2):
        batch.iterate([it, it], [TAU, TAU], [0.0, 0.0])
        alone.iterate(it, TAU, 0.0)
    assert orc.iterate(1, 0.0)["rc"] == 1
    assert full.error() == (1, 1) and ok.error() == (0, 0)
    with pytest.raises(NgpuError):
        full.stats()
    _kept(full, orc)
    for x, y in zip(sort_walkers(*ok.download()[:2]), sort_walkers(*alone.download()[:2])):
        np.testing.assert_array_equal(x, y)
    batch.close()
    for e in (full, ok, alone):
        e.close()
