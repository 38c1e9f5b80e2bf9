"""The spawn bins and the merge's LDS table at their edges.

Spawned records go to a bin chosen by a hash of their determinant; a wave
merges a bin in an LDS table of 128 determinants (64 for more than two
replicas), in further rounds when more meet there, and a full bin sends its
records to a spill area and, past that, to the overflow list.  Through the
explicit-list entry point (the same bins and merge as an iteration), lists of
integer amplitudes, whose sums are exact in any order, must give the oracle's
merged list:
* "few": fewer spawns than one bin takes;
* "wave": a list of 64 and of 65 distinct determinants in one bin;
* "crowded": distinct determinants whose hashes all fall into one 256th of
  the range, so that a few bins take them all: several rounds of the table,
  spill areas and overflow list;
* "one": every spawn on one determinant.
One- and two-word determinants, one, two and three replicas, FP64 and FP32
records.
"""
import numpy as np
import pytest

from common import hubbard_spec, mol_spec, sort_walkers

pytestmark = pytest.mark.gpu


def _bin_hash(d):
    """The engine's bin hash (high word) of (n, W) determinants."""
    d = d.view(np.uint64)
    with np.errstate(over="ignore"):
        h = d[:, 0] * np.uint64(0x9E3779B97F4A7C15)
        if d.shape[1] == 2:
            h = h + (d[:, 1] ^ (d[:, 1] >> np.uint64(29))) * np.uint64(0xBF58476D1CE4E5B9)
            h = (h ^ (h >> np.uint64(31))) * np.uint64(0x94D049BB133111EB)
    return (h >> np.uint64(32)).astype(np.uint64)


def _dets(spec, n, rng):
    """n random determinants with the reference's spin counts (repeats possible)."""
    nsp = spec.nbasis // 2
    out = np.zeros((n, spec.W), dtype=np.uint64)
    for spin in (1, 0):
        k = sum(1 for o in spec.ref_orbs if o % 2 == spin)
        occ = np.argpartition(rng.random((n, nsp)), k - 1, axis=1)[:, :k]
        bit = 2 * occ + (0 if spin else 1)
        for j in range(k):
            np.bitwise_or.at(out, (np.arange(n), bit[:, j] >> 6), np.uint64(1) << (bit[:, j] & 63).astype(np.uint64))
    return out.view(np.int64)


def _list(kind, spec, rng):
    if kind == "few":
        return _dets(spec, 7, rng)[rng.integers(0, 7, 20)]
    if kind == "one":
        return np.repeat(_dets(spec, 1, rng), 6000, axis=0)
    pool = np.unique(_dets(spec, 400_000, rng), axis=0)
    h = _bin_hash(pool)
    if kind.startswith("wave"):
        return pool[np.argsort(h)[:int(kind[4:])]]  # neighbours in the hash: one bin of a two- or three-bin list
    crowd = pool[h < np.uint64(1 << 24)]
    assert len(crowd) > 600
    sdet = crowd[rng.integers(0, len(crowd), 6000)]
    sdet[:len(crowd)] = crowd[:len(sdet)]
    return sdet


@pytest.mark.parametrize("kind", ["few", "wave64", "wave65", "crowded", "one"])
@pytest.mark.parametrize("system,nrep,fp32", [("one", 1, False), ("one", 1, True), ("one", 2, False), ("one", 3, False),
                                              ("two", 1, False), ("two", 1, True), ("two", 3, False)])
def test_merge_at_the_edges(kind, system, nrep, fp32):
    from neci_stable_amd.engine import Engine
    from oracle_ctypes import Oracle
    rng = np.random.default_rng(31)
    kw = dict(init_walkers=6000, max_spawned=6100, max_walkers=20000, n_hash_buckets=8000, n_replicas=nrep, seed=3,
              spawn_fp32=fp32)
    spec = hubbard_spec(18, 18, 4.0, **kw) if system == "one" else mol_spec(33, 8, rank=4, **kw)
    assert spec.W == (1 if system == "one" else 2)
    sdet = _list(kind, spec, rng)
    n = len(sdet)
    assert n <= 6100
    sval = rng.integers(-3, 4, n).astype(float)
    sval[sval == 0] = 1.0
    sinfo = ((rng.random(n) < 0.3).astype(np.uint32) << 8) | rng.integers(0, nrep, n).astype(np.uint32)
    eng, orc = Engine(spec), Oracle(spec, 0.01)
    # half of the list's determinants are resident, some with opposite signs
    res = np.unique(sdet, axis=0)[::2]
    sg = rng.integers(1, 6, (len(res), nrep)) * rng.choice([-1.0, 1.0], (len(res), nrep))
    eng.upload(eng.rows(res, sg))
    orc.add_walkers(res, sg, np.zeros(len(res), dtype=np.uint32))
    for it in (3, 4):  # the second list finds the counters the first left
        a, md, ms, mf = eng.annihilate(it, sdet, sval, sinfo)
        b, md2, ms2, mf2 = orc.annihilate(it, sdet, sval, sinfo)
        assert b["rc"] == 0
        for x, y in zip(sort_walkers(md, ms, mf), sort_walkers(md2, ms2, mf2)):
            np.testing.assert_array_equal(x, y)
        for f in ("nannihil", "naborted", "nremoved", "tot_parts", "norm_sq"):
            np.testing.assert_array_equal(a[f][:nrep], b[f][:nrep], err_msg=f)
        assert a["n_unique"] == b["n_unique"] and a["tot_walkers"] == b["tot_walkers"]
    eng.close()
