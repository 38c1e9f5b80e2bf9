"""Explicit spawned lists of real amplitudes: the records of a determinant are
summed in the order of the list, so that the merged list is the same to the
last bit on every call (CompressSpawnedList sums a sorted list front to back).
Lists short and long, spread and crowded into a few bins whose records spill
into their areas and the overflow list, and longer than one step of the upload.
Only bits 0 to 8 of the info word mean anything (include/neci_gpu.h): others
change nothing."""
import numpy as np
import pytest

from common import hubbard_spec, mol_spec, sort_walkers
from test_gpu_bins import _dets, _list

pytestmark = pytest.mark.gpu


def _case(kind, system, nrep, fp32):
    rng = np.random.default_rng(41)
    n = 300_000 if kind == "long" else 6000
    kw = dict(init_walkers=6000, max_spawned=n + 100, max_walkers=20000, n_hash_buckets=8000, n_replicas=nrep, seed=3,
              spawn_fp32=fp32, all_real_coeff=True)
    spec = hubbard_spec(18, 18, 4.0, **kw) if system == "one" else mol_spec(33, 8, rank=4, **kw)
    if kind in ("spread", "long"):
        pool = np.unique(_dets(spec, 500, rng), axis=0)
        sdet = pool[rng.integers(0, len(pool), n)]
    else:
        sdet = _list(kind, spec, rng)
    sval = rng.standard_normal(len(sdet)) * 10.0 ** rng.uniform(-3, 3, len(sdet))
    sinfo = ((rng.random(len(sdet)) < 0.3).astype(np.uint32) << 8) | rng.integers(0, nrep, len(sdet)).astype(np.uint32)
    return spec, sdet, sval, sinfo


def _in_list_order(spec, sdet, sval, sinfo, fp32):
    d, inv = np.unique(sdet, axis=0, return_inverse=True)
    s = np.zeros((len(d), spec.S))
    v = sval.astype(np.float32).astype(np.float64) if fp32 else sval
    np.add.at(s, (inv.reshape(-1), (sinfo & 0xFF).astype(int)), v)  # one record after another
    return sort_walkers(d, s)


@pytest.mark.parametrize("kind", ["spread", "crowded", "one", "long"])
@pytest.mark.parametrize("system,nrep,fp32", [("one", 1, False), ("one", 1, True), ("one", 2, False), ("two", 1, False),
                                              ("two", 3, False)])
def test_sums_in_list_order(kind, system, nrep, fp32):
    from neci_stable_amd.engine import Engine
    spec, sdet, sval, sinfo = _case(kind, system, nrep, fp32)
    want = _in_list_order(spec, sdet, sval, sinfo, fp32)
    for _ in range(2):
        eng = Engine(spec)
        _, md, ms, _ = eng.annihilate(3, sdet, sval, sinfo)
        got = sort_walkers(md, ms)
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
        eng.close()


@pytest.mark.parametrize("kind", ["crowded", "spread"])
def test_other_bits_of_the_info_word_mean_nothing(kind):
    from neci_stable_amd.engine import Engine
    spec, sdet, sval, sinfo = _case(kind, "one", 2, False)
    out = []
    for extra in (0, 0xFFFFFE00):
        eng = Engine(spec)
        a, md, ms, mf = eng.annihilate(3, sdet, sval, sinfo | np.uint32(extra))
        out.append(sort_walkers(md, ms, mf) + (a["n_unique"], a["n_new"]))
        eng.close()
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
