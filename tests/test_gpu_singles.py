"""The queued single excitations where their division of the lanes can go wrong.

A wave takes up to 64 attempts a trip, with one lane each outside the weights
and 4, 8 or 16 lanes each for those, a lane holding pairs of neighbouring
orbitals.  Against the oracle, which draws one attempt at a time, from random
determinants (all orbitals of the reference replaced for many of them, so that
the lists of differing orbitals are as long as they get):
* numbers of orbitals at the ends of each instance's range, odd ones too, with
  one- and two-word determinants;
* a small grid, so that a wave makes several trips with all of its rounds, and
  the default one, where a trip is a part of a round.
Integer amplitudes: every statistic and walker is the same.
"""
import numpy as np
import pytest

from common import mol_spec
from test_gpu_parity import assert_same_walkers, assert_stats, random_dets

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [4, 8, 16])
@pytest.mark.parametrize("nspat,nel", [(3, 2), (15, 7), (16, 8), (17, 5), (24, 6), (25, 4), (32, 9), (33, 6), (40, 4),
                                       (41, 5), (48, 4), (49, 3)])
def test_singles_at_the_edges(nspat, nel, lanes):
    from neci_stable_amd.engine import Engine
    from oracle_ctypes import Oracle
    spec = mol_spec(nspat, nel, rank=4, init_walkers=4000, max_spawned=400000, max_walkers=200000,
                    n_hash_buckets=200000, seed=5, psingles=0.5)
    tau = 0.002
    rng = np.random.default_rng(nspat)
    dets = np.unique(random_dets(spec, 400, rng), axis=0)
    for blocks, amp in ((64, 300), (0, 3)):
        sg = rng.integers(1, amp + 1, (len(dets), 1)) * rng.choice([-1.0, 1.0], (len(dets), 1))
        eng, orc = Engine(spec), Oracle(spec, tau)
        eng.set_launch_shape(grid_blocks=blocks, single_lanes=lanes)
        eng.upload(eng.rows(dets, sg))
        orc.add_walkers(dets, sg, np.zeros(len(dets), dtype=np.uint32))
        for it in (1, 2):
            a = eng.iterate(it, tau, [0.1])
            b = orc.iterate(it, [0.1])
            assert b["rc"] == 0
            assert_stats(a, b, 1)
        assert_same_walkers(eng, orc)
        eng.close()
