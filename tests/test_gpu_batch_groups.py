"""Launch groups of a batch: engines are grouped by what their kernels need.
The radix tile of the launch shape shapes no kernel, so engines that differ
in it alone share their launches; lanes per single attempt select another
kernel instance, so those do not."""
import pytest

from common import mol_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,groups", [(dict(radix_items=8), 1), (dict(radix_items=2), 1), (dict(single_lanes=8), 2)])
def test_groups_follow_the_kernels(shape, groups):
    from neci_stable_amd.engine import Batch, Engine
    engines = [Engine(mol_spec(8, 6, init_walkers=1000, seed=s)) for s in (1, 2)]
    engines[1].set_launch_shape(**shape)
    for e in engines:
        e.start_single_part(100.0)
    batch = Batch(engines)
    assert batch.groups()[1] == groups
    batch.iterate([1, 1], [0.01, 0.01], [0.0, 0.0])
    for e in engines:
        assert e.stats()["n_attempts"] == 100
    batch.close()
    for e in engines:
        e.close()
