"""Stochastic rounding of spawns and deaths outside what a 64-bit integer
holds.  The integer part is a 64-bit conversion (INT of the reference), so a
NaN probability spawns and kills nothing and an infinite or huge one gives a
finite number within the integer range; inside the range it is the truncated
value, never a negative zero."""
import numpy as np
import pytest

from common import hubbard_spec

pytestmark = pytest.mark.gpu
LIMIT = 2.0 ** 63


def test_integer_part():
    from neci_stable_amd.engine import Engine
    eng = Engine(hubbard_spec(10, 10, 4.0))
    inside = np.array([0.0, -0.0, 0.3, -0.3, 0.7, -0.7, 1.0, -1.0, 2.5e9, 4.5e15 + 0.5, LIMIT - 1024.0, -LIMIT + 1024.0])
    outside = np.array([np.inf, 1e19, 1e25, 1e300, LIMIT])
    outside = np.concatenate([outside, -outside])
    u = 0.5
    for x, call in ((1.0, lambda v: eng.attempt_die(v, np.ones(len(v)), np.full(len(v), u), 1.0, 0.0)),
                    (-1.0, lambda v: eng.attempt_create(v, np.ones(len(v)), np.ones(len(v)), np.full(len(v), u), 1.0))):
        got = call(inside)
        v = x * inside  # a spawn of H > 0 from a positive parent is negative
        want = np.trunc(v) + np.where(np.abs(v - np.trunc(v)) > u, np.sign(v), 0.0)
        np.testing.assert_array_equal(got, want)
        assert not np.signbit(got[got == 0.0]).any()
        got = call(outside)
        assert np.isfinite(got).all() and (np.sign(got) == np.sign(x * outside)).all()
        assert (np.abs(got) <= LIMIT).all() and (np.abs(got) >= LIMIT - 2.0 ** 32).all()
        np.testing.assert_array_equal(call(np.array([np.nan])), [0.0])
    eng.close()


def test_a_shift_that_is_not_a_number_kills_nothing():
    from neci_stable_amd.engine import Engine
    eng = Engine(hubbard_spec(10, 10, 4.0, init_walkers=1000, seed=3))
    eng.start_single_part(200.0)
    a = eng.iterate(1, 1e-12, float("nan"))
    assert a["ndied"][0] == 0.0 and a["tot_parts"][0] == 200.0
    d, s = eng.download()[:2]
    assert len(d) == 1 and s[0, 0] == 200.0
    eng.close()
