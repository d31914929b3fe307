"""Every uniform gets an index: the first basis whose running FP64 sum exceeds
it, the last basis if none does. Uniforms below 0 and far above the total, and
states whose running sum turns infinite or NaN (a NaN exceeds nothing), in the
single-launch form, in the table form with one and with several groups of
blocks, sorted and unsorted; and more shots than one launch takes."""
import numpy as np
import pytest

from circuits import random_state

pytestmark = pytest.mark.gpu


def _first_exceeding(cum, u):
    with np.errstate(invalid="ignore"):
        past = [np.flatnonzero(cum > x) for x in u]
    return np.array([p[0] if p.size else cum.size - 1 for p in past], np.int64)


def _check(hip, orc, s, u):
    n = int(np.log2(s.size))
    want = _first_exceeding(orc.cumulative(s), u)
    d = hip.DeviceState(n)
    d.upload(s)
    # Whatever the pool's memory held before, it is not these answers.
    got = d.sample(np.sort(u)).astype(np.int64)
    assert np.array_equal(got, _first_exceeding(orc.cumulative(s), np.sort(u)))
    assert np.array_equal(d.sample_unsorted(u).astype(np.int64), want)
    one = np.array([d.sample(u[i:i + 1])[0] for i in range(0, u.size, max(u.size // 6, 1))], np.int64)
    assert np.array_equal(one, want[::max(u.size // 6, 1)])
    d.free()


SIZES = [1, 6, 11, 12, 14, 15, 19, 21, 22]


@pytest.mark.parametrize("n", SIZES)
def test_uniforms_outside_the_range(orc, hip, n):
    s = random_state(n, n)
    s[:s.size // 4] = 0          # a uniform below 0 is exceeded before there is any mass
    u = np.concatenate([-np.random.default_rng(n).random(40), [-1e300, -5e-324, -0.0, 0.0, 0.25, 0.75, 2.0, 1e300],
                        np.random.default_rng(n + 1).random(20)])
    _check(hip, orc, s, np.random.default_rng(2).permutation(u))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("at", ["first", "early", "middle", "last"])
@pytest.mark.parametrize("value", [np.nan, np.inf, 1e200])
def test_sums_that_are_not_finite(orc, hip, n, at, value):
    """1e200 squared is the infinity."""
    s = random_state(n, n + 50)
    s[{"first": 0, "early": s.size // 100, "middle": s.size // 2 - 1, "last": s.size - 1}[at]] = value
    u = np.concatenate([np.random.default_rng(n).random(24), [-1.0, 0.0, 1e-9, 0.4999, 0.5001, 1.5]])
    _check(hip, orc, s, u)


def test_more_shots_than_one_launch(orc, hip):
    """2^23 shots a launch: the boundary falls inside a block's shots."""
    n, shots = 15, (1 << 23) + 1000
    s = random_state(n, 9)
    u = np.sort(np.random.default_rng(3).random(shots))
    d = hip.DeviceState(n)
    d.upload(s)
    got = d.sample(u).astype(np.int64)
    d.free()
    want = np.minimum(np.searchsorted(orc.cumulative(s), u, side="right"), s.size - 1)
    assert np.array_equal(got, want)
