"""Every uniform gets an index: the first basis whose running FP64 sum exceeds
it, the last basis if none does. Uniforms below 0 and far above the total, and
states whose running sum turns infinite or NaN (a NaN exceeds nothing), in the
single-launch form, in the table form with one and with several groups of
blocks, sorted and unsorted; and more shots than one
launch, one workgroup or one reading of a block takes."""
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


@pytest.mark.parametrize("n,shots", [(3, 1024), (3, 1025), (9, 50000), (14, 4097), (14, 40000), (15, 1023), (15, 70001),
                                     (17, 300000), (21, 100000)])
def test_many_shots(orc, hip, n, shots):
    """Both sides of the shots that a workgroup takes and of the forms for many
    in no order, half of them on a few bases, with values below 0 and beyond
    the total among them."""
    s = random_state(n, n + 7)
    s[s.size // 2:] *= 1e-3
    cum = orc.cumulative(s)
    rng = np.random.default_rng(shots)
    u = np.concatenate([rng.random(shots // 2) * cum[-1], 0.3 + 1e-4 * rng.random(shots - shots // 2 - 20),
                        -rng.random(10), cum[-1] + rng.random(10)])
    want = np.minimum(np.searchsorted(cum, u, side="right"), s.size - 1)
    order = np.argsort(u, kind="stable")
    d = hip.DeviceState(n)
    d.upload(s)
    assert np.array_equal(d.sample(u[order]).astype(np.int64), want[order])
    assert np.array_equal(d.sample_unsorted(u).astype(np.int64), want)
    d.free()


@pytest.mark.parametrize("n,draws", [(10, 1), (11, 5000), (12, 4095), (12, 4096), (14, 1), (15, 32768), (15, 32769),
                                     (20, 40000), (21, 65536), (22, 65537), (23, 70000)])
def test_draws_in_no_order(orc, hip, n, draws):
    from menos_amd import workloads as W
    r = hip.HipDenseEngine().execute(W.random_circuit(n, 3, n), statevector=True, region_sampler=True)
    u = np.random.default_rng(draws).random(draws)
    cum = orc.cumulative(r.statevector)
    with r.region_sampler as s:
        assert np.array_equal(s.draw(u).astype(np.int64),
                              np.minimum(np.searchsorted(cum, u, side="right"), cum.size - 1))
