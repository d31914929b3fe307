"""Wide blocks under a budget of exactly what the estimate says: their tables go
up for as few passes at a time as it leaves room for, with the same state."""
import pytest

from menos_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [4, 6])
@pytest.mark.parametrize("n", [14, 17])
def test_tables_within_the_budget(hip, n, width):
    c = W.random_circuit(n, 24, 6)
    eng = hip.HipDenseEngine()
    kw = dict(fusion=hip.FUSE_WIDTH, fusion_width=width)
    need = eng.estimate(c, **kw)
    want = eng.execute(c, targets=[], width=0, **kw)
    for budget in (need.device_bytes, need.device_bytes + (1 << 17), 1 << 30):
        got = eng.execute(c, targets=[], width=0, budget_bytes=budget, **kw)
        assert got.num_passes > 4 and got.statevector.tobytes() == want.statevector.tobytes(), budget
    with pytest.raises(hip.ResourceExceeded, match="budget"):
        eng.execute(c, targets=[], width=0, budget_bytes=need.device_bytes - 1, **kw)
