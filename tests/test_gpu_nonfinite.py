"""An amplitude that is not finite: what a block makes of its own group is the
pass's (exact permutations move it, real blocks leave out products by zero), but
nothing outside the qubits that the blocks act on changes: every amplitude that
no chain of groups joins to it has the oracle's bits."""
import numpy as np
import pytest

from circuits import random_state, random_unitary

pytestmark = pytest.mark.gpu

X = np.array([[0, 1], [1, 0]], np.complex128)
H = np.array([[1, 1], [1, -1]], np.complex128) / np.sqrt(2)
CX = np.eye(4)[[0, 3, 2, 1]].astype(np.complex128)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,width", [(8, 2), (13, 2), (16, 2), (16, 4)])
def test_the_rest_of_the_state_is_untouched(orc, hip, n, width, bad):
    rng = np.random.default_rng(n + width)
    mine = sorted(int(q) for q in rng.permutation(n)[:5])
    at = int(rng.integers(0, 1 << n))
    start = random_state(n, n)
    start[at] = complex(bad, 0.5)
    blocks = []
    for _ in range(20):
        q = [int(x) for x in rng.permutation(mine)]
        k = int(rng.integers(0, 5 if width == 4 else 4))
        blocks.append([(X, q[:1]), (H, q[:1]), (CX, q[:2]), (random_unitary(2, rng), q[:2]),
                       (random_unitary(4, rng), q[:4])][k])
    d = hip.DeviceState(n)
    d.upload(start)
    d.apply_blocks(blocks)
    got = d.download()
    d.free()
    want = start.copy()
    for m, qs in blocks:
        orc.apply_generic(want, m, qs)
    mask = sum(1 << q for q in mine)
    apart = ((np.arange(1 << n) ^ at) & ~mask & ((1 << n) - 1)) != 0
    assert apart.sum() == (1 << n) - 32
    assert got[apart].tobytes() == want[apart].tobytes()
    assert not np.all(np.isfinite(got[~apart]))
