"""Windows that a caller asks for, at the sizes where their runs and wavefronts
change (13 | 14, 22 | 23, 24 and 25 qubits): the same state as with the default
window, bit for bit at complex128 (whose last pass leaves no -0), equal at
complex64 (the operations on an amplitude do not depend on the window)."""
import numpy as np
import pytest

from circuits import random_unitary

pytestmark = pytest.mark.gpu

CX = np.eye(4)[[0, 3, 2, 1]].astype(np.complex128)


@pytest.mark.parametrize("n", [10, 13, 14, 22, 23, 24, 25])
@pytest.mark.parametrize("precision", [0, 1])
def test_asked_windows_equal_the_default(hip, precision, n):
    rng = np.random.default_rng(n)
    blocks = []
    for _ in range(40):
        a, b = (int(q) for q in rng.permutation(n)[:2])
        kind = int(rng.integers(0, 4))
        if kind == 0:
            blocks.append((random_unitary(1, rng), [a]))
        elif kind == 1:
            blocks.append((random_unitary(2, rng), [a, b]))
        elif kind == 2:
            blocks.append((CX, [a, b]))
        else:
            blocks.append((np.diag(np.exp(1j * rng.uniform(-3, 3, 4))), [a, b]))
    want, got = hip.DeviceState(n, precision), hip.DeviceState(n, precision)
    want.init()
    want.apply_blocks(blocks)
    for window in (7, 8, 10):
        got.init()
        got.apply_blocks(blocks, window_qubits=window)
        assert got.max_abs_diff(want) == 0.0, window
        if precision == 0:
            assert got.digest() == want.digest(), window
    want.free()
    got.free()
