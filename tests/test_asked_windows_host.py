"""Windows that a caller asks for, on the host: the runs that every window keeps
leave the same number of its qubits to the blocks at every state size, so a block
list takes no more passes on a large state than on a small one (below 33 qubits,
from where complex128 passes carry less)."""
import numpy as np
import pytest

from menos_amd import hip as H


@pytest.mark.parametrize("window", [7, 8, 10])
@pytest.mark.parametrize("precision", [H.C128, H.C64])
def test_passes_do_not_grow_with_the_state(precision, window):
    rng = np.random.default_rng(3)

    def unitary(k):
        d = 1 << k
        return np.linalg.qr(rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))[0]

    blocks = [(unitary(1 + i % 2), rng.choice(20, 1 + i % 2, replace=False).tolist()) for i in range(60)]
    counts = {n: len(H.plan_passes(n, blocks, precision, window_qubits=window)) for n in (20, 23, 24, 25, 30, 32)}
    assert len(set(counts.values())) == 1, counts
