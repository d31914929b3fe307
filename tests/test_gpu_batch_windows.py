"""Batches whose windows are few, and batches that mix states of one window with
larger ones: their passes are laid out otherwise than those of a large batch or
of one state, with the same amplitudes bit for bit."""
import numpy as np
import pytest

from menos_amd import workloads as W

pytestmark = pytest.mark.gpu


def _circuits(sizes, seed):
    rng = np.random.default_rng(seed)
    return [W.FlatAnsatz(n, d, rng.uniform(-3, 3, 2 * n * d)) for n, d in sizes]


# Windows of 13 qubits: 2, 254, 256 (as many as CUs), and mixed states.
SIZES = {
    "one of 14": [(14, 5)],
    "127 of 14": [(14, 2)] * 127,
    "128 of 14": [(14, 2)] * 128,
    "two of 20": [(20, 2)] * 2,
    "13 beside 15": [(13, 12), (15, 3), (10, 12), (11, 4), (12, 9)],
    "13 alone": [(13, 12), (10, 12), (12, 9)],
}


@pytest.mark.parametrize("fusion", [0, 1, 3])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(SIZES))
def test_states_equal_the_engine(hip, name, precision, fusion):
    circuits = _circuits(SIZES[name], 7)
    got = hip.batch_execute(circuits, [[] for _ in circuits], precision=precision, fusion=fusion, statevectors=True)
    engine = hip.HipDenseEngine()
    for i in sorted({0, 1, len(circuits) // 2, len(circuits) - 1} & set(range(len(circuits)))):
        want = engine.execute(circuits[i], precision=precision, fusion=fusion, targets=[], width=0).statevector
        assert got.statevectors[i].tobytes() == want.tobytes(), i
