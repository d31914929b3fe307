"""A captured batch whose parameters take entries to exactly 0 and back: how a
block runs depends on its matrix (a real one leaves its zero parts out), and the
graph takes parameters that need a narrower form, or a wider one, as long as the
block keeps its class. Terms equal the batch entry point's bit for bit; what
changes a block's class is refused and the graph keeps its parameters."""
import math

import numpy as np
import pytest

from menos_amd import workloads as W

pytestmark = pytest.mark.gpu


def _same(a, b):
    return all(x.tobytes() == y.tobytes() for x, y in zip(a, b))


def _ansatz(n, depth, rng, rz):
    """RY at random angles; rz(layer, qubit, random angle) for the others."""
    angles = rng.uniform(0.1, math.pi - 0.1, (depth, 2, n))
    for layer in range(depth):
        for q in range(n):
            angles[layer, 1, q] = rz(layer, q, angles[layer, 1, q])
    return W.FlatAnsatz(n, depth, angles.reshape(-1))


@pytest.mark.parametrize("fusion", [1, 3])
@pytest.mark.parametrize("precision", [0, 1])
def test_rotations_by_zero_and_back(hip, precision, fusion):
    sizes, depth = (12, 14, 16), 3
    terms = [W.random_paulis(n, 6, n) for n in sizes]

    def circuits(seed, rz):
        rng = np.random.default_rng(seed)
        return [_ansatz(n, depth, rng, rz) for n in sizes]

    def full(layer, q, a):
        return a

    def flat(layer, q, a):  # every RZ by 0 but qubit 0's
        return a if q == 0 else 0.0

    def one(layer, q, a):
        return 0.0 if q == 3 and layer == depth - 1 else a

    for first, rest in ((full, (one, flat, full, one)), (flat, (full, flat, one))):
        with hip.BatchGraph(circuits(1, first), terms, precision=precision, fusion=fusion) as g:
            for step, rz in enumerate((first,) + rest):
                cs = circuits(10 + step, rz)
                g.update(cs)
                want = hip.batch_execute(cs, terms, precision=precision, fusion=fusion).expectation
                for _ in range(2):
                    got, _ = g.run()
                    assert _same(got, want), (first.__name__, step, rz.__name__)


CLEAR, SET = np.diag([1, 0]), np.diag([0, 1])
FLIP = np.array([[0, 1], [1, 0]])


def _rotation(a, phase=0.0):
    return np.array([[math.cos(a), -math.sin(a)], [math.sin(a), math.cos(a)]]) * np.exp(1j * phase)


def _controlled(clear, set_, control):
    """Operand `control` (0: the index's low bit) chooses the other's block."""
    return np.kron(clear, CLEAR) + np.kron(set_, SET) if control == 0 else np.kron(CLEAR, clear) + np.kron(SET, set_)


SWAP = np.eye(4)[[0, 2, 1, 3]]
CLASSES = {
    # One qubit, first entry real: a flip, real, its other entries complex.
    "first real": [FLIP, _rotation(0.7), np.array([[0.6, 0.8j], [0.8j, 0.6]])],
    "first complex": [_rotation(0.4, 0.3), _rotation(1.1, -0.9)],
    # Controlled by operand 1: a flip where it is clear, rows exchanged (real,
    # complex), columns exchanged, any pair.
    "control 1": [_controlled(FLIP, np.eye(2), 1), _controlled(_rotation(0.5), FLIP @ _rotation(0.5), 1),
                  _controlled(_rotation(0.5, 0.2), FLIP @ _rotation(0.5, 0.2), 1),
                  _controlled(_rotation(0.5, 0.2), _rotation(0.5, 0.2) @ FLIP, 1),
                  _controlled(_rotation(0.5, 0.2), _rotation(1.3, 0.8), 1)],
    "control 0": [_controlled(_rotation(0.3), _rotation(0.9), 0), _controlled(_rotation(0.3, 1.0), _rotation(0.3, 1.0) @ FLIP, 0)],
    "full": [SWAP, np.kron(_rotation(0.4), _rotation(0.8)), np.kron(_rotation(0.4, 0.1), _rotation(0.8, 0.6)),
             np.eye(4)[[3, 2, 1, 0]]],
}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", sorted(CLASSES))
def test_a_unitary_moves_within_its_class_only(hip, precision, name):
    n = 14
    rng = np.random.default_rng(8)
    paulis = [W.random_paulis(n, 8, 3)]

    def circuit(m):
        c = W.Circuit(n)
        for q in range(n):
            c.append(W.H, (q,))
            c.append(W.T, (q,))
        qs = (2, 11) if len(m) == 4 else (5,)
        params = np.ascontiguousarray(m, np.complex128).reshape(-1).view(np.float64)
        c.append(W.UNITARY, qs, tuple(params))
        for q in range(0, n - 1, 2):
            c.append(W.CX, (q, q + 1))
        for q in range(n):
            c.append(W.RX, (q,), (0.1 + q,))
        return c

    mine = CLASSES[name]
    order = list(range(len(mine))) + rng.permutation(len(mine)).tolist()
    for first in (0, len(mine) - 1):
        # No fusion: the unitary stays a block of its own.
        with hip.BatchGraph([circuit(mine[first])], paulis, precision=precision, fusion=0) as g:
            want = None
            for k in order:
                g.update([circuit(mine[k])])
                want = hip.batch_execute([circuit(mine[k])], paulis, precision=precision, fusion=0).expectation
                got, _ = g.run()
                assert _same(got, want), (first, k)
            for other, theirs in CLASSES.items():
                if other == name or len(theirs[0]) != len(mine[0]):
                    continue
                for m in theirs:
                    with pytest.raises(hip.HipError, match="pass program"):
                        g.update([circuit(m)])
            with pytest.raises(hip.HipError, match="pass program"):
                g.update([circuit(np.diag([1, -1] if len(mine[0]) == 2 else [1, 1, 1, -1]))])
            got, _ = g.run()
            assert _same(got, want)
