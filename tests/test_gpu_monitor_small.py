"""The execution monitor of states that are one window: it is asked between
passes of bounded arithmetic, a run can be abandoned there, and the amplitudes
are those of a run without a monitor."""
import pytest

from menos_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [10, 11, 12, 13])
def test_small_states_keep_their_boundaries(hip, n, precision):
    eng = hip.HipDenseEngine()
    c = W.random_circuit(n, 24, 9)
    seen = []
    r = eng.execute(c, precision=precision, monitor=seen.append, targets=[], width=0)
    plain = eng.execute(c, precision=precision, targets=[], width=0)
    assert seen == list(range(1, r.num_passes + 1)) and plain.num_passes == 1
    # 24 layers of U3, at least 14 operations an amplitude each, in passes of at
    # most 160: more than one pass a layer and ten qubits, half of that asked.
    assert r.num_passes >= 24 * n * 14 // 160 // 2
    assert r.statevector.tobytes() == plain.statevector.tobytes()


def test_a_small_run_is_abandoned(hip):
    class Abandon(Exception):
        pass

    def stop(crossed):
        if crossed == 2:
            raise Abandon

    eng = hip.HipDenseEngine()
    c = W.random_circuit(12, 40, 4)
    with pytest.raises(Abandon):
        eng.execute(c, monitor=stop, statevector=False, targets=[], width=0)
    assert eng.execute(c, targets=[], width=0).statevector is not None
