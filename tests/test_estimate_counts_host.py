"""What an estimate counts, on the host: the sampler's and the reductions'
launches by state size and term shape, and the device bytes of wide blocks'
tables and of small states' sampler tables."""
import pytest

from menos_amd import hip as H
from menos_amd import workloads as W

ENGINE = H.HipDenseEngine()


def _estimate(n, **kw):
    return ENGINE.estimate(W.random_circuit(n, 2, 3), **kw)


@pytest.mark.parametrize("n,launches", [(8, 1), (14, 1), (15, 7), (19, 7), (20, 8), (21, 7), (22, 8), (30, 8)])
def test_sampler_launches(n, launches):
    plain, shots = _estimate(n), _estimate(n, shots=100)
    assert shots.launches - plain.launches == launches


@pytest.mark.parametrize("n", [12, 25, 26, 33])
def test_reduction_launches(n):
    plain = _estimate(n).launches
    reach = 12 if n <= 25 else 11  # X bits of a tiled term, the low three counted
    tiled = [(1 << q, 1) for q in range(n)] + [(0, 3), (((1 << reach) - 1), 0)]
    assert _estimate(n, terms=tiled).launches - plain == 2
    if n > reach:
        wide = [((1 << (reach + 1)) - 1, 0)]
        assert _estimate(n, terms=wide).launches - plain == 2
        assert _estimate(n, terms=tiled + wide).launches - plain == 3


@pytest.mark.parametrize("precision,amp,width", [(H.C128, 16, 6), (H.C128, 16, 4), (H.C64, 8, 4)])
def test_wide_tables_are_counted(precision, amp, width):
    c = W.random_circuit(20, 12, 3)
    e = ENGINE.estimate(c, precision=precision, fusion=H.FUSE_WIDTH, fusion_width=width)
    one = amp << (2 * width)
    assert e.blocks > 16 and (amp << 20) + 16 * one <= e.device_bytes <= (amp << 20) + 16 * (one + 1024) + (1 << 17)
    # No wide pass takes complex64 blocks of five and six qubits.
    e = ENGINE.estimate(c, precision=H.C64, fusion=H.FUSE_WIDTH, fusion_width=1)
    assert e.device_bytes <= (8 << 20) + (1 << 17)


@pytest.mark.parametrize("n", [15, 20])
def test_small_sampler_tables_are_counted(n):
    """48 bytes for each 2^11 amplitudes, 16 a shot, beside the pass programs' 64 KiB."""
    e = _estimate(n, shots=1000)
    assert e.device_bytes >= (16 << n) + 48 * (1 << (n - 11)) + 16 * 1000 + (64 << 10)
