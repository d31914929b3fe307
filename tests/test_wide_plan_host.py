"""Which passes the plan makes of blocks of three and more qubits, on the host:
they share tiles up to the largest state whose tiles fit one launch (34 qubits);
larger states keep one pass a block (the per-group kernel's)."""
import numpy as np
import pytest

from menos_amd import hip as H


def _blocks(widths):
    rng = np.random.default_rng(4)
    out = []
    for i, k in enumerate(widths):
        m = rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k))
        out.append((np.linalg.qr(m)[0], [4 + i + j for j in range(k)]))
    return out


@pytest.mark.parametrize("precision,n,passes", [
    (H.C64, 12, 1), (H.C64, 34, 1), (H.C64, 35, 3), (H.C64, 40, 3),
    (H.C128, 12, 1), (H.C128, 34, 1), (H.C128, 35, 3),
])
def test_blocks_share_a_tile_while_its_launch_fits(precision, n, passes):
    blocks = _blocks([3, 3, 4])
    assert len(H.plan_passes(n, blocks, precision)) == passes
