"""CPU: the prefill workspace sizes (no launch)."""
import ctypes

import pytest


def _pair(pkg, gate, down, E, I, D):
    """(gate, down) tables of E experts; their planes are never read."""
    out = []
    for qt, R, K in ((gate, I, D), (down, D, I)):
        t = pkg._lib.MiTable()
        t.qtype, t.rows, t.cols, t.n_experts = pkg._lib.QTYPES[qt], R, K, E
        out.append(ctypes.byref(t))
    return out


@pytest.mark.parametrize("E", [0, -1])
@pytest.mark.parametrize("qtype", ["CB3", "IQ3_S"])
def test_no_experts_has_no_size(pkg, qtype, E):
    assert pkg._lib.lib().mi_moe_prefill_workspace(*_pair(pkg, qtype, qtype, E, 256, 512), 8, 2, -1) == 0
