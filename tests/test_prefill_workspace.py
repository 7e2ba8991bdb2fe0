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


@pytest.mark.parametrize("gate,down", [("IQ3_S", "IQ3_S"), ("IQ2_S", "IQ4_XS"), ("CB3", "CB3"), ("CB3", "IQ4_XS")])
@pytest.mark.parametrize("E,k,shared", [(64, 8, -1), (65, 8, 64), (32, 6, -1), (1, 1, -1), (3, 2, 2), (512, 8, -1)])
@pytest.mark.parametrize("combine", [0, 2])
def test_sizes_grow_with_the_piece(pkg, gate, down, E, k, shared, combine):
    """A workspace sized for the longest piece serves every shorter one, wide plans (which pad an expert's rows to more)
    or narrow: around the edges between them, the limits of a plan's 32-bit offsets included (512 experts)."""
    L, (g, d) = pkg._lib.lib(), _pair(pkg, gate, down, E, 2048, 6144)
    kk = k + (shared >= 0)
    edges = [r * E // kk + o for r in (80, 128, 160, 240, 256) for o in range(-3, 4)]
    sizes = [(t, L.mi_moe_prefill_form_workspace(g, d, t, k, shared, combine))
             for t in sorted({t for t in edges + list(range(1, 18000, 37)) if t > 0})]
    sizes = [(t, n) for t, n in sizes if n or t < 3000]
    assert len(sizes) > 50 and all(n > 0 for _, n in sizes)
    for (t0, a), (t1, b) in zip(sizes, sizes[1:]):
        assert a <= b, (t0, a, t1, b)


@pytest.mark.parametrize("T,tm", [(512, 80), (1024, 128), (1999, 128)])
def test_size_is_rows_and_piece_sums(pkg, T, tm):
    """The padded rows of h and y, the plan's arrays and the split tasks' piece sums: 40 KB on each of 3 slots per CU or
    80 KB (CB3) on 2 in narrow plans, 64 KB on 2 in wide ones; 256 CUs."""
    L, E, k, I, D = pkg._lib.lib(), 64, 8, 2048, 6144
    G = -(-T * k // tm) + E
    need = G * tm * 2 * (I + D) + 4 * (3 * G + 2 * G * tm + T * k) + (512 * 80 if tm == 80 else 512 * 64) * 1024
    got = L.mi_moe_prefill_workspace(*_pair(pkg, "IQ3_S", "IQ3_S", E, I, D), T, k, -1)
    assert need <= got < need + (1 << 14)
