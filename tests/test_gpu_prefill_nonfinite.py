"""GPU: an infinite block scale of a K-quant expert reaches the prefill's output as the reference's dequant has it."""
import numpy as np
import pytest
import torch

from oracle import moe as omoe
from oracle.bf16 import rel_l2, round_bf16
from tests.util import Layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", ["Q2_K", "Q3_K"])
@pytest.mark.parametrize("wide", [0, 1])
def test_infinite_scale_of_zero_quants(pkg, gpu, qtype, wide):
    """A down block with d = inf whose values are all 0 (Q3_K: 2-bit value 0 and high bit set, 4 - 4): inf * 0, so its
    row of the output is NaN and every other one is finite."""
    rng = np.random.default_rng(17)
    E, D, I, T = 2, 512, 512, 40
    L = Layer(rng, qtype, E, D, I)
    blk = L.raw["down"][:, 5, 1]                       # row 5's second block of every expert
    if qtype == "Q2_K":
        blk[:, 0:16], blk[:, 16:80], blk[:, 80:82] = 0x11, 0, (0x00, 0x7C)
    else:
        blk[:, 0:32], blk[:, 32:96], blk[:, 108:110] = 0xFF, 0, (0x00, 0x7C)
    tbs = L.tables(pkg)
    idx = rng.integers(0, E, (T, 1)).astype(np.int32)
    w = np.ones((T, 1), np.float32)
    x = round_bf16(rng.standard_normal((T, D)).astype(np.float32))
    with np.errstate(invalid="ignore"):
        want = omoe.prefill_apply(L.deq, x, idx, w, 10.0, E, combine="matmul")
    assert np.isnan(want[:, 5]).all() and np.isfinite(np.delete(want, 5, axis=1)).all()
    print("non-finite %s wide=%d" % (qtype, wide), flush=True)
    with pkg.tuning(PF_WIDE=wide):
        got = pkg.moe_prefill(tbs["gate"], tbs["up"], tbs["down"], torch.from_numpy(x).cuda().to(torch.bfloat16),
                              torch.from_numpy(idx).cuda(), torch.from_numpy(w).cuda(), 10.0)[0].cpu().numpy()
    assert np.isnan(got[:, 5]).all()
    assert rel_l2(np.delete(got, 5, axis=1), np.delete(want, 5, axis=1)) < 1e-3
