"""GPU parity of the CB3 prefill on both sides of the row length from which its launches split tasks along K."""
import numpy as np
import pytest
import torch

from oracle import moe as omoe
from oracle.bf16 import rel_l2, round_bf16
from tests.util import Layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [4352, 4608])
def test_row_length_of_the_split(pkg, gpu, D):
    """7 super tiles of 640 columns (whole tasks) and 8 (split; the last one a fifth of a super tile): within the prefill
    tests' rel-L2 1e-3 of the oracle."""
    rng = np.random.default_rng(D)
    E, I, T = 2, 256, 90
    L = Layer(rng, "CB3", E, D, I)
    tbs = L.tables(pkg)
    idx, w = rng.integers(0, E, (T, 1)).astype(np.int32), rng.random((T, 1)).astype(np.float32)
    x = round_bf16(rng.standard_normal((T, D)).astype(np.float32))
    got = pkg.moe_prefill(tbs["gate"], tbs["up"], tbs["down"], torch.from_numpy(x).cuda().to(torch.bfloat16),
                          torch.from_numpy(idx).cuda(), torch.from_numpy(w).cuda(), 10.0)[0].cpu().numpy()
    assert rel_l2(got, omoe.prefill_apply(L.deq, x, idx, w, 10.0, E, combine="matmul")) < 1e-3
