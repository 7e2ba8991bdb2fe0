"""GPU: the prefill GEMMs' wide blocks (up to 128 rows) against the narrow ones (up to 80), whose outputs the prefill
tests pin to the oracle: a row's products are summed in the same order either way, so the bits are the same."""
import numpy as np
import pytest
import torch

from oracle.bf16 import round_bf16
from tests.util import Layer, zipf_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gu,dn", [("IQ2_S", "IQ4_XS"), ("IQ3_S", "IQ3_S"), ("Q2_K", "Q3_K"), ("IQ4_XS", "Q2_K")])
@pytest.mark.parametrize("combine", ["matmul", "xla_sweep"])
def test_wide_blocks_equal_narrow(pkg, gpu, gu, dn, combine):
    """Experts of 1 .. 300 rows around the edges of both block sizes (16, 80, 81, 128, 129, 161, 257), zipf-skewed ones
    and one with no row."""
    rng = np.random.default_rng(97)
    E, D, I, limit = 8, 1024, 512, 10.0
    planes = {"gate": (gu, I, D), "up": (gu, I, D), "down": (dn, D, I)}
    L = {q: Layer(rng, q, E, D, I).tables(pkg) for q in {gu, dn}}
    tb = {m: L[q][m] for m, (q, _, _) in planes.items()}
    cases = [np.repeat(np.arange(7), n) for n in ([1, 16, 80, 81, 128, 129, 161], [300, 17, 257, 15, 33, 79, 97])]
    routings = [(c.astype(np.int32)[rng.permutation(len(c))][:, None], rng.random((len(c), 1), np.float32)) for c in cases]
    routings.append(zipf_routing(rng, 190, E, 3))
    for idx, w in routings:
        T = idx.shape[0]
        x = torch.from_numpy(round_bf16(rng.standard_normal((T, D)).astype(np.float32))).cuda().to(torch.bfloat16)
        it, wt = torch.from_numpy(np.ascontiguousarray(idx)).cuda(), torch.from_numpy(w).cuda()
        out = []
        for wide in (0, 1):
            with pkg.tuning(PF_WIDE=wide):
                out.append(pkg.moe_prefill(tb["gate"], tb["up"], tb["down"], x, it, wt, limit, combine=combine, chunk=4)[0])
        assert torch.isfinite(out[0]).all() and torch.equal(out[0], out[1]), (gu, dn, T)
