"""GPU: the prefill GEMMs' wide blocks (up to 128 rows) against the narrow ones (up to 80), whose outputs the prefill
tests pin to the oracle, and against the oracle where the two plans split other tasks along K (whole tasks and pieces sum
a row's products in another order, so the bits may then differ)."""
import numpy as np
import pytest
import torch

from oracle import moe as omoe
from oracle.bf16 import rel_l2, round_bf16
from tests.util import Layer, zipf_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gu,dn", [("IQ2_S", "IQ4_XS"), ("IQ3_S", "IQ3_S"), ("Q2_K", "Q3_K"), ("IQ4_XS", "Q2_K")])
@pytest.mark.parametrize("combine", ["matmul", "xla_sweep"])
def test_wide_blocks_equal_narrow(pkg, gpu, gu, dn, combine):
    """Experts of 1 .. 300 rows around the edges of both block sizes (16, 80, 81, 128, 129, 161, 257), zipf-skewed ones
    and one with no row.  The same bits: either plan's launches are one partial round, whose gate/up tasks all run as two
    pieces (1024 columns are two super tiles) and whose down tasks (one super tile) run whole."""
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


@pytest.mark.parametrize("gu,dn", [("IQ2_S", "IQ4_XS"), ("IQ3_S", "Q2_K"), ("Q3_K", "IQ3_S")])
def test_wide_blocks_whole_and_split(pkg, gpu, gu, dn):
    """46 wide blocks of 90 .. 110 rows at D = I = 1536 (3 super tiles): gate/up 1104 tasks and down 552 on 512 slots, whole
    rounds and a last one of 4 blocks in 3 pieces each.  Within the prefill tests' rel-L2 1e-3 of the oracle.  The 46
    experts are 4 different ones in turn."""
    rng = np.random.default_rng(46)
    E, n, D, I = 46, 4, 1536, 1536
    L = Layer(rng, gu, n, D, I, down_qtype=dn)
    tb = {}
    for m, (R, K) in L.shapes.items():
        planes = {key: np.concatenate([a.reshape(n, -1, a.shape[-1])[e % n] for e in range(E)])
                  for key, a in L.planes(m, pkg.formats).items()}
        tb[m] = pkg.ExpertTable(L.qtypes[m], pkg.to_device_planes(planes), R, K)
    rows = np.concatenate([100 + rng.permutation(21) - 10, 100 + rng.permutation(21) - 10, np.full(4, 100)])
    idx = rng.permutation(np.repeat(np.arange(E), rows)).astype(np.int32)[:, None]
    T = len(idx)
    w = rng.random((T, 1)).astype(np.float32)
    x = round_bf16(rng.standard_normal((T, D)).astype(np.float32))
    print("wide, whole and split", gu, dn, T, flush=True)
    got = pkg.moe_prefill(tb["gate"], tb["up"], tb["down"], torch.from_numpy(x).cuda().to(torch.bfloat16),
                          torch.from_numpy(idx).cuda(), torch.from_numpy(w).cuda(), 10.0)[0].cpu().numpy()
    want = omoe.prefill_apply(lambda m, e: L.deq(m, e % n), x, idx, w, 10.0, E, combine="matmul")
    assert rel_l2(got, want) < 1e-3
