"""GPU: a prefill call gives the same bits every time where the launches split some of many equal blocks along K."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype,E,D", [("CB3", 270, 5120), ("IQ4_XS", 392, 2048)])
def test_repeated_calls_equal(pkg, gpu, qtype, E, D):
    """One block of one row per expert, so every block ties with every other in the launch order, over several of the
    plan's wavefronts.  I 256 gives the gate/up launch 2 (CB3) or 4 workgroups per block, 540 or 1568 tasks: a last round
    of 28 or 32 tasks on 512 or 768 slots, whose 14 or 8 blocks are each summed in 4 pieces."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(31)
    I = 256
    table = {"CB3": pkg.random_cb3_table,
             "IQ4_XS": lambda *a: pkg.resident.random_iq4xs_table(*a, scale=2e-5)}[qtype]
    gate, up, down = (table(E, R, K, gen) for R, K in ((I, D), (I, D), (D, I)))
    x = torch.randn((E, D), device="cuda", generator=gen).to(torch.bfloat16)
    idx = torch.from_numpy(np.random.default_rng(3).permutation(E).astype(np.int32)[:, None]).cuda()
    w = torch.ones((E, 1), device="cuda")
    first = pkg.moe_prefill(gate, up, down, x, idx, w, 10.0)[0]
    assert torch.isfinite(first).all()
    for _ in range(40):
        assert torch.equal(pkg.moe_prefill(gate, up, down, x, idx, w, 10.0)[0], first)


def test_more_blocks_than_threads(pkg, gpu):
    """1200 blocks, more than the plan kernel has threads (1024): 1023 experts of one row and one of 14,160 (177 blocks).
    Every token's row within rel-L2 1e-3 (the prefill tests' bound) of the same token in calls of fewer blocks."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(32)
    E, D, I = 1024, 256, 256
    gate, up, down = (pkg.random_cb3_table(E, R, K, gen) for R, K in ((I, D), (I, D), (D, I)))
    ids = np.concatenate([np.arange(E - 1), np.full(177 * 80, E - 1)]).astype(np.int32)
    idx = torch.from_numpy(np.random.default_rng(4).permutation(ids)[:, None]).cuda()
    T = len(ids)
    x = torch.randn((T, D), device="cuda", generator=gen).to(torch.bfloat16)
    w = torch.ones((T, 1), device="cuda")
    out = pkg.moe_prefill(gate, up, down, x, idx, w, 10.0)[0]
    step = T // 4
    part = torch.cat([pkg.moe_prefill(gate, up, down, x[i:i + step], idx[i:i + step], w[i:i + step], 10.0)[0]
                      for i in range(0, T, step)])
    assert torch.linalg.norm(out - part) <= 1e-3 * torch.linalg.norm(part)
    assert torch.equal(pkg.moe_prefill(gate, up, down, x, idx, w, 10.0)[0], out)
