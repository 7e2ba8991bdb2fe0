"""GPU parity of mlp_partial for more tokens than one streaming call takes (mi_mlp_many: dense GEMMs on the matrix
cores) against the oracle and against the 32-token calls: every weight form, token counts around the tile edges, and
forced column splits."""
import numpy as np
import pytest
import torch

from oracle import int8 as oi8
from oracle.bf16 import rel_l2, round_bf16

pytestmark = pytest.mark.gpu


def _leaves(pkg, rng, form, D, I):
    """(leaves for mlp_partial, the oracle's weights) of one form."""
    shapes = ((D, I), (D, I), (I, D))
    if form == "bf16":
        W = [round_bf16(rng.standard_normal(s).astype(np.float32) * 0.05) for s in shapes]
        return [pkg.bf16_leaf(torch.from_numpy(w).cuda().to(torch.bfloat16)) for w in W], W
    axes = {"col": (1, 1), "tiled": (1, 1), "row": (0, 0), "col_row": (1, 0)}[form]
    ax = (axes[0], axes[0], axes[1])
    W = [oi8.quantize_array(rng.standard_normal(s).astype(np.float32) * 0.05, a) for s, a in zip(shapes, ax)]
    leaves = [pkg.resident.int8_leaf({"q": q, "s": s}) for q, s in W]
    if form == "tiled":
        leaves = [(pkg.int8_tile(q), s, a) for q, s, a in leaves]
    return leaves, W


@pytest.mark.parametrize("form", ["bf16", "col", "tiled", "row", "col_row"])
@pytest.mark.parametrize("B,D,I", [(33, 512, 256), (64, 256, 512), (65, 768, 256), (128, 512, 768), (129, 1024, 256),
                                   (300, 2048, 768)])
def test_mlp_many(pkg, gpu, form, B, D, I):
    """The f32 output within rel-L2 1e-4 of the oracle (an element of g, u or h next to a bf16 rounding boundary may
    round the other way, as in the streaming calls' tests) and the bf16 output that f32 output rounded once."""
    rng = np.random.default_rng(B * 31 + D + I)
    leaves, W = _leaves(pkg, rng, form, D, I)
    x = round_bf16(rng.standard_normal((B, D)).astype(np.float32) * 2)
    xt = torch.from_numpy(x).cuda().to(torch.bfloat16)
    print("mlp_many %s B=%d D=%d I=%d" % (form, B, D, I), flush=True)
    call = pkg.bf16_mlp if form == "bf16" else pkg.int8_mlp
    yb, yf = call(xt, *leaves, 7.0, want_f32=True)
    want = oi8.mlp_partial_f32(x, *W, 7.0)
    assert rel_l2(yf.cpu().numpy(), want) < 1e-4
    assert np.array_equal(yb.float().cpu().numpy(), round_bf16(yf.cpu().numpy()))
    assert torch.equal(pkg.mlp_partial(dict(zip(("gate", "up", "down"), leaves)), xt, 7.0), yb)
    for s1, s2, nt in ((1, 1, 2), (1, 1, 4), (3, 2, 2), (2, 3, 4)):     # splits that do not divide the steps too
        with pkg.tuning(DG_S1=s1, DG_S2=s2, DG_NT=nt):
            ys, fs = call(xt, *leaves, 7.0, want_f32=True)
        assert rel_l2(fs.cpu().numpy(), want) < 1e-4, (s1, s2, nt)


def test_mlp_many_other_routes(pkg, gpu):
    """What the dense GEMMs do not take keeps the 32-token calls' results: a kept workspace of their size (whose
    counters stay zero); a large kept workspace goes to the GEMMs behind its counters."""
    rng = np.random.default_rng(5)
    B, D, I = 250, 512, 256
    leaves, W = _leaves(pkg, rng, "col", D, I)
    x = round_bf16(rng.standard_normal((B, D)).astype(np.float32))
    xt = torch.from_numpy(x).cuda().to(torch.bfloat16)
    want = oi8.mlp_partial_f32(x, *W, 7.0)
    L = pkg._lib.lib()
    small = torch.zeros(L.mi_int8_mlp_workspace(32, D, I, 1, 1), dtype=torch.uint8, device="cuda")
    big = torch.zeros(pkg._lib.I8_CTR_BYTES + L.mi_mlp_many_workspace(B, D, I), dtype=torch.uint8, device="cuda")
    assert small.numel() < big.numel()
    for ws in (small, big):
        yf = pkg.int8_mlp(xt, *leaves, 7.0, want_f32=True, workspace=ws)[1]
        assert rel_l2(yf.cpu().numpy(), want) < 1e-4
        assert int(ws[:pkg._lib.I8_CTR_BYTES].count_nonzero()) == 0


def test_mlp_many_last_piece(pkg, gpu):
    """More than the 4096 tokens of one piece, the last piece of a size whose split sums need more scratch than the
    first's: the bits of the pieces by themselves, without and with a kept workspace sized for the first piece."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    B, D, I = 4096 + 512, 2048, 768
    w = [torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) * 0.02 for s in ((D, I), (D, I), (I, D))]
    leaves = [pkg.bf16_leaf(v) for v in w]
    x = torch.randn((B, D), device="cuda", generator=gen).to(torch.bfloat16)
    kept = torch.zeros(pkg._lib.I8_CTR_BYTES + pkg._lib.lib().mi_mlp_many_workspace(4096, D, I), dtype=torch.uint8,
                       device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        got = [pkg.bf16_mlp(x, *leaves, 7.0, workspace=ws) for ws in (None, kept)]
        want = torch.cat([pkg.bf16_mlp(x[:4096], *leaves, 7.0), pkg.bf16_mlp(x[4096:], *leaves, 7.0)])
        torch.cuda.synchronize()
    assert torch.equal(got[0], want) and torch.equal(got[1], want)


def test_mlp_many_and_route_captured(pkg, gpu):
    """A captured MLP of 64 tokens and a captured router call, replayed between eager calls of more tokens on the capture
    stream: every replay gives the eager bits."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(12)
    D, I, E, k = 1024, 512, 64, 8
    w = [torch.randn(s, device="cuda", generator=gen).to(torch.bfloat16) * 0.02 for s in ((D, I), (D, I), (I, D))]
    leaves = [pkg.bf16_leaf(v) for v in w]
    rw = torch.randn((D, E), device="cuda", generator=gen) / 32
    x = torch.randn((64, D), device="cuda", generator=gen).to(torch.bfloat16)
    more = torch.randn((700, D), device="cuda", generator=gen).to(torch.bfloat16)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        want = (pkg.bf16_mlp(x, *leaves, 7.0), *pkg.route(x, rw, None, k))
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            got = (pkg.bf16_mlp(x, *leaves, 7.0), *pkg.route(x, rw, None, k))
        for _ in range(4):
            eager = pkg.bf16_mlp(more, *leaves, 7.0), pkg.route(more, rw, None, k)
            for t in got:
                t.zero_()
            graph.replay()
            stream.synchronize()
            assert all(torch.equal(a, b) for a, b in zip(got, want))
            del eager
