"""CPU: host validation of mi_mlp_many (no launch: every call here is refused) and the sizes its workspace function
takes and refuses."""
import ctypes

import pytest
import torch


def test_mlp_many_validation(pkg):
    L, lib = pkg._lib.lib(), pkg._lib
    P = ctypes.c_void_p

    def call(B=64, D=512, I=256, gf=lib.MI_I8_COL_SCALES, df=lib.MI_I8_COL_SCALES, gw=P(0x1000), gs=P(0x2000), limit=7.0,
             x=P(0x10000), y=P(0x20000), wsb=1 << 30):
        return L.mi_mlp_many(x, B, D, I, gw, gs, P(0x3000), P(0x4000), gf, P(0x5000), P(0x6000), df, ctypes.c_float(limit),
                             y, None, P(0x100000), wsb, None)

    assert call(B=0) == 4 and call(B=(1 << 14) + 1) == 4                                # MI_ERR_TOKENS
    assert call(D=640) == 3 and call(I=300) == 3                                        # MI_ERR_SHAPE
    assert call(limit=0.0) == 8 and call(gw=P(0x1008)) == 8 and call(x=P(0x10002)) == 8  # MI_ERR_ARG
    assert call(gf=lib.MI_I8_COL_AFTER) == 8 and call(gf=lib.MI_W_BF16 | lib.MI_I8_TILED) == 8
    assert call(gf=lib.MI_I8_ROW_SCALES, gs=P(0x2004)) == 8
    assert call(gw=None) == 1 and call(gs=None) == 1 and call(y=None) == 1              # MI_ERR_NULL
    assert call(wsb=16) == 5                                                            # MI_ERR_WORKSPACE
    assert L.mi_mlp_many_workspace(512, 6144, 2048) > 0
    for bad in ((0, 512, 256), (64, 500, 256), (64, 512, 100), (64, 131072, 256), (64, 65536, 32768)):
        assert L.mi_mlp_many_workspace(*bad) == 0, bad


def test_mlp_many_workspace_serves_fewer_tokens(pkg):
    """A call of more than 4096 tokens runs 4096 at a time and its last piece in the same workspace: no piece needs
    more than the size of the largest."""
    size = pkg._lib.lib().mi_mlp_many_workspace
    for D, I in ((6144, 2048), (4096, 1536), (3072, 1280), (2048, 768), (256, 256), (65536, 256)):
        sizes = [size(b, D, I) for b in range(1, 4097)]
        assert all(a <= b for a, b in zip(sizes, sizes[1:])), (D, I)


@pytest.mark.parametrize("B", [8, 33, 5000])
@pytest.mark.parametrize("gu,down", [(2, 2), (1, 2), (2, 1), (3, 3), (1, 3), (7, 1)])
def test_int8_mlp_refuses_other_scale_forms(pkg, B, gu, down):
    """Scale forms that an MLP does not take (the lm_head's, and the code that mi_mlp_many has for bf16 weights) are a
    ValueError before any launch, for every token count."""
    q, s = torch.zeros((256, 256), dtype=torch.int8), torch.ones(256)
    with pytest.raises(ValueError):
        pkg.int8_mlp(torch.zeros((B, 256), dtype=torch.bfloat16), (q, s, gu), (q, s, gu), (q, s, down), 7.0)
