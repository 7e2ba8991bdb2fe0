"""CPU: the workspace sizes of the streaming projections and MLPs never fall as the batch grows, so one workspace sized for
the largest batch serves every batch (fewer tokens can have more column splits, each with its own partials)."""
import ctypes

import pytest


@pytest.mark.parametrize("n_in", [256, 1024, 1536, 2048, 4096, 6144, 8192])
def test_sizes_grow_with_the_batch(pkg, n_in):
    L = pkg._lib.lib()

    def check(size, *what):
        sizes = [size(b) for b in range(1, 33)]
        assert sizes[0] > 0 and all(a <= b for a, b in zip(sizes, sizes[1:])), what

    for n_out in (16, 256, 768, 2048, 4096, 6144, 151552):
        check(lambda b: L.mi_bf16_project_workspace(b, n_in, n_out), "bf16", n_out)
        for axis in (0, 1, 2):
            check(lambda b: L.mi_int8_project_workspace(b, n_in, n_out, axis), "int8", n_out, axis)
        if n_out % 256 == 0:
            check(lambda b: L.mi_bf16_mlp_workspace(b, n_in, n_out), "bf16 mlp", n_out)
            for gu, dn in ((0, 0), (0, 1), (1, 0), (1, 1)):
                check(lambda b: L.mi_int8_mlp_workspace(b, n_in, n_out, gu, dn), "int8 mlp", n_out, gu, dn)
    for outs in ((n_in,) * 3, (n_in, n_in // 2, n_in // 2), (n_in, 128, 128)):
        arr = (ctypes.c_int32 * 3)(*outs)
        check(lambda b: L.mi_int8_project_many_workspace(b, n_in, arr, 3, 1), "many", outs)
