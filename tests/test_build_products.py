"""The build's S and T products through LDS tiles (tree_gemm_lds_kernel) at the orders where its three tile
shapes begin, and with the merges beside them that keep the register tiles: the operators and
the solution against the oracle, with the parity tests' tolerances.
"""
import pytest

import test_gpu_parity as gp
from test_merge_inverse import merge_case


# n = 32 (1 x 4 and 4 x 1 waves); 16, 32, 64 (2 x 2); 24, 48 (register tiles), 96 (1 x 4, 4 x 1, several tiles); 8 .. 128
@pytest.mark.gpu
@pytest.mark.parametrize("N,level", [(32, 1), (16, 3), (24, 3), (8, 5)])
def test_build_products(ctx, N, level):
    gp.say(f"build products of uniform level {level}, N={N}")
    merge_case(ctx, N, level, -1.0, nodes=[0, 1, 2])


def test_emu_build_products(emu_ctx):
    """n = 32: one merge, m = 128."""
    merge_case(emu_ctx, 32, 1, -1.0, nodes=[0])
