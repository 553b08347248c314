"""The merges' inversion in natural order (inv_small_kernel, inv_mult_kernel, inv_update_kernel) at
the edges of its tiles and steps, and its fallback to the pivoted inversion: the operators
S = -X^-1 S_RHS and T and the solution against the oracle, with the parity tests' tolerances.
"""
import numpy as np
import pytest

import oracle
import test_gpu_parity as gp
from oracle import mesh as omesh


def merge_case(ctx, N, level, lam, nodes):
    """Interface systems of order 4 N 2^j, j < level."""
    O, D, uo, ug = gp.solve_both(ctx, omesh.uniform(level), N, (-1, 1, -1, 1), lam=lam, check_ops=True, nodes=nodes)
    assert gp.rel(ug, uo) < gp.TOL_U
    return O


def largest_multiplier(X):
    """max |l| of Gauss-Jordan on X without row exchanges."""
    A, top = np.array(X), 0.0
    for j in range(len(A)):
        col = A[:, j] / A[j, j]
        col[j] = 0.0
        top = max(top, np.abs(col).max())
        row = A[j].copy()
        row[j] = 1.0
        row /= A[j, j]
        old = A[:, j].copy()
        A[:, j] = 0.0
        A -= np.outer(old, row)
        A[j] = row
    return top


# m = 16 .. 128 in registers (whole and partial tiles), then 160, 192, 256 (partial and whole steps), 512, 1024
@pytest.mark.gpu
@pytest.mark.parametrize("N,level", [(4, 1), (6, 1), (8, 1), (10, 2), (12, 2), (16, 1), (20, 2), (24, 2), (28, 1), (32, 2),
                                     (16, 4), (20, 4), (32, 4)])
def test_merge_inverse(ctx, N, level):
    gp.say(f"merges of uniform level {level}, N={N}")
    merge_case(ctx, N, level, -1.0, nodes=[0, 1])


@pytest.mark.gpu
def test_merge_inverse_falls_back(ctx):
    """lambda = 60 on [-1,1]^2: indefinite interface systems, one with a multiplier beyond the limit."""
    gp.say("merges with large multipliers in natural order")
    O = merge_case(ctx, 8, 3, 60.0, nodes=None)
    assert max(largest_multiplier(O.get(i, "X")) for i in range(5)) > 4.0


@pytest.mark.parametrize("N,level", [(6, 1), (10, 1)])
def test_emu_merge_inverse(emu_ctx, N, level):
    """m = 24 and 40."""
    merge_case(emu_ctx, N, level, -1.0, nodes=[0])


def test_emu_merge_inverse_falls_back(emu_ctx):
    O = merge_case(emu_ctx, 4, 1, 30.0, nodes=[0])
    assert largest_multiplier(O.get(0, "X")) > 4.0
