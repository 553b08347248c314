"""Variable-coefficient leaf solves of the sides without a kernel of their own (bt_solve_kernel): eight leaves
times all right-hand sides of a batch after one another, from N = 8 on; leaf counts that leave the last eight
partly empty.  Every operation against the oracle, every column of a batch bit for bit as alone."""
import numpy as np
import pytest

import test_patches as tp


def general_case(ctx, N, P, nrhs):
    from ellipticforest_amd import _lib
    rng = np.random.default_rng(N + P)
    bounds = tp.random_bounds(rng, P)
    cell = tp.variable_cells(bounds, N)
    pv = _lib.Patches(ctx, bounds, N, solver_type=_lib.EF_SOLVER_FIVE_POINT, cell=cell)
    assert pv.variable and not pv.packed
    tp.check_against_oracle(pv, bounds, N, rng, nrhs=nrhs, coeffs=cell, dtn=False)
    g, f = rng.standard_normal((nrhs, P, 4 * N)), rng.standard_normal((nrhs, P, N * N))
    u, h, hp = pv.solve(g, f, nrhs), pv.map_d2n(g, f, nrhs), pv.map_d2n(None, f, nrhs)
    for c in range(nrhs):
        assert np.array_equal(u[c], pv.solve(g[c], f[c])[0]), c
        assert np.array_equal(h[c], pv.map_d2n(g[c], f[c])[0]), c
        assert np.array_equal(hp[c], pv.map_d2n(None, f[c])[0]), c


@pytest.mark.gpu
@pytest.mark.parametrize("N,P,nrhs", [(6, 9, 3), (10, 1, 2), (12, 8, 3), (12, 17, 18), (24, 7, 5)])
def test_general_solve(patch_ctx, N, P, nrhs):
    tp.say(f"variable-coefficient leaf solves N={N}, {P} patches, {nrhs} right-hand sides")
    general_case(patch_ctx, N, P, nrhs)


def test_emu_general_solve(emu_ctx):
    general_case(emu_ctx, 10, 9, 2)
