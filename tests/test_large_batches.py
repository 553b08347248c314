"""Batches of large patches that fill the chip: one wave takes a whole block there (sides up to 64), and Neumann
data form the blocks of the edge cells only; every patch's bits are those of a batch of one, and those of a
patch are checked against the oracle in test_large_patches.py."""
import numpy as np
import pytest

import test_patches as tp


# 33, 47: tiles past the matrix, three blocks of k; 64: whole; 65, 100: three and four blocks a side
@pytest.mark.gpu
@pytest.mark.parametrize("N,P,nrhs", [(33, 256, 1), (47, 86, 3), (64, 255, 1), (64, 256, 1), (65, 130, 1), (100, 70, 1)])
def test_large_batches(patch_ctx, N, P, nrhs):
    from ellipticforest_amd import _lib
    tp.say(f"large patches N={N}, {P} patches, {nrhs} right-hand sides against single ones")
    rng = np.random.default_rng(N)
    bounds = tp.random_bounds(rng, P)
    pt = _lib.Patches(patch_ctx, bounds, N, lambda0=-1.0)
    g, f = rng.standard_normal((nrhs, P, 4 * N)), rng.standard_normal((nrhs, P, N * N))
    u, h, hp = pt.solve(g, f, nrhs), pt.map_d2n(g, f, nrhs), pt.map_d2n(None, f, nrhs)
    h0 = pt.map_d2n(g, None, nrhs)
    for p in (0, P // 2, P - 1):
        one = _lib.Patches(patch_ctx, bounds[p:p + 1], N, lambda0=-1.0)
        for c in range(nrhs):
            gc, fc = g[c, p:p + 1], f[c, p:p + 1]
            assert np.array_equal(u[c, p], one.solve(gc, fc)[0, 0])
            assert np.array_equal(h[c, p], one.map_d2n(gc, fc)[0, 0])
            assert np.array_equal(hp[c, p], one.map_d2n(None, fc)[0, 0])
            assert np.array_equal(h0[c, p], one.map_d2n(gc, None)[0, 0])


@pytest.mark.gpu
def test_large_dtn_fills(patch_ctx):
    """4 x 64 columns of the DtN of a 64 x 64 patch: 1,024 blocks."""
    from ellipticforest_amd import _lib
    tp.say("DtN of a large patch, one wave per block")
    rng = np.random.default_rng(1)
    bounds = tp.random_bounds(rng, 2)
    pt = _lib.Patches(patch_ctx, bounds, 64, lambda0=-1.0)
    tp.check_against_oracle(pt, bounds, 64, rng, nrhs=1, lam=-1.0, dtn=True)
