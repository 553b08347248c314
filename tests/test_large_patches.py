"""Large patches (N > 32, patch_large_gemm_kernel) at sides that leave partial tiles and unequal quarters of
the k range: every operation against the oracle, batches against single patches bit for bit."""
import numpy as np
import pytest

import test_patches as tp


def large_case(ctx, N, P, nrhs, dtn):
    from ellipticforest_amd import _lib
    rng = np.random.default_rng(N)
    bounds = tp.random_bounds(rng, P)
    pt = _lib.Patches(ctx, bounds, N, lambda0=-1.0)
    tp.check_against_oracle(pt, bounds, N, rng, nrhs=nrhs, lam=-1.0, dtn=dtn)
    g, f = rng.standard_normal((nrhs, P, 4 * N)), rng.standard_normal((nrhs, P, N * N))
    u = pt.solve(g, f, nrhs)
    one = _lib.Patches(ctx, bounds[-1:], N, lambda0=-1.0)
    assert np.array_equal(u[-1, -1], one.solve(g[-1, -1:], f[-1, -1:])[0, 0])


@pytest.mark.gpu
@pytest.mark.parametrize("N,P,nrhs", [(33, 3, 2), (47, 1, 1), (65, 2, 1), (81, 1, 2), (130, 1, 1)])
def test_large_patches(patch_ctx, N, P, nrhs):
    tp.say(f"large patches N={N}, {P} patches, {nrhs} right-hand sides")
    large_case(patch_ctx, N, P, nrhs, dtn=N < 65)


def test_emu_large_patches(emu_ctx):
    large_case(emu_ctx, 33, 1, 1, dtn=False)
