"""Sweep tiles on a level whose products are not split: 1,024 merges of n = 8, 2,048 row tiles of w and u (a
launch of fewer than 1,024 is split over k and runs 16 x 16 tiles whatever is asked for).  The fixed rule, every
forced tile and the timed choice give the same bits, and a column of the batch those of its own solve."""
import numpy as np
import pytest

import test_gpu_parity as gp
from oracle import mesh as omesh


@pytest.mark.gpu
@pytest.mark.parametrize("k", [7, 40])
def test_unsplit_sweep_tiles(ctx, k):
    import ellipticforest_amd as ef
    gp.say(f"sweep tiles of unsplit products, uniform level 6, N=8, {k} right-hand sides")
    leaves = omesh.uniform(6)
    D = ef.DeviceMesh(ctx, leaves, 8, (-1, 1, -1, 1))
    D.build(lambda0=-1.0)
    rng = np.random.default_rng(6)
    f, r = rng.standard_normal((k, len(leaves), 64)), rng.standard_normal((k, 4 * D.M))
    ref = None
    for mode in (0, 11, 12, 22, 1):
        D.set_autotune(mode)
        w, _, u = D.sweep_tiles(k)[5]  # the deepest merges
        if mode > 1:
            assert w == mode and u == mode, (mode, w, u)
        if mode == 0:
            assert w == u == (11 if k <= 16 else 22), (w, u)
        D.upwards(f)
        out = D.solve(r, 1.0)
        ref = out if ref is None else ref
        assert np.array_equal(out, ref), mode
    for j in (0, k - 1):
        D.upwards(f[j])
        assert np.array_equal(D.solve(r[j], 1.0), ref[j]), j
