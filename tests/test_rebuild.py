"""A mesh built again keeps its sweep plans and captured sweeps where no address moved: every build of
a sequence (coefficients, kinds of leaf, and back) gives a new mesh's results, bit for bit."""
import numpy as np
import pytest

import test_gpu_parity as gp
from oracle import mesh as omesh


def rebuild_case(ctx, leaves, N, bounds, ks):
    import ellipticforest_amd as ef
    from ellipticforest_amd import _lib
    rng = np.random.default_rng(1)
    nl = len(leaves)
    cell = np.ones((nl, 6, N * N))
    cell[:, 5] = -0.5
    per_leaf = cell * (1.0 + rng.random((nl, 1, 1)))
    varying = cell.copy()
    varying[:, 1:5] += rng.random((nl, 1, N * N))
    five = dict(solver_type=_lib.EF_SOLVER_FIVE_POINT)
    builds = [dict(lambda0=0.0), dict(lambda0=-2.0), dict(five, cell=varying), dict(five, cell=varying * 1.5),
              dict(five, cell=per_leaf), dict(lambda0=0.0), dict(five, alpha0=1.25, beta0=2.0, lambda0=-1.0)]
    D = ef.DeviceMesh(ctx, leaves, N, bounds)
    D.set_autotune(0)
    for kw in builds:
        D.build(**kw)
        E = ef.DeviceMesh(ctx, leaves, N, bounds)
        E.set_autotune(0)
        E.build(**kw)
        for k in ks:
            f, r = rng.standard_normal((k, nl, N * N)), rng.standard_normal((k, 4 * D.M))
            u = []
            for mesh in (D, E):
                mesh.upwards(f)
                u.append(mesh.solve(r, 1.0))
            assert np.array_equal(u[0], u[1]), (sorted(kw), k)


@pytest.mark.gpu
def test_rebuild(ctx):
    gp.say("builds of one mesh in a row, adaptive")
    leaves = omesh.refine_by_function(lambda x, y: np.abs(gp.F(x, y)) > 1.2, 8, 8, -10, 10, -10, 10, 0, 4)
    rebuild_case(ctx, leaves, 8, (-10, 10, -10, 10), (1, 3))


def test_emu_rebuild(emu_ctx):
    rebuild_case(emu_ctx, omesh.uniform(1), 4, (0, 1, 0, 1), (2,))
