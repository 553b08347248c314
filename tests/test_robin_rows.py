"""Robin root systems a u + b du/dn = r by their rows: b = 0 on some, signs of a / b that change, and rows whose a / b
is beyond the range of a double; several widths in turn on one mesh, against the oracle."""
import numpy as np
import pytest

import oracle
import test_gpu_parity as gp
from oracle import mesh as omesh


def root_rows(m, kind):
    """a and b of a root with 4 m / 4 faces: `plus` and `minus` by the sign of a / b outwards, `rows` with b = 0 on
    every third row and signs of a / b that change beside it, `far` with a / b = 1e320 on every second row."""
    rng = np.random.default_rng(m)
    a = 3.0 + 0.5 * rng.random(m)
    b = np.repeat([-1.0, 1.0, -1.0, 1.0], m // 4) * (0.25 + rng.random(m))  # du/dn outwards on W, E, S, N
    if kind == "minus":
        b = -b
    elif kind == "rows":
        b[::3] = 0.0
        b[1::6] *= -1.0
    elif kind == "far":
        a[::2] *= 1e200
        b[::2] *= 1e-120
    return a, b


def root_case(ctx, N, level, lam, kind, ks=(1, 5, 1)):
    import ellipticforest_amd as ef
    leaves, bounds = omesh.uniform(level), (-1, 1, -1, 1)
    O = oracle.Forest(leaves, N, bounds, solver=oracle.FISHPACK, lambda0=lam)
    O.build()
    D = ef.DeviceMesh(ctx, leaves, N, bounds)
    D.build(lambda0=lam)
    m = 4 * D.M
    a, b = root_rows(m, kind)
    rng = np.random.default_rng(N)
    f = rng.standard_normal((max(ks), D.nleaves, N * N))
    r = a * rng.standard_normal((max(ks), m))
    for k in ks:
        D.upwards(f[:k])
        u = D.solve(r[:k], a, b)
        for c in range(k):
            O.upwards(f[c])
            assert gp.rel(u[c], O.solve(r[c], a, b)) < gp.TOL_U, (kind, k, c)
    return O, a, b


def rebuild_case(ctx, N, level, ks):
    """One mesh built again: the root's system is formed from the new T, and its product's plan, kept where no address
    moved, reads the new inverse."""
    import ellipticforest_amd as ef
    leaves, bounds = omesh.uniform(level), (-1, 1, -1, 1)
    D = ef.DeviceMesh(ctx, leaves, N, bounds)
    a, b = root_rows(4 * D.M, "plus")
    rng = np.random.default_rng(N)
    for lam in (-1.0, -30.0, -1.0):
        O = oracle.Forest(leaves, N, bounds, solver=oracle.FISHPACK, lambda0=lam)
        O.build()
        D.build(lambda0=lam)
        for k in ks:
            f, r = rng.standard_normal((k, D.nleaves, N * N)), rng.standard_normal((k, 4 * D.M))
            D.upwards(f)
            u = D.solve(r, a, b)
            for c in range(k):
                O.upwards(f[c])
                assert gp.rel(u[c], O.solve(r[c], a, b)) < gp.TOL_U, (lam, k, c)


@pytest.mark.gpu
def test_root_after_rebuild(ctx):
    gp.say("Robin roots of one mesh built again, order 160")
    rebuild_case(ctx, 20, 1, (1, 3))


def test_emu_root_after_rebuild(emu_ctx):
    rebuild_case(emu_ctx, 4, 1, (1,))


@pytest.mark.gpu
@pytest.mark.parametrize("N,level,kind", [(8, 1, "far"), (20, 1, "far"), (20, 1, "rows"), (20, 1, "plus")])
def test_root_rows(ctx, N, level, kind):
    gp.say(f"Robin root of order {4 * N * 2 ** level}, {kind}")
    root_case(ctx, N, level, -1.0, kind)


@pytest.mark.parametrize("kind", ["far", "rows"])
def test_emu_root_rows(emu_ctx, kind):
    root_case(emu_ctx, 4, 1, -1.0, kind, ks=(1, 3))
