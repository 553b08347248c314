"""Systems whose elimination in natural order stops at a large multiplier and goes on with row exchanges: merges
and Robin roots that stop in every step of the blocked inversion, whole and partial, against the oracle with the
parity tests' tolerances; and what such a build does beside that."""
import ctypes

import numpy as np
import pytest

import oracle
import test_gpu_parity as gp
import test_merge_inverse as tm
import test_robin_rows as tr
from oracle import mesh as omesh


def first_large(X):
    """First column of Gauss-Jordan on X without row exchanges with a multiplier beyond 4; the order if none has."""
    A = np.array(X)
    for j in range(len(A)):
        col = A[:, j] / A[j, j]
        col[j] = 0.0
        if not np.abs(col).max() <= 4.0:
            return j
        row = A[j].copy()
        row[j] = 1.0
        row /= A[j, j]
        old = A[:, j].copy()
        A[:, j] = 0.0
        A -= np.outer(old, row)
        A[j] = row
    return len(A)


def merge_case(ctx, N, level, lam, step):
    """The root merge stops in step `step` (64 columns each), its children's nowhere."""
    O = tm.merge_case(ctx, N, level, lam, nodes=[0, 1])
    if level > 1:
        X = O.get(1, "X")
        assert first_large(X) == len(X)
    assert first_large(O.get(0, "X")) // 64 == step


# order 160 (the last step 32 wide) and 256
@pytest.mark.gpu
@pytest.mark.parametrize("N,level,lam,step", [(20, 2, 40.0, 0), (20, 2, 10.0, 1), (20, 2, 15.0, 2), (16, 3, 8.0, 3)])
def test_merge_stops(ctx, N, level, lam, step):
    gp.say(f"merge of order {4 * N * 2 ** (level - 1)} that stops in step {step}")
    merge_case(ctx, N, level, lam, step)


def root_case(ctx, N, level, lam, kind, step):
    """A Robin root that stops in step `step` (-1: nowhere) of its rows as the solve scales them."""
    O, a, b = tr.root_case(ctx, N, level, lam, kind)
    T = O.get(0, "T")
    scale = np.where(b == 0.0, 1.0, 2.0 ** -np.floor(np.log2(np.abs(np.where(b == 0.0, 1.0, b)))))
    stop = first_large((scale * b)[:, None] * T + np.diag(np.where(b == 0.0, np.diag(T), scale * a)))
    assert (stop // 64 if stop < len(T) else -1) == step, stop


# order 64 and 128 (in registers), 160 and 256; step -1: nowhere
ROOTS = [(8, 1, -1.0, "rows", 0), (8, 2, -1.0, "minus", 0), (20, 1, -1.0, "rows", -1), (20, 1, -1.0, "minus", 0),
         (16, 2, 20.0, "plus", 1), (16, 2, 5.0, "minus", 1), (16, 2, 60.0, "rows", 0)]


@pytest.mark.gpu
@pytest.mark.parametrize("N,level,lam,kind,step", ROOTS)
def test_root_stops(ctx, N, level, lam, kind, step):
    gp.say(f"Robin root of order {4 * N * 2 ** level}, lambda = {lam}, {kind}")
    root_case(ctx, N, level, lam, kind, step)


def test_emu_stop_ends_the_natural_order(emu_ctx):
    """lambda = 60 and 100 on merges of order 16 and 32, the deeper group with a large multiplier: a build takes
    its rows in natural order up to there, and each group's S and T products once (before: as many again)."""
    import ellipticforest_amd as ef
    emu_ctx.L.emu_count.restype = ctypes.c_longlong
    D = ef.DeviceMesh(emu_ctx, omesh.uniform(2), 4, (-1, 1, -1, 1))
    products = {}
    for lam in (-1.0, 60.0, 100.0):
        before = emu_ctx.L.emu_count(b"products")
        D.build(lambda0=lam)
        products[lam] = emu_ctx.L.emu_count(b"products") - before
    assert max(products[60.0], products[100.0]) <= products[-1.0], products


def rough(x, y):
    """beta in [1, 1e4], another at every face."""
    return 10.0 ** (4.0 * np.modf(np.abs(np.sin(np.round(40 * x) * 12.9898 + np.round(40 * y) * 78.233)) * 43758.5453)[0])


def contrast_case(ctx, N, level):
    """A beta whose contrast stops the merges: T, S and u against the oracle."""
    import ellipticforest_amd as ef
    leaves, bounds = omesh.uniform(level), (-1.0, 1.0, -1.0, 1.0)
    fns = (gp.ALPHA, rough, gp.LAMBDA)
    O = oracle.Forest(leaves, N, bounds, solver=oracle.FIVE_POINT, coeff_fns=fns)
    O.build()
    X = O.get(0, "X")
    assert first_large(X) < len(X)
    f = O.sample_rhs(gp.F3)
    O.upwards(f)
    r, a, b = O.boundary_data(lambda s, x, y: (gp.U3(x, y), 1.0, 0.0))
    D = ef.DeviceMesh(ctx, leaves, N, bounds)
    cell = np.concatenate([oracle.sample_coeffs(N, tuple(D.node_bounds[n]), *fns).ravel() for n in D.leaf_nodes])
    D.build(solver_type=ef._lib.EF_SOLVER_FIVE_POINT, cell=cell)
    for which in ("T", "S"):
        assert gp.rel(D.get(0, which), O.get(0, which)) < gp.TOL_OP, which
    D.upwards(f)
    assert gp.rel(D.solve(r, a), O.solve(r, a, b)) < gp.TOL_U


@pytest.mark.gpu
@pytest.mark.parametrize("N,level", [(8, 3), (16, 3)])
def test_contrast_stops(ctx, N, level):
    gp.say(f"beta of contrast 1e4, uniform level {level}, N={N}")
    contrast_case(ctx, N, level)


def test_emu_contrast_stops(emu_ctx):
    contrast_case(emu_ctx, 4, 2)
