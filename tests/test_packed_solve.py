"""The packed variable-coefficient leaf solve (bt_solve_mfma_kernel): right-hand sides that fill its
groups of four and leave remainders, few patches and more items than resident waves.  Every
operation against the oracle, and every column of a batch bit for bit as alone.
"""
import numpy as np
import pytest

import test_patches as tp


def packed_case(ctx, N, P, nrhs, seed, check=True):
    from ellipticforest_amd import _lib
    rng = np.random.default_rng(seed)
    bounds = tp.random_bounds(rng, P)
    cell = tp.variable_cells(bounds, N)
    pv = _lib.Patches(ctx, bounds, N, solver_type=_lib.EF_SOLVER_FIVE_POINT, cell=cell)
    assert pv.packed
    if check:
        tp.check_against_oracle(pv, bounds, N, rng, nrhs=nrhs, coeffs=cell, dtn=False)
    g, f = rng.standard_normal((nrhs, P, 4 * N)), rng.standard_normal((nrhs, P, N * N))
    u, h, hp = pv.solve(g, f, nrhs), pv.map_d2n(g, f, nrhs), pv.map_d2n(None, f, nrhs)
    for c in range(nrhs):
        assert np.array_equal(u[c], pv.solve(g[c], f[c])[0]), c
        assert np.array_equal(h[c], pv.map_d2n(g[c], f[c])[0]), c
        assert np.array_equal(hp[c], pv.map_d2n(None, f[c])[0]), c


@pytest.mark.gpu
@pytest.mark.parametrize("N,P,nrhs", [(16, 1, 1), (16, 5, 3), (16, 3, 5), (32, 1, 4), (32, 3, 7), (32, 2, 18)])
def test_packed_solve(patch_ctx, N, P, nrhs):
    tp.say(f"packed leaf solves N={N}, {P} patches, {nrhs} right-hand sides")
    packed_case(patch_ctx, N, P, nrhs, seed=N + 10 * P + nrhs)


@pytest.mark.gpu
def test_packed_solve_strided(patch_ctx):
    tp.say("packed leaf solves, more items than resident waves: N=16, 700 patches, 14 right-hand sides")
    packed_case(patch_ctx, 16, 700, 14, seed=4, check=False)


def test_emu_packed_solve(emu_ctx):
    packed_case(emu_ctx, 16, 1, 5, seed=3)


@pytest.mark.gpu
def test_packed_work_is_bounded(patch_ctx):
    """Neumann maps of 16 right-hand sides keep at most 256 MiB of work for a batch whose 16 would take 288."""
    import ctypes
    from ellipticforest_amd import _lib
    N, P, k = 32, 2304, 16
    tp.say(f"packed Neumann maps, {P} patches, N={N}, {k} right-hand sides: work space")
    rng = np.random.default_rng(8)
    bounds = tp.random_bounds(rng, P)
    pv = _lib.Patches(patch_ctx, bounds, N, solver_type=_lib.EF_SOLVER_FIVE_POINT, cell=tp.variable_cells(bounds, N))
    assert pv.packed
    f = rng.standard_normal((k, P, N * N))
    fd, hd = _lib.DeviceArray(patch_ctx, f.shape), _lib.DeviceArray(patch_ctx, (k, P, 4 * N))
    fd.upload(f)

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value

    before = free()
    pv.apply_device(_lib.EF_PATCH_MAP_D2N, None, fd.ptr, hd.ptr, k)
    pv.sync()
    assert before - free() <= 260 << 20
    h = hd.download().reshape(k, P, 4 * N)
    for c in (0, 11, 12, 15):
        assert np.array_equal(h[c], pv.map_d2n(None, f[c])[0]), c
