"""EF_GRAPH=1: the captured sweeps replay the eager launches' bits, on every replay, with other work between
replays, with changed inputs under the same pointers and after a build that keeps the captures."""

import numpy as np
import pytest

import test_gpu_parity as gp
from oracle import mesh as omesh


def captured_case(ctx, leaves, N, k, monkeypatch):
    from ellipticforest_amd import _lib
    D = _lib.DeviceMesh(ctx, leaves, N, (0, 1, 0, 1))
    D.set_autotune(0)
    D.build(lambda0=-1.0)
    nl, m = len(leaves), 4 * D.M
    rng = np.random.default_rng(2)
    f, r, a = rng.standard_normal((2, k, nl, N * N)), rng.standard_normal((2, k, m)), np.ones(m)
    fd, rd, ad, ud = (_lib.DeviceArray(ctx, s) for s in (f[0].shape, r[0].shape, a.shape, f[0].shape))
    ad.upload(a)

    def sweep(i, graph):
        monkeypatch.setenv("EF_GRAPH", "1" if graph else "0")
        fd.upload(f[i])
        rd.upload(r[i])
        D.upwards_device(fd.ptr, k)
        D.solve_device(fd.ptr, rd.ptr, ad.ptr, None, ud.ptr, k)
        D.sync()
        return ud.download()

    for lam in (-1.0, -3.0):
        D.build(lambda0=lam)
        eager = [sweep(i, False) for i in (0, 1)]
        for rep in range(3):
            for i in (0, 1):
                assert np.array_equal(sweep(i, True), eager[i]), (lam, rep, i)
            D.upwards(f[0][:1])
            D.solve(r[0][:1], a)


@pytest.mark.gpu
def test_captured_sweeps(ctx, monkeypatch):
    gp.say("captured sweeps, adaptive, replayed over two builds")
    leaves = omesh.refine_by_function(lambda x, y: (x < 0.2) & (y < 0.2), 8, 8, 0, 1, 0, 1, 1, 4)
    captured_case(ctx, leaves, 8, 3, monkeypatch)


def test_emu_captured_sweeps(emu_ctx, monkeypatch):
    captured_case(emu_ctx, omesh.uniform(1), 4, 2, monkeypatch)
