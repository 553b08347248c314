"""The cases of test_gpu_parity.py that compare captured sweeps with eager ones, with the capture asked for:
sweeps are captured only where EF_GRAPH is set to something other than 0, and those cases leave it unset on their
captured side.  The arena regrown, and the packed leaves' work grown with the width, between replays."""
import ctypes
import os
import types

import pytest

import test_gpu_parity as gp
from oracle import mesh as omesh


class _Environ:
    """os.environ for a case: where it takes EF_GRAPH away again, captures are on."""

    def __setitem__(self, key, value):
        os.environ[key] = value

    def __delitem__(self, key):
        os.environ[key] = "1"


@pytest.fixture
def captured(monkeypatch):
    monkeypatch.setenv("EF_GRAPH", "1")
    monkeypatch.setattr(gp, "os", types.SimpleNamespace(environ=_Environ(), path=os.path, cpu_count=os.cpu_count))


def replays(ctx):
    ctx.L.emu_count.restype = ctypes.c_longlong
    return ctx.L.emu_count(b"graph launches")


@pytest.mark.gpu
def test_graph_replay(ctx, captured):
    leaves = omesh.refine_by_function(lambda x, y: abs(gp.F(x, y)) > 1.2, 8, 8, -10, 10, -10, 10, 0, 5)
    gp.say("captured sweeps against eager ones, adaptive N=8 mesh, arena regrown")
    gp.graph_replay_case(ctx, leaves, 8, (-10, 10, -10, 10))


@pytest.mark.gpu
def test_graph_widths(ctx, captured):
    gp.variable_graph_widths_case(ctx)


def test_emu_graph_replay(emu_ctx, captured):
    """Two stages each: seven steps of the compared width, one of the wider one, three on host arrays."""
    leaves = omesh.refine_by_function(lambda x, y: (x < 0.2) & (y < 0.2), 4, 4, 0, 1, 0, 1, 0, 3)
    before = replays(emu_ctx)
    gp.graph_replay_case(emu_ctx, leaves, 4, (0, 1, 0, 1), k=2)
    assert replays(emu_ctx) - before == 2 * 7 + 2 + 2 * 3


def test_emu_graph_widths(emu_ctx, captured):
    before = replays(emu_ctx)
    gp.variable_graph_widths_case(emu_ctx)
    assert replays(emu_ctx) - before == 2 * 4
