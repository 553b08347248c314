"""The workloads that the framework's speed is measured on, through its public entry points.

A user of the framework refines a mesh, factorises it once (``build``) and then solves for many
right-hand sides on it (``upwards`` + ``solve``), or hands batches of independent leaf patches to
the patch solver.  The cases below are that work over its real range: a handful of patches, where
launches and latency count; a mesh of 64 leaves; the adaptive Poisson mesh of the benchmark (7,750
leaves) for one request, for a served batch and for 64 right-hand sides; a variable-coefficient
mesh of 2048 x 2048 cells; factorisation of each; and a driver that keeps its arrays on the host.
Everything is FP64, the framework's only data type at its entry points.

``listed`` names the cases, ``draw`` gives more of the same ranges, ``prepare`` makes what a
program holds before the call, ``run`` is one pass, ``work`` the bytes and operations one pass
cannot do without, ``exact`` the same results from plain torch in 64 bits.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import ellipticforest_amd as ef
from ellipticforest_amd import _lib, serving

# The meshes of the adaptive cases: |sin x + sin y| > 1.2 on [-10, 10]^2 is refined, as in the
# benchmark's Poisson problem.  Variable-coefficient and uniform meshes lie on [-1, 1]^2.
ADAPTIVE = (-10.0, 10.0, -10.0, 10.0)
SQUARE = (-1.0, 1.0, -1.0, 1.0)
ROBIN = 0.5  # b of the driver's root condition u + b du/dn = r


def listed():
    return [
        # a few patches and right-hand sides: a program that tries the leaf solver out
        dict(name="patch_solve_few", kind="patch", op="solve", P=6, N=16, k=2, var=False),
        # every leaf of the benchmark's mesh, 16 right-hand sides: the leaf stage of a solve
        dict(name="patch_solve_leaves", kind="patch", op="solve", P=7750, N=16, k=16, var=False),
        # Neumann data of a variable-coefficient leaf set
        dict(name="patch_d2n_variable", kind="patch", op="d2n", P=4096, N=32, k=1, var=True),
        # one finite-volume grid on its own (the reference's single-patch solver test, n = 512)
        dict(name="grid_solve", kind="patch", op="solve", P=1, N=512, k=1, var=False),
        # one request on a small factorised mesh (64 leaves)
        dict(name="solve_uniform_1", kind="solve", mesh="uniform", level=3, N=16, k=1, var=False, lam=0.0),
        # one request on the benchmark's mesh
        dict(name="solve_adaptive_1", kind="solve", mesh="adaptive", level=7, N=16, k=1, var=False, lam=0.0),
        # 64 right-hand sides at once on it: the benchmark's step
        dict(name="solve_adaptive_64", kind="solve", mesh="adaptive", level=7, N=16, k=64, var=False, lam=0.0),
        # four right-hand sides with variable coefficients (4,096 leaves of 32 x 32 cells)
        dict(name="solve_variable_4", kind="solve", mesh="uniform", level=6, N=32, k=4, var=True, lam=-1.0),
        # a served batch of odd width: loads evaluated on the device, then the solve
        dict(name="serve_batch", kind="serve", mesh="adaptive", level=6, N=8, k=21, var=False, lam=0.0),
        # a driver's whole run on host arrays with a Robin condition at the root: build, upwards, solve
        dict(name="driver_robin", kind="driver", mesh="uniform", level=4, N=16, k=1, var=False, lam=-1.0),
        # factorisation of the benchmark's mesh and its first solve
        dict(name="factor_adaptive", kind="factor", mesh="adaptive", level=7, N=16, k=1, var=False, lam=0.0),
        # factorisation with new variable coefficients and a first solve (1,024 leaves of 32 x 32 cells)
        dict(name="factor_variable", kind="factor", mesh="uniform", level=5, N=32, k=1, var=True, lam=-1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["patch", "patch", "grid", "solve", "solve", "solve", "serve", "driver", "factor", "factor"])
    if kind == "grid":
        return dict(kind="patch", op=rng.choice(["solve", "d2n"]), P=1, N=_log(rng, 40, 512), k=1, var=False)
    if kind == "patch":
        var = rng.random() < 0.4
        N = rng.choice([8, 16, 32]) if var else rng.choice([4, 8, 10, 12, 16, 20, 24, 32])
        cells = 7750 * 256 if var else 7750 * 256 * 4
        k = _log(rng, 1, 4 if var else 16)
        return dict(kind="patch", op=rng.choice(["solve", "d2n"]), P=_log(rng, 3, max(4, cells // (N * N * k))), N=N, k=k,
                    var=var)
    # mesh cases: level and N so that no mesh is larger than the listed one of its kind
    N = rng.choice([8, 12, 16, 32])
    lg = 5 if N == 32 else 4 if N > 8 else 3
    lam = rng.choice([0.0, -1.0])
    if kind == "serve":
        return dict(kind=kind, mesh="adaptive", level=rng.randint(4, 9 - lg), N=N, k=_log(rng, 2, 21), var=False, lam=lam)
    if kind == "driver":
        return dict(kind=kind, mesh="uniform", level=rng.randint(2, 8 - lg), N=N, k=1, var=False, lam=lam)
    var = N != 12 and rng.random() < 0.3
    mesh = "uniform" if var else rng.choice(["uniform", "adaptive", "adaptive"])
    level = rng.randint(2, 9 - lg) if mesh == "uniform" else rng.randint(4, 11 - lg)
    k = 1 if kind == "factor" else _log(rng, 1, 4 if var else 64)
    return dict(kind=kind, mesh=mesh, level=level, N=N, k=k, var=var, lam=lam)


# ----- what a program has in hand ------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _context():
    return ef.Context(0)


@functools.lru_cache(maxsize=None)
def _stream():
    """The one stream the program queues its work on."""
    return torch.cuda.Stream()


@functools.lru_cache(maxsize=64)
def _leaves(mesh, level, N):
    if mesh == "adaptive":
        return tuple(ef.refine_by_function(lambda x, y: np.abs(np.sin(x) + np.sin(y)) > 1.2, N, N, ADAPTIVE, 0, level))
    out = []
    for z in range(4 ** level):  # z-order: x in the even bits
        ix = sum(((z >> (2 * b)) & 1) << b for b in range(level))
        iy = sum(((z >> (2 * b + 1)) & 1) << b for b in range(level))
        out.append((level, ix, iy))
    return tuple(out)


def _bounds(case):
    return ADAPTIVE if case["mesh"] == "adaptive" else SQUARE


def _leaf_bounds(case):
    xl, xu, yl, yu = _bounds(case)
    q = np.array(_leaves(case["mesh"], case["level"], case["N"]), np.float64)
    w = 2.0 ** -q[:, 0]
    return np.stack([xl + (xu - xl) * q[:, 1] * w, xl + (xu - xl) * (q[:, 1] + 1) * w,
                     yl + (yu - yl) * q[:, 2] * w, yl + (yu - yl) * (q[:, 2] + 1) * w], 1)


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _gen(seed):
    return torch.Generator(device=_device()).manual_seed(seed)


def _centres(bounds, N):
    """Cell centres of patches, x and y as [P, N, 1] and [P, 1, N] (cell index x-major)."""
    b = torch.as_tensor(bounds, dtype=torch.float64, device=_device())
    t = torch.arange(N, dtype=torch.float64, device=_device()) + 0.5
    x = b[:, 0:1] + t * ((b[:, 1] - b[:, 0]) / N)[:, None]
    y = b[:, 2:3] + t * ((b[:, 3] - b[:, 2]) / N)[:, None]
    return x[:, :, None], y[:, None, :]


def _waves(p, x, y):
    """Four plane waves a sin(kx x + ky y + phi) for every right-hand side: p is [k, 4, 4]."""
    out = 0.0
    for q in range(4):
        a, kx, ky, phi = (p[:, q, c].reshape(-1, *([1] * (x + y).dim())) for c in range(4))
        out = out + a * torch.sin(kx * x + ky * y + phi)
    return out


def _cells(bounds, N, seed, lam):
    """Per-cell samples [P][6][N*N] of alpha = 1, beta = 1 + 0.5 sin(a x + b y) at the four faces, lambda."""
    a, b = (torch.rand(2, generator=_gen(seed + 7), dtype=torch.float64, device=_device()) * 4.0).tolist()
    x, y = _centres(bounds, N)
    d = torch.as_tensor(bounds, dtype=torch.float64, device=_device())
    dx, dy = ((d[:, 1] - d[:, 0]) / N)[:, None, None], ((d[:, 3] - d[:, 2]) / N)[:, None, None]
    beta = lambda x, y: 1.0 + 0.5 * torch.sin(a * x + b * y)
    full = torch.ones(len(bounds), N, N, dtype=torch.float64, device=_device())
    return torch.stack([full, beta(x - dx / 2, y), beta(x + dx / 2, y), beta(x, y - dy / 2), beta(x, y + dy / 2),
                        lam * full], 1).reshape(len(bounds), 6, N * N)


def _patch_bounds(P):
    """Patches of a sheet of quadrants of three sizes."""
    i = np.arange(P)
    w = 0.5 ** (1 + i % 3)
    x, y = 0.25 * (i % 64), 0.25 * (i // 64)
    return np.stack([x, x + w, y, y + w], 1)


def _patch_inputs(case, seed):
    P, N, k, g = case["P"], case["N"], case["k"], _gen(seed)
    rn = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64, device=_device())
    return rn(k, P, 4 * N), rn(k, P, N * N)


def _root_points(case, M):
    xl, xu, yl, yu = _bounds(case)
    t = (torch.arange(M, dtype=torch.float64, device=_device()) + 0.5) / M
    one = torch.ones_like(t)
    return (torch.cat([xl * one, xu * one, xl + (xu - xl) * t, xl + (xu - xl) * t]),
            torch.cat([yl + (yu - yl) * t, yl + (yu - yl) * t, yl * one, yu * one]))


def _mesh_inputs(case, M, seed):
    """Loads f [k][leaf][N*N] and root data r [k][4M]: plane waves with seeded numbers and phases."""
    g, k, N = _gen(seed), case["k"], case["N"]
    p = torch.randn(2, k, 4, 4, generator=g, dtype=torch.float64, device=_device())
    f = _waves(p[0], *_centres(_leaf_bounds(case), N))
    r = _waves(p[1], *_root_points(case, M))
    return f.reshape(k, -1, N * N).contiguous(), r.contiguous()


def _serve_params(case, seed):
    return serving.workload_params(np.random.default_rng(seed), _bounds(case), case["k"])


def prepare(case, seed):
    N, k, ctx = case["N"], case["k"], _context()
    s = dict(case=case)
    if case["kind"] == "patch":
        bounds = _patch_bounds(case["P"])
        if case["var"]:
            s["pt"] = ef.Patches(ctx, bounds, N, solver_type=_lib.EF_SOLVER_FIVE_POINT,
                                 cell=_cells(bounds, N, seed, -1.0).cpu().numpy())
        else:
            s["pt"] = ef.Patches(ctx, bounds, N, lambda0=-1.0)
        _lib.check(ctx.L.ef_patches_set_stream(s["pt"].h, ctypes.c_void_p(_stream().cuda_stream)), ctx.L)
        s["g"], s["f"] = _patch_inputs(case, seed)
        s["op"] = _lib.EF_PATCH_SOLVE if case["op"] == "solve" else _lib.EF_PATCH_MAP_D2N
        s["out"] = torch.empty_like(s["f"] if case["op"] == "solve" else s["g"])
        return s
    leaves = _leaves(case["mesh"], case["level"], N)
    D = s["D"] = ef.DeviceMesh(ctx, leaves, N, _bounds(case))
    D.set_stream(_stream().cuda_stream)
    s["coef"] = dict(lambda0=case["lam"])
    if case["var"]:
        s["coef"] = dict(solver_type=_lib.EF_SOLVER_FIVE_POINT,
                         cell=_cells(_leaf_bounds(case), N, seed, case["lam"]).cpu().numpy())
    if case["kind"] in ("solve", "serve"):
        D.build(**s["coef"])
        del s["coef"]
    s["a"] = torch.ones(4 * D.M, dtype=torch.float64, device="cuda")
    if case["kind"] == "serve":
        s["params"] = torch.as_tensor(_serve_params(case, seed)).cuda()
        s["f"] = torch.empty(k, len(leaves), N * N, dtype=torch.float64, device="cuda")
        s["r"] = torch.empty(k, 4 * D.M, dtype=torch.float64, device="cuda")
    else:
        s["f"], s["r"] = _mesh_inputs(case, D.M, seed)
    if case["kind"] == "driver":
        s["f"], s["r"], s["a"] = (s[n].cpu().numpy() for n in ("f", "r", "a"))
        s["b"] = np.repeat([-ROBIN, ROBIN, -ROBIN, ROBIN], D.M)  # outward derivative on W, E, S, N
    else:
        s["u"] = torch.empty_like(s["f"])
    return s


def run(s):
    case = s["case"]
    kind, k = case["kind"], case["k"]
    if kind == "patch":
        s["pt"].apply_device(s["op"], s["g"].data_ptr(), s["f"].data_ptr(), s["out"].data_ptr(), k)
        return s["out"]
    D = s["D"]
    if kind == "driver":
        D.build(**s["coef"])
        D.upwards(s["f"])
        return D.solve(s["r"], s["a"], s["b"])
    if kind == "factor":
        D.build(**s["coef"])
    f, r, u = s["f"], s["r"], s["u"]
    if kind == "serve":
        _lib.check(D.L.ef_mesh_eval_load(D.h, ctypes.c_void_p(s["params"].data_ptr()), k, ctypes.c_void_p(f.data_ptr()),
                                         ctypes.c_void_p(r.data_ptr())), D.L)
    D.upwards_device(f.data_ptr(), k)
    D.solve_device(f.data_ptr(), r.data_ptr(), s["a"].data_ptr(), None, u.data_ptr(), k)
    return dict(f=f, r=r, u=u) if kind == "serve" else u


# ----- what a pass cannot do without ---------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _merges(mesh, level, N):
    """Interface size n of every merge, and the root's side."""
    size = {q: N for q in _leaves(mesh, level, N)}
    ns, lv = [], max(q[0] for q in size)
    cur = dict(size)
    for l in range(lv, 0, -1):
        for (_, x, y) in {(l - 1, q[1] // 2, q[2] // 2) for q in cur if q[0] == l}:
            n = min(cur[(l, 2 * x + c % 2, 2 * y + c // 2)] for c in range(4))
            ns.append(n)
            cur[(l - 1, x, y)] = 2 * n
    return ns, cur[(0, 0, 0)]


def work(case):
    N, k = case["N"], case["k"]
    if case["kind"] == "patch":
        P, io = case["P"], 2 * N * N + 4 * N if case["op"] == "solve" else N * N + 8 * N
        # variable coefficients: half a band of factor per cell line; constant: four N x N x N products
        return dict(bytes=8.0 * P * (k * io + (N ** 3 / 2 if case["var"] else 0)), flops=float(P * k * (4 if case["var"] else 8) * N ** 3))
    ns, M = _merges(case["mesh"], case["level"], N)
    nl = len(_leaves(case["mesh"], case["level"], N))
    n2, n3 = float(sum(n * n for n in ns)), float(sum(n ** 3 for n in ns))
    # the sweeps read each merge's X^-1, H and S (64 n^2) and the leaf factors once, each leaf's f and write its u
    lf = N ** 3 / 2 if case["var"] else 0
    by = 8.0 * (64 * n2 + nl * (lf + 2 * N * N * k) + 4 * M * k)
    fl = 128 * n2 * k + 2.0 * nl * k * (4 if case["var"] else 8) * N ** 3
    if case["kind"] == "serve":  # f written by the load evaluation
        by += 8.0 * nl * N * N * k
        fl += 16.0 * nl * N * N * k
    if case["kind"] in ("driver", "factor"):  # X^-1, S and T (112 n^2) written; X inverted, S and T formed
        by += 8.0 * (112 * n2 + (nl * (6 * N * N + 16 * N * N + lf) if case["var"] else 0))
        fl += 512 * n3 + (nl * (2.0 * N ** 4 + 16.0 * N ** 4) if case["var"] else 0)
    if case["kind"] == "driver":
        fl += 2.0 * (4 * M) ** 3 / 3  # the root's boundary system
    return dict(bytes=by, flops=fl)


# ----- the same results from plain torch in 64 bits ------------------------------------------
def _modes(n, end=0.0):
    """Eigenvectors and eigenvalues of tridiag(1, -2, 1) with -3 + end in both corners."""
    K = torch.diag(torch.full((n,), -2.0, dtype=torch.float64)) + torch.diag(torch.ones(n - 1, dtype=torch.float64), 1) \
        + torch.diag(torch.ones(n - 1, dtype=torch.float64), -1)
    K[0, 0] = K[-1, -1] = -3.0 + end
    if end == 0.0:
        i, q = torch.arange(n, dtype=torch.float64) + 0.5, torch.arange(1, n + 1, dtype=torch.float64)
        Q = torch.sin(math.pi * i[:, None] * q / n) * math.sqrt(2.0 / n)
        Q[:, -1] *= math.sqrt(0.5)
        mu = -4.0 * torch.sin(math.pi * q / (2 * n)) ** 2
    else:
        mu, Q = torch.linalg.eigh(K)
    return Q.to(_device()), mu.to(_device())


def _separable(b, dx, dy, lam, end=(0.0, 0.0), scale=1.0):
    """u with scale (u_xx + u_yy) + lam u = b on [..., n, n] cells, homogeneous boundary terms; dx, dy may be [..., 1, 1]."""
    (Qx, mx), (Qy, my) = _modes(b.shape[-2], end[0]), _modes(b.shape[-1], end[1])
    d = scale * (mx[:, None] / dx ** 2 + my / dy ** 2) + lam
    return Qx @ ((Qx.T @ b @ Qy) / d) @ Qy.T


def _varying(b, c, dx, dy):
    """The five-point system with cells c [..., 6, n, n] (alpha = 1): conjugate gradients on the separable inverse."""
    cW, cE, cS, cN, lam = c[..., 1, :, :] / dx ** 2, c[..., 2, :, :] / dx ** 2, c[..., 3, :, :] / dy ** 2, \
        c[..., 4, :, :] / dy ** 2, c[..., 5, :, :]
    centre = -(cW + cE + cS + cN) + lam
    centre[..., 0, :] -= cW[..., 0, :]
    centre[..., -1, :] -= cE[..., -1, :]
    centre[..., :, 0] -= cS[..., :, 0]
    centre[..., :, -1] -= cN[..., :, -1]

    def A(u):
        o = centre * u
        o[..., 1:, :] += cW[..., 1:, :] * u[..., :-1, :]
        o[..., :-1, :] += cE[..., :-1, :] * u[..., 1:, :]
        o[..., :, 1:] += cS[..., :, 1:] * u[..., :, :-1]
        o[..., :, :-1] += cN[..., :, :-1] * u[..., :, 1:]
        return o

    dot = lambda x, y: (x * y).sum((-2, -1), keepdim=True)
    M = lambda x: _separable(x, dx, dy, lam[..., :1, :1], scale=1.0)
    u, r = torch.zeros_like(b), b.clone()
    z = M(r)
    p, rz, r0 = z.clone(), dot(r, z), dot(b, b).max()
    for _ in range(60):
        Ap = A(p)
        al = rz / dot(p, Ap).where(rz != 0, torch.ones_like(rz))
        u += al * p
        r -= al * Ap
        if dot(r, r).max() < 1e-30 * r0:
            break
        z = M(r)
        new = dot(r, z)
        p = z + new / rz.where(rz != 0, torch.ones_like(rz)) * p
        rz = new
    return u


def _boundary_terms(b, g, cx, cy, c=None):
    """b - 2 c_side g_side on the edge cells; g is [..., 4, n] (W, E, S, N); c: cells, or constant coefficients."""
    w = [1.0, 1.0, 1.0, 1.0] if c is None else [c[..., 1, 0, :], c[..., 2, -1, :], c[..., 3, :, 0], c[..., 4, :, -1]]
    b = b.clone()
    b[..., 0, :] -= 2 * cx * w[0] * g[..., 0, :]
    b[..., -1, :] -= 2 * cx * w[1] * g[..., 1, :]
    b[..., :, 0] -= 2 * cy * w[2] * g[..., 2, :]
    b[..., :, -1] -= 2 * cy * w[3] * g[..., 3, :]
    return b


def _neumann(u, g, dx, dy):
    return torch.stack([2 / dx * (u[..., 0, :] - g[..., 0, :]), -2 / dx * (u[..., -1, :] - g[..., 1, :]),
                        2 / dy * (u[..., :, 0] - g[..., 2, :]), -2 / dy * (u[..., :, -1] - g[..., 3, :])], -2)


def _exact_patch(case, seed):
    P, N, k = case["P"], case["N"], case["k"]
    g, f = _patch_inputs(case, seed)
    g, f = g.reshape(k, P, 4, N), f.reshape(k, P, N, N)
    bounds = _patch_bounds(P)
    b = torch.as_tensor(bounds, device=_device())
    dx, dy = ((b[:, 1] - b[:, 0]) / N)[:, None], ((b[:, 3] - b[:, 2]) / N)[:, None]
    D = (dx[..., None], dy[..., None])
    if case["var"]:
        c = _cells(bounds, N, seed, -1.0).reshape(P, 6, N, N)
        u = torch.stack([_varying(_boundary_terms(x, y, 1 / dx ** 2, 1 / dy ** 2, c), c, *D) for x, y in zip(f, g)])
    else:
        u = _separable(_boundary_terms(f, g, 1 / dx ** 2, 1 / dy ** 2), *D, -1.0)
    return u.reshape(k, P, N * N) if case["op"] == "solve" else _neumann(u, g, dx, dy).reshape(k, P, 4 * N)


def _exact_uniform(case, f, r, seed):
    """The global five-point system of a uniform mesh."""
    N, k, side = case["N"], case["k"], 2 ** case["level"]
    n = N * side
    q = torch.as_tensor([(x, y) for _, x, y in _leaves(case["mesh"], case["level"], N)], device=_device())

    def put(v):  # [..., leaf, N, N] -> [..., n, n]
        o = torch.empty(*v.shape[:-3], side, side, N, N, dtype=v.dtype, device=v.device)
        o[..., q[:, 0], q[:, 1], :, :] = v
        return o.transpose(-3, -2).reshape(*v.shape[:-3], n, n)

    xl, xu, yl, yu = _bounds(case)
    dx, dy, g = (xu - xl) / n, (yu - yl) / n, r.reshape(k, 4, n)
    end = (0.0, 0.0)
    if case["kind"] == "driver":  # the ghost value from u + ROBIN du/dn = r at the face
        g = torch.stack([g[:, 0] / (1 + 2 * ROBIN / dx), g[:, 1] / (1 + 2 * ROBIN / dx), g[:, 2] / (1 + 2 * ROBIN / dy),
                         g[:, 3] / (1 + 2 * ROBIN / dy)], 1)
        end = (4 * ROBIN / dx / (1 + 2 * ROBIN / dx), 4 * ROBIN / dy / (1 + 2 * ROBIN / dy))
    F = put(f.reshape(k, -1, N, N))
    if case["var"]:
        c = put(_cells(_leaf_bounds(case), N, seed, case["lam"]).reshape(-1, 6, N, N).transpose(0, 1))
        u = torch.stack([_varying(_boundary_terms(x, y, 1 / dx ** 2, 1 / dy ** 2, c), c, dx, dy) for x, y in zip(F, g)])
    else:
        u = _separable(_boundary_terms(F, g, 1 / dx ** 2, 1 / dy ** 2), dx, dy, case["lam"], end)
    return u.reshape(k, side, N, side, N).transpose(2, 3)[:, q[:, 0], q[:, 1]].reshape(k, -1, N * N)


# Of a merge of four children (SW, SE, NW, NE; sides W, E, S, N): the block of [interfaces 0-3 | parent boundary
# 4-11 in the order W, E, S, N] that each child's side is, and the two sides of each interface.
_BLOCK = ((4, 2, 8, 0), (2, 6, 9, 1), (5, 3, 0, 10), (3, 7, 1, 11))
_IFACE = (((0, 3), (2, 2)), ((1, 3), (3, 2)), ((0, 1), (1, 0)), ((2, 1), (3, 0)))
_OUTER = ((0, 0), (2, 0), (1, 1), (3, 1), (0, 2), (1, 2), (2, 3), (3, 3))


def _halve(n):
    return torch.repeat_interleave(torch.eye(n // 2, dtype=torch.float64, device=_device()), 2, 1) * 0.5


def _double(n):
    """Coarse to fine on a side: 3/4, 1/4 in between, quadratic at both ends."""
    L = torch.zeros(n, n // 2, dtype=torch.float64)
    i = torch.arange(n // 2 - 1)
    L[2 * i + 1, i], L[2 * i + 1, i + 1], L[2 * i + 2, i], L[2 * i + 2, i + 1] = 0.75, 0.25, 0.25, 0.75
    w = torch.tensor([1.40625, -0.5625, 0.15625], dtype=torch.float64)
    L[0, :3], L[-1, -3:] = w, w.flip(0)
    return L.to(_device())


def _exact_adaptive(case, f, r):
    """The four-to-one merges of the tree with dense matrices, level by level."""
    N, k, lam, (xl, xu, yl, yu) = case["N"], case["k"], case["lam"], _bounds(case)
    leaves = _leaves(case["mesh"], case["level"], N)
    f = f.reshape(k, len(leaves), N, N)
    at = {q: i for i, q in enumerate(leaves)}
    T, h, S, w, size, groups = {}, {}, {}, {}, {}, []
    eye = torch.eye(4 * N, dtype=torch.float64, device=_device()).reshape(4 * N, 4, N)
    by_level = {}
    for q in leaves:
        by_level.setdefault(q[0], []).append(q)
    step = {l: ((xu - xl) / 2 ** l / N, (yu - yl) / 2 ** l / N) for l in range(max(by_level) + 1)}

    def leaf(b, g, l):
        dx, dy = step[l]
        return _separable(_boundary_terms(b, g, 1 / dx ** 2, 1 / dy ** 2), dx, dy, lam)

    for l, qs in by_level.items():
        Tl = _neumann(leaf(torch.zeros(4 * N, N, N, dtype=torch.float64, device=_device()), eye, l), eye, *step[l])
        Tl = Tl.reshape(4 * N, 4 * N).T.contiguous()
        z = torch.zeros(k, len(qs), 4, N, dtype=torch.float64, device=_device())
        hl = _neumann(leaf(f[:, [at[q] for q in qs]], z, l), z, *step[l])
        for i, q in enumerate(qs):
            T[q], h[q], size[q] = Tl, hl[:, i], N
    for l in range(max(by_level), 0, -1):
        nodes = {}
        for (_, x, y) in sorted({(l, q[1] // 2, q[2] // 2) for q in size if q[0] == l}):
            ch = [(l, 2 * x + c % 2, 2 * y + c // 2) for c in range(4)]
            nodes.setdefault(min(size[c] for c in ch), []).append(((l - 1, x, y), ch))
        for n, items in nodes.items():
            for _, ch in items:
                for c in ch:
                    m = size[c]
                    Tc = T[c].reshape(4, m, 4, m)
                    while m > n:
                        Tc = torch.einsum("ij,ajbk,kl->aibl", _halve(m), Tc, _double(m))
                        h[c] = h[c] @ _halve(m).T
                        m //= 2
                    T[c] = Tc.reshape(4 * n, 4 * n)
            B = len(items)
            Tc = torch.stack([torch.stack([T[c] for c in ch]) for _, ch in items]).reshape(B, 4, 4, n, 4, n)
            hc = torch.stack([torch.stack([h[c] for c in ch]) for _, ch in items])  # [B, 4, k, 4, n]
            K = torch.zeros(B, 4, 4, n, 12, n, dtype=torch.float64, device=_device())
            for c in range(4):
                K[:, c, :, :, list(_BLOCK[c])] = Tc[:, c]
            jump = lambda v: torch.stack([v[:, c2, s2] - v[:, c1, s1] for (c1, s1), (c2, s2) in _IFACE], 1)
            outer = lambda v: torch.stack([v[:, c, s] for c, s in _OUTER], 1)
            J, O = jump(K).reshape(B, 4 * n, 12 * n), outer(K).reshape(B, 8 * n, 12 * n)
            hv = hc.permute(0, 1, 3, 4, 2)  # [B, child, side, n, k]
            rhs = torch.cat([J[:, :, 4 * n:], jump(hv).reshape(B, 4 * n, k)], 2)
            sol = -torch.linalg.solve(J[:, :, :4 * n].cpu(), rhs.cpu()).to(rhs.device)
            Sg, wg = sol[:, :, :8 * n], sol[:, :, 8 * n:]
            Tg = O[:, :, 4 * n:] + O[:, :, :4 * n] @ Sg
            hg = outer(hv).reshape(B, 8 * n, k) + O[:, :, :4 * n] @ wg
            for i, (q, ch) in enumerate(items):
                T[q], S[q], w[q], size[q] = Tg[i], Sg[i], wg[i], 2 * n
                h[q] = hg[i].T.reshape(k, 4, 2 * n)
            groups.append((n, items))
    g = {(0, 0, 0): r.reshape(k, 4, -1)}
    for n, items in reversed(groups):
        for q, ch in items:
            gq = g[q].reshape(k, 8 * n)
            blocks = torch.cat([gq @ S[q].T + w[q].T, gq], 1).reshape(k, 12, n)
            for c, key in enumerate(ch):
                v, m = blocks[:, list(_BLOCK[c])], n
                while m < size[key]:
                    m *= 2
                    v = v @ _double(m).T
                g[key] = v
    u = torch.empty_like(f)
    for l, qs in by_level.items():
        ids = [at[q] for q in qs]
        u[:, ids] = leaf(f[:, ids], torch.stack([g[q] for q in qs], 1), l)
    return u.reshape(k, len(leaves), N * N)


def _exact_loads(case, seed, M):
    """Gaussians at the cell centres, Fourier modes at the root's boundary points."""
    p = torch.as_tensor(_serve_params(case, seed), device=_device()).reshape(-1, 16, 4)
    x, y = _centres(_leaf_bounds(case), case["N"])
    X, Y = _root_points(case, M)
    f = r = 0.0
    for q in range(8):
        amp, cx, cy, w = (p[:, q, c].reshape(-1, 1, 1, 1) for c in range(4))
        w = torch.where(amp != 0, w, torch.ones_like(w))
        f = f + amp * torch.exp(-((x - cx) ** 2 + (y - cy) ** 2) / (2 * w * w))
        a, kx, ky, phi = (p[:, 8 + q, c].reshape(-1, 1) for c in range(4))
        r = r + a * torch.cos(kx * X + ky * Y + phi)
    return f.reshape(case["k"], -1, case["N"] ** 2), r


def exact(case, seed):
    if case["kind"] == "patch":
        return _exact_patch(case, seed)
    M = _merges(case["mesh"], case["level"], case["N"])[1]
    f, r = _exact_loads(case, seed, M) if case["kind"] == "serve" else _mesh_inputs(case, M, seed)
    u = _exact_uniform(case, f, r, seed) if case["mesh"] == "uniform" else _exact_adaptive(case, f, r)
    return dict(f=f, r=r, u=u) if case["kind"] == "serve" else u.cpu().numpy() if case["kind"] == "driver" else u
