"""GPU: the pairwise upwind SEDG stage kernel at the edges of its launches and rules.

Against the oracle: blocks that are not full and grids that 8 does not divide (the XCD regrouping
keeps the last ones), one to two cells per axis (a cell that is its own neighbour), every order,
walls on all axes, both precisions. Tolerances: FP64 populations 1e-12 of the largest value after
each of two steps; FP32 stores shifted populations and RK registers, two roundings of 2^-24 per
stage of values below 0.2, times the growth of the upwind operator over a stage (below 3): 10
stages stay below 1e-5 of the largest value.

Beyond the Infinity Cache (256 MiB) the kernel keeps the launch order and streams its stores: a
periodic tiling of a small mesh must reproduce the small mesh in every tile (the cells' Jacobians
agree to rounding, so 1e-12 again).
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import box_vertices, perturbed_vertices
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _fields(x, L):
    D = len(L)
    k = [2 * math.pi / L[d] for d in range(D)]
    rho = 1 + 0.02 * np.cos(k[0] * x[:, 0]) * np.cos(k[1] * x[:, 1])
    u = np.stack([0.1 * np.sin(k[(d + 1) % D] * x[:, (d + 1) % D] + d) for d in range(D)])
    return rho, u


@pytest.mark.parametrize("stencil,p,N,precision,closed", [
    ("D2Q9", 1, [1, 2], "fp64", False),
    ("D2Q9", 2, [29, 9], "fp32", False),
    ("D2Q9", 2, [57, 4], "fp64", True),
    ("D2Q9", 3, [17, 1], "fp64", False),
    ("D2Q9", 5, [8, 9], "fp32", True),
    ("D2Q9", 6, [11, 5], "fp64", False),
    ("D3Q19", 1, [5, 3, 9], "fp64", True),
    ("D3Q19", 2, [1, 4, 5], "fp32", False),
    ("D3Q19", 3, [3, 5, 1], "fp32", False),
    ("D3Q19", 3, [3, 2, 3], "fp32", True),
    ("D3Q19", 4, [2, 3, 3], "fp64", True),
    ("D3Q27", 1, [7, 3, 2], "fp32", True),
    ("D3Q27", 3, [1, 2, 5], "fp64", False),
    ("D3Q27", 4, [2, 1, 3], "fp32", False),
])
def test_pair_stage_edges(stencil, p, N, precision, closed):
    D = len(N)
    L = [0.5 * n for n in N]
    v = perturbed_vertices(D, N, [0] * D, L, amplitude=0.1, seed=3) if min(N) > 1 else box_vertices(D, N, [0] * D, L)
    walls = {2 * a + s: [0.02 * (s + 1) * (d != a) for d in range(D)] for a in range(D) for s in (0, 1)}
    kw = dict(cartesian=False, periodic=[0 if closed else 1] * D, scaling=20.0, viscosity=0.05, cfl=0.4,
              scheme="SEDG", wall_velocity=walls if closed else {})
    g = nat.Solver(stencil, p, N, v, precision=precision, **kw)
    o = Oracle(stencil, p, N, v, **kw)
    o.assemble()
    rho, u = _fields(g.coords(), L)
    g.init_equilibrium(rho, u)
    o.init(rho, u)
    g.collide()
    o.collide()
    tol = 1e-12 if precision == "fp64" else 1e-5
    for _ in range(2):
        g.step(1)
        o.steps(1)
        a, b = g.download_f(), o.get_f()
        assert np.abs(a - b).max() <= tol * np.abs(b).max()


@pytest.mark.parametrize("stencil,p,N,tiles", [
    ("D3Q19", 3, [7, 7, 7], [3, 3, 3]),   # 270 MB in FP64: just beyond
    ("D2Q9", 2, [31, 33], [12, 12]),      # 286 MB
])
def test_pair_stage_tiled_beyond_cache(stencil, p, N, tiles):
    D = len(N)
    L = [0.5 * n for n in N]
    out = []
    for m in ([1] * D, tiles):
        M, LL = [n * k for n, k in zip(N, m)], [x * k for x, k in zip(L, m)]
        g = nat.Solver(stencil, p, M, box_vertices(D, M, [0] * D, LL), cartesian=False, scaling=20.0, viscosity=0.05,
                       cfl=0.4, scheme="SEDG")
        rho, u = _fields(g.coords(), L)
        g.init_equilibrium(rho, u)
        g.collide()
        g.step(2)
        nl = (p + 1) ** D
        f = g.download_f()
        out.append(f.reshape([f.shape[0]] + M[::-1] + [nl]))
        del g
    small, big = out
    reps = [1] + tiles[::-1] + [1]
    assert np.abs(big - np.tile(small, reps)).max() <= 1e-12 * np.abs(small).max()
