"""GPU: a mesh moved between steps. The reassembly keeps the start points of its walks in the idle
population buffer: it must leave the populations that the next step reads, whichever of the two
buffers holds them, and the step after it must be that of a context made on the moved mesh.

All values pass through unchanged, so everything is compared bit for bit (uploads are exact in FP64;
FP32 and compressible contexts are compared with a context that moved before it was given the state).
"""
import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import perturbed_vertices

pytestmark = pytest.mark.gpu


def _mesh(N, seed):
    return perturbed_vertices(len(N), N, [0] * len(N), [0.5 * n for n in N], amplitude=0.08, seed=seed)


def _solver(stencil, p, N, precision, walls, seed):
    comp = stencil == "D2Q25H"
    D = len(N)
    kw = dict(compressible=True, gamma=1.4) if comp else {}
    return nat.Solver(stencil, p, N, _mesh(N, seed), cartesian=False, precision=precision,
                      periodic=([1, 0, 1] if walls else [1, 1, 1])[:D], scaling=2.0 if comp else 20.0, viscosity=0.05,
                      cfl=0.4, wall_velocity={3: [0.05] + [0.0] * (D - 1)} if walls else {}, **kw)


def _init(g, comp):
    x = g.coords()
    L = x.max(axis=0)
    rho = 1 + 0.05 * np.cos(2 * np.pi * x[:, 0] / L[0])
    u = 0.1 * np.sin(2 * np.pi * x.T[::-1][:g.D] / L[0])
    g.init_equilibrium(rho, u, 1 + 0.1 * np.cos(2 * np.pi * x[:, 1] / L[1]) if comp else None)
    g.collide()


def _state(g):
    return [g.download_f()] + ([g.download_g()] if g.compressible else [])


@pytest.mark.parametrize("steps", [0, 1, 4, 5])
@pytest.mark.parametrize("stencil,p,N,precision,walls", [
    ("D2Q9", 4, [8, 7], "fp32", True),
    ("D2Q9", 2, [13, 9], "fp64", False),
    ("D3Q19", 2, [6, 5, 4], "fp64", True),
    ("D3Q27", 3, [3, 4, 3], "fp32", False),
    ("D2Q25H", 2, [12, 9], "fp64", True),
    ("D2Q25H", 3, [7, 9], "fp32", False),
])
def test_step_move_step(stencil, p, N, precision, walls, steps):
    comp = stencil == "D2Q25H"
    a = _solver(stencil, p, N, precision, walls, 3)
    _init(a, comp)
    dt = a.dt
    if steps:
        a.step(steps)
    before = _state(a)
    a.set_vertices(_mesh(N, 4))
    for x, y in zip(before, _state(a)):
        np.testing.assert_array_equal(x, y)
    # b: on the moved mesh from the start, brought to the same state by the same steps
    b = _solver(stencil, p, N, precision, walls, 3)
    b.set_vertices(_mesh(N, 4))
    b.set_vertices(_mesh(N, 3))
    _init(b, comp)
    if steps:
        b.step(steps)
    c = _solver(stencil, p, N, precision, walls, 4)
    c.set_dt(dt)
    b.set_vertices(_mesh(N, 4))
    for n in (1, 3):
        a.step(n)
        b.step(n)
        for x, y in zip(_state(a), _state(b)):
            assert np.isfinite(x).all()
            np.testing.assert_array_equal(x, y)
    if precision == "fp64":
        c.upload_f(before[0])
        if comp:
            c.upload_g(before[1])
        c.step(1)
        c.step(3)
        for x, y in zip(_state(a), _state(c)):
            np.testing.assert_array_equal(x, y)
