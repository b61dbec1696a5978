"""GPU: departure records after a mesh move equal those of a context made on the moved mesh.

The walks of all directions start from unit coordinates found once per DoF, kept in the idle
population buffer: block remainders, long walks (several cells), walls, Cartesian cells. Both sides
run the same kernels on the same numbers, so the populations are equal bit for bit; the FP64 ones
are held against the oracle as well (1e-12 of the largest value).
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import box_vertices, perturbed_vertices
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stencil,p,N,precision,walls,amplitude,cfl", [
    ("D2Q9", 1, [3, 2], "fp64", False, 0.1, 0.4),
    ("D2Q9", 4, [8, 7], "fp32", True, 0.1, 0.4),
    ("D2Q9", 2, [31, 9], "fp64", True, 0.03, 4.0),
    ("D2Q9", 3, [10, 9], "fp64", False, 0.0, 3.0),
    ("D3Q19", 2, [5, 4, 3], "fp64", False, 0.1, 0.4),
    ("D3Q19", 2, [6, 5, 4], "fp32", True, 0.02, 3.0),
    ("D3Q27", 3, [3, 3, 2], "fp64", True, 0.05, 1.0),
    ("D3Q27", 1, [6, 5, 7], "fp32", False, 0.1, 0.4),
])
def test_moved_mesh_equals_fresh_context(stencil, p, N, precision, walls, amplitude, cfl):
    D = len(N)
    hi = [1.0 * n for n in N]
    grow = [1.25 * n for n in N]

    def mesh(seed, h):
        if amplitude == 0.0:
            return box_vertices(D, N, [0] * D, h)
        return perturbed_vertices(D, N, [0] * D, h, amplitude=amplitude, seed=seed)

    kw = dict(cartesian=amplitude == 0.0, periodic=[0 if walls else 1] + [1] * (D - 1), scaling=20.0, viscosity=0.05,
              cfl=cfl, wall_velocity={0: [0.0] + [0.05] * (D - 1), 1: [0.0] * D} if walls else {})
    moved = nat.Solver(stencil, p, N, mesh(3, hi), precision=precision, backend="general", **kw)
    fresh = nat.Solver(stencil, p, N, mesh(4, grow), precision=precision, backend="general", **kw)
    oracle = Oracle(stencil, p, N, mesh(4, grow), **kw)
    moved.set_vertices(mesh(4, grow))
    moved.set_dt(fresh.dt)
    moved.set_vertices(mesh(4, grow))  # the records of the last call are the ones in use
    oracle.assemble()
    x = fresh.coords()
    assert np.array_equal(moved.coords(), x)
    rho = 1 + 0.01 * np.cos(2 * math.pi * x[:, 0] / grow[0])
    u = 0.1 * np.sin(2 * math.pi * x.T[::-1] / grow[0])
    for s in (moved, fresh):
        s.init_equilibrium(rho, u)
        s.collide()
        s.step(2)
    oracle.init(rho, u)
    oracle.collide()
    oracle.steps(2)
    f = fresh.download_f()
    assert np.array_equal(moved.download_f(), f)
    tol = 1e-12 if precision == "fp64" else 1e-6
    assert np.abs(f - oracle.get_f()).max() <= tol * np.abs(f).max()
