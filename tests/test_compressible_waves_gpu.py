"""GPU: the compressible stream + collide kernel with 8 and with 4 waves per block.

The launch picks 8 waves for grids of about one block (64 DoFs) per CU and 4 above (FP32 other
than p = 3 above 410 blocks), and p = 4 loads a stencil's rows in groups: meshes on both sides of
each line, with a last block that is not full, Cartesian (cut-off terms) and perturbed, with and
without reflected rows, against the FP64 oracle.

Tolerances: FP64 as everywhere, 1e-12 of the largest value after each of two steps. FP32 stores
shifted populations, one rounding of 2^-24 per stored value and step, amplified by the
interpolation by less than 3: 2 steps stay below 1e-6 of the largest value.
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import box_vertices, perturbed_vertices
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,p,precision,perturb,closed", [
    ([2, 2], 1, "fp32", False, True),      # one block, 8 waves
    ([63, 64], 2, "fp64", False, False),   # 252 blocks: 8 waves
    ([65, 64], 2, "fp64", False, True),    # 264 blocks: 4 waves
    ([79, 80], 2, "fp32", True, True),     # 400 blocks: 8 waves
    ([83, 80], 2, "fp32", False, True),    # 420 blocks: 4 waves
    ([131, 128], 1, "fp64", True, False),  # 262 blocks: 4 waves
    ([43, 44], 3, "fp32", False, True),    # 271 blocks: 4 waves
    ([43, 44], 3, "fp64", True, True),
    ([31, 32], 4, "fp32", False, False),   # 248 blocks: 8 waves
    ([33, 34], 4, "fp64", False, True),    # 285 blocks: 4 waves
    ([41, 41], 4, "fp32", True, True),     # 426 blocks: 4 waves
])
def test_compressible_waves(N, p, precision, perturb, closed):
    ext = [n / max(N) for n in N]
    v = perturbed_vertices(2, N, [0, 0], ext, amplitude=0.1, seed=5) if perturb else box_vertices(2, N, [0, 0], ext)
    kw = dict(cartesian=not perturb, periodic=[1, 0] if closed else [1, 1], scaling=2.0, viscosity=1e-2, cfl=0.4,
              compressible=True, gamma=1.4, wall_velocity={3: [0.2, 0.0]} if closed else {})
    g = nat.Solver("D2Q25H", p, N, v, precision=precision, **kw)
    o = Oracle("D2Q25H", p, N, v, **kw)
    o.assemble()
    x = g.coords()
    rho = 1 + 0.2 * np.cos(2 * math.pi * x[:, 0]) * np.cos(math.pi * x[:, 1])
    T = 1 + 0.1 * np.sin(2 * math.pi * x[:, 0]) * np.sin(math.pi * x[:, 1])
    u = np.stack([0.1 * np.sin(math.pi * x[:, 1]), 0.05 * np.sin(2 * math.pi * x[:, 0])])
    g.init_equilibrium(rho, u, T)
    o.init(rho, u, T)
    g.collide()
    o.collide()
    tol = 1e-12 if precision == "fp64" else 1e-6
    for _ in range(2):
        g.step(1)
        o.steps(1)
        for a, b in ((g.download_f(), o.get_f()), (g.download_g(), o.get_g())):
            assert np.abs(a - b).max() <= tol * np.abs(b).max()
