"""Runs of several steps of a structured context (collide-then-stream launches) against the same
steps taken one at a time (one fused stream-then-collide launch each).

The two forms do the same FP64 operations in the same order and round to storage precision at the
same places, so populations and fields are compared bit for bit. Sizes: fewer cells than a tile,
whole tiles, and one cell more along each axis (ragged tiles); every stencil, order and storage
precision of the form, the stabilizer, and more steps than one captured chunk.
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import box_vertices, lbm_parameters, tgv2d_fields, tgv3d_fields

pytestmark = pytest.mark.gpu


def _solver(stencil, N, p, precision, stabilizer=False):
    D = len(N)
    cs, s = lbm_parameters(1.0, 0.1)
    h = 2 * math.pi / N[0]
    v = box_vertices(D, N, [0.0] * D, [h * n for n in N])
    g = nat.Solver(stencil, p, N, v, scaling=s, viscosity=0.01, cfl=0.4, precision=precision, stabilizer=stabilizer)
    assert g.backend_name == "structured"
    x = g.coords()
    rho, u = tgv2d_fields(x, 0.01, cs) if D == 2 else tgv3d_fields(x, cs)
    rng = np.random.default_rng(5)  # periodic noise: all directions of all nodes differ
    k = rng.integers(1, 4, size=(6, D)) * np.array([2 * math.pi / (h * n) for n in N])
    ph = rng.uniform(0, 2 * math.pi, size=6)
    u = u + 0.05 * sum(np.sin(x @ k[i] + ph[i]) for i in range(6))
    g.init_equilibrium(rho, u)
    g.collide()
    return g


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("stencil,N,p,steps,stab", [
    ("D2Q9", [4, 4], 2, 3, False),
    ("D2Q9", [9, 5], 2, 37, True),
    ("D2Q9", [130, 128], 2, 2, False),   # large tile
    ("D2Q9", [3, 2], 3, 5, True),
    ("D2Q9", [5, 9], 3, 4, False),
    ("D2Q9", [3, 5], 4, 70, False),
    ("D2Q9", [103, 101], 4, 2, True),    # large tile (FP32)
    ("D3Q19", [2, 3, 2], 2, 3, True),
    ("D3Q27", [5, 3, 3], 2, 34, False),
    ("D3Q27", [27, 25, 26], 2, 2, False),
    ("D3Q27", [31, 31, 30], 2, 2, False),  # large tile (FP32)
    ("D3Q19", [34, 33, 31], 2, 2, True),   # small tile past one round (FP64)
    ("D3Q27", [16, 16, 16], 4, 96, False),  # exactly one round of the fused kernel: long runs only (FP32)
    ("D3Q19", [11, 11, 11], 4, 2, False),  # small tile (FP64), large (FP32)
    ("D3Q19", [4, 2, 2], 3, 3, False),
    ("D3Q27", [5, 3, 2], 3, 3, False),
    ("D3Q19", [21, 21, 20], 3, 2, True),   # large tile (FP32)
    ("D3Q27", [2, 2, 2], 4, 3, False),
    ("D3Q19", [3, 3, 2], 4, 35, True),
    ("D3Q27", [13, 11, 9], 4, 2, False),   # large tile (FP32)
])
def test_runs_equal_single_steps(stencil, N, p, steps, stab, precision):
    a = _solver(stencil, N, p, precision, stab)
    b = _solver(stencil, N, p, precision, stab)
    for n in (steps, 2):  # a second run starts from the other buffer where steps is odd
        a.step(n)
        for _ in range(n):
            b.step(1)
        np.testing.assert_array_equal(a.download_f(), b.download_f())
        for x, y in zip(a.macro()[:2], b.macro()[:2]):
            np.testing.assert_array_equal(x, y)
    assert a.time == b.time


def test_low_density_is_reported_by_a_run():
    g = _solver("D2Q9", [4, 4], 2, "fp64")
    f = g.download_f()
    g.upload_f(f * 1e-12)
    with pytest.raises(nat.DensityZeroError):
        g.step(4)
