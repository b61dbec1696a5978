"""GPU: the general SL kernel's form of two waves per 64 DoFs, which is the default from 5/2 blocks
per CU on (256 CUs: 81,921 DoFs in FP64, 163,841 in FP32) in 2D and 3D.

Both forms work on the same departure records with the same sums in the same order, so pinned on
small meshes they must agree bit for bit: every order, both storage precisions, walls, Cartesian
meshes (whole waves of cut-off rows), mesh sizes that leave partial blocks and groups of rows. At
its default sizes the form is held against the oracle in 2D. Tolerances there: FP64 1e-12 of the
largest value after each of two steps; FP32 stores shifted populations, one rounding of 2^-24 per
value and step, amplified by the interpolation by less than 3: two steps stay below 1e-6.
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import perturbed_vertices
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _problem(N, amplitude, closed):
    D = len(N)
    L = [0.5 * n for n in N]
    v = perturbed_vertices(D, N, [0] * D, L, amplitude=amplitude, seed=3)
    kw = dict(cartesian=False, periodic=([1, 0, 1] if closed else [1, 1, 1])[:D], scaling=20.0, viscosity=0.05, cfl=0.4,
              wall_velocity={3: [0.05] + [0.0] * (D - 1)} if closed else {})
    return v, kw


def _fields(x):
    D = x.shape[1]
    k = 2 * math.pi / x.max(axis=0)
    rho = 1 + 0.02 * np.cos(k[0] * x[:, 0]) * np.cos(k[1] * x[:, 1])
    u = np.stack([0.1 * np.sin(k[(d + 1) % D] * x[:, (d + 1) % D] + d) for d in range(D)])
    return rho, u


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("amplitude,closed", [(0.0, True), (0.1, False), (1e-3, True)])
@pytest.mark.parametrize("stencil,p,N", [
    ("D2Q9", 1, [2, 3]), ("D2Q9", 1, [37, 9]), ("D2Q9", 2, [15, 11]), ("D2Q9", 3, [8, 7]), ("D2Q9", 4, [9, 33]),
    ("D2Q9", 5, [5, 6]), ("D2Q9", 6, [4, 5]),
    ("D3Q19", 1, [5, 4, 7]), ("D3Q27", 2, [4, 5, 3]), ("D3Q19", 3, [4, 3, 5]), ("D3Q27", 3, [2, 3, 3]),
    ("D3Q19", 4, [3, 2, 3]), ("D3Q27", 4, [2, 3, 2]), ("D3Q19", 6, [2, 2, 3]), ("D3Q27", 6, [1, 2, 2]),
])
def test_forms_agree(stencil, p, N, precision, amplitude, closed):
    v, kw = _problem(N, amplitude if min(N) > 1 else 0.0, closed)
    out = []
    for form in (0, 1):
        g = nat.Solver(stencil, p, N, v, precision=precision, backend="general", **kw)
        assert g.step_form() == 1
        g.set_step_form(form)
        assert g.step_form() == form
        g.init_equilibrium(*_fields(g.coords()))
        g.collide()
        g.step(4)
        f = g.download_f()
        g.stream()
        out.append((f, g.download_f()) + g.macro()[:2])
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("stencil,p,N,precision,closed", [
    ("D2Q9", 1, [301, 290], "fp64", True),
    ("D2Q9", 2, [205, 202], "fp32", True),
    ("D2Q9", 4, [72, 71], "fp64", True),
    ("D2Q9", 3, [97, 99], "fp64", False),
])
def test_default_sizes_against_oracle(stencil, p, N, precision, closed):
    v, kw = _problem(N, 0.1, closed)
    g = nat.Solver(stencil, p, N, v, precision=precision, backend="general", **kw)
    assert g.step_form() == 0 and g.n > 640 * (256 if precision == "fp32" else 128)
    o = Oracle(stencil, p, N, v, **kw)
    o.assemble()
    rho, u = _fields(g.coords())
    g.init_equilibrium(rho, u)
    o.init(rho, u)
    g.collide()
    o.collide()
    tol = 1e-12 if precision == "fp64" else 1e-6
    for _ in range(2):
        g.step(1)
        o.steps(1)
        a, b = g.download_f(), o.get_f()
        assert np.abs(a - b).max() <= tol * np.abs(b).max()


def test_other_forms_are_refused():
    v, kw = _problem([4, 4], 0.1, False)
    g = nat.Solver("D2Q9", 2, [4, 4], v, backend="general", **kw)
    for form in (-2, 2):
        with pytest.raises(nat.NatError):
            g.set_step_form(form)
