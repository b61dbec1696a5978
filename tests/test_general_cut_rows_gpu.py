"""Rows of the general SL operator under the reference's cut-off (|w| < 1e-10 dropped,
advection/SemiLagrangianTools.cpp:15-64), which waves sum in two ways: a few such rows together,
a term per lane, or each lane its own row.

The size of the distortion sets how many of a wave's lanes have such a row: none moved (every lane
of the directions along an axis, and whole planes of zero weights), 1e-6 h (most lanes), 1e-3 and
0.1 h (a few). Orders 1-6, 2D and 3D, mesh sizes that leave partial blocks. FP64: every population
within 1e-12 of the oracle after each of 4 steps. FP32 storage: eight and sixteen waves per block,
which sum different numbers of rows together, agree bit for bit.
"""
import math

import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import lbm_parameters, perturbed_vertices, tgv2d_fields, tgv3d_fields
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu


def _mesh(N, amplitude):
    L = 2 * math.pi
    return perturbed_vertices(len(N), N, [0] * len(N), [L] * len(N), amplitude=amplitude, seed=8)


def _fields(x, cs):
    return tgv2d_fields(x, 0.01, cs) if x.shape[1] == 2 else tgv3d_fields(x, cs)


@pytest.mark.parametrize("amplitude", [0.0, 1e-6, 1e-3, 0.1])
@pytest.mark.parametrize("stencil,p,N", [("D3Q19", 1, [4, 5, 3]), ("D3Q27", 2, [3, 4, 3]), ("D3Q19", 3, [4, 3, 3]),
                                         ("D3Q19", 4, [3, 2, 2]), ("D3Q19", 6, [2, 2, 2]), ("D2Q9", 3, [7, 5]),
                                         ("D2Q9", 6, [4, 3])])
def test_cut_rows_against_oracle(stencil, p, N, amplitude):
    cs, s = lbm_parameters(1.0, 0.05)
    v = _mesh(N, amplitude)
    kw = dict(cartesian=False, scaling=s, viscosity=0.01, cfl=0.4)
    g = nat.Solver(stencil, p, N, v, backend="general", **kw)
    o = Oracle(stencil, p, N, v, **kw)
    o.assemble()
    rho, u = _fields(g.coords(), cs)
    for x in (g, o):
        (x.init_equilibrium if x is g else x.init)(rho, u)
        x.collide()
    for step in range(4):
        g.step(1)
        o.steps(1)
        fo = o.get_f()
        e = float(np.abs(g.download_f() - fo).max() / np.abs(fo).max())
        assert e < 1e-12, (step, e)


@pytest.mark.parametrize("amplitude", [0.0, 1e-3, 0.1])
@pytest.mark.parametrize("stencil,p,N", [("D3Q27", 3, [5, 4, 3]), ("D3Q19", 4, [3, 3, 2]), ("D3Q19", 6, [2, 2, 2])])
def test_forms_agree_on_cut_rows(stencil, p, N, amplitude):
    cs, s = lbm_parameters(1.0, 0.05)
    out = []
    for form in (0, 1):
        g = nat.Solver(stencil, p, N, _mesh(N, amplitude), cartesian=False, scaling=s, viscosity=0.01, cfl=0.4,
                       backend="general", precision="fp32")
        g.set_general_form(form)
        g.init_equilibrium(*_fields(g.coords(), cs))
        g.collide()
        g.step(6)
        out.append(g.download_f())
    np.testing.assert_array_equal(out[0], out[1])
