"""GPU: a broken value in the upwind SEDG step goes where the upwind flux takes it, and nowhere else.

A face is upwind for one of two opposite directions; the other one must not read it. Streaming
couples the directions at walls only, so with one direction infinite everywhere all others must
stream as if it were not there, and with walls its opposite only within five cells (one per
Runge-Kutta stage) of the wall that it runs into.

The pairwise stage kernel against the kernel that takes one direction at a time: the same bits, with
and without walls, and the same non-finite values where the state is broken.
"""
import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import perturbed_vertices

pytestmark = pytest.mark.gpu

OPPOSITE = {9: [0, 3, 4, 1, 2, 7, 8, 5, 6]}


def _solver(stencil, p, N, precision, closed, form=-1):
    D = len(N)
    L = [0.5 * n for n in N]
    v = perturbed_vertices(D, N, [0] * D, L, amplitude=0.1, seed=3)
    walls = {2 * a + s: [0.02 * (s + 1) * (d != a) for d in range(D)] for a in range(D) for s in (0, 1)}
    per = [1, 0, 1][:D] if closed else [1] * D
    g = nat.Solver(stencil, p, N, v, cartesian=False, periodic=per, scaling=20.0, viscosity=0.05, cfl=0.4,
                   scheme="SEDG", precision=precision,
                   wall_velocity={f: w for f, w in walls.items() if f in (2, 3)} if closed else {})
    g.set_step_form(form)
    assert g.step_form() == (form if form >= 0 else 1)
    x = g.coords()
    rho = 1 + 0.02 * np.cos(2 * np.pi * x[:, 0] / L[0]) * np.cos(2 * np.pi * x[:, 1] / L[1])
    u = np.stack([0.1 * np.sin(2 * np.pi * x[:, (d + 1) % D] / L[(d + 1) % D] + d) for d in range(D)])
    g.init_equilibrium(rho, u)
    g.collide()
    return g


def _streamed(g, al=None):
    f = g.download_f()
    if al is not None:
        f = f.copy()
        f[al] = np.inf
    g.upload_f(f)
    g.stream()
    return g.download_f()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("stencil,p,N", [("D2Q9", 2, [5, 4]), ("D3Q19", 3, [3, 2, 3]), ("D3Q27", 1, [3, 4, 2])])
def test_infinite_direction_leaves_the_others(stencil, p, N, precision):
    clean = _streamed(_solver(stencil, p, N, precision, False))
    assert np.isfinite(clean).all()
    for al in range(1, clean.shape[0], 3):
        broken = _streamed(_solver(stencil, p, N, precision, False), al)
        rest = [q for q in range(clean.shape[0]) if q != al]
        np.testing.assert_array_equal(broken[rest], clean[rest])


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_infinite_direction_at_walls(precision):
    p, N = 2, [3, 9]
    nodes = N[0] * (p + 1) ** 2  # DoFs of a row of cells
    clean = _streamed(_solver("D2Q9", p, N, precision, True))
    for al, up in ((2, True), (4, False), (5, True), (8, False)):  # towards the upper wall, or the lower
        broken = _streamed(_solver("D2Q9", p, N, precision, True), al)
        op = OPPOSITE[9][al]
        for q in range(9):
            if q == al:
                continue
            far = slice(None) if q != op else (slice(0, 4 * nodes) if up else slice(5 * nodes, None))
            np.testing.assert_array_equal(broken[q, far], clean[q, far])
            if q == op:
                assert not np.isfinite(broken[q]).all()  # the reflected values are broken indeed


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("closed", [False, True])
@pytest.mark.parametrize("stencil,p,N", [("D2Q9", 1, [9, 7]), ("D2Q9", 3, [7, 5]), ("D2Q9", 6, [3, 4]),
                                         ("D3Q19", 2, [4, 3, 5]), ("D3Q19", 3, [3, 4, 2]), ("D3Q27", 3, [2, 3, 3]),
                                         ("D3Q27", 4, [2, 2, 3])])
def test_pairs_equal_one_direction_at_a_time(stencil, p, N, precision, closed):
    out = []
    for form in (0, 1):
        g = _solver(stencil, p, N, precision, closed, form)
        g.step(2)
        g.stream()
        fine = g.download_f()
        f = fine.copy()
        f[3, g.n // 2] = np.inf
        f[6, g.n // 3] = np.nan
        g.upload_f(f)
        g.stream()
        out.append((fine, g.download_f()))
    assert np.isfinite(out[0][0]).all() and not np.isfinite(out[0][1]).all()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_central_flux_has_one_form():
    g = nat.Solver("D2Q9", 2, [4, 4], perturbed_vertices(2, [4, 4], [0, 0], [1, 1], amplitude=0.0, seed=1),
                   scaling=20.0, viscosity=0.05, cfl=0.4, scheme="SEDG_CENTRAL")
    assert g.step_form() == 0
    g.set_step_form(0)
    with pytest.raises(nat.NatError):
        g.set_step_form(1)
