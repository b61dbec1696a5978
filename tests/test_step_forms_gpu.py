"""GPU: which form a run of structured steps takes, and that all forms give the same bits.

Every instantiated tile of the collide-then-stream form is pinned on boxes that are ragged for it
along each axis and held against the fused kernel bit for bit: both do the same FP64 operations in
the same order and round to storage precision at the same places. The rule is asserted on both sides
of each of its lines: short runs on populations of more than 3 MB, boxes too thin for the large
tile, meshes that fill one round of the fused kernel's tiles.
"""
import numpy as np
import pytest

import natrium_amd as nat
from natrium_amd.problems import box_vertices

pytestmark = pytest.mark.gpu


def _solver(stencil, N, p, precision, init=True, stabilizer=False):
    D = len(N)
    g = nat.Solver(stencil, p, N, box_vertices(D, N, [0.0] * D, [0.5 * n for n in N]), scaling=20.0, viscosity=0.01,
                   cfl=0.4, precision=precision, stabilizer=stabilizer)
    assert g.backend_name == "structured"
    if init:
        # every node of the periodic lattice its own velocity, the copies on the upper faces alike
        x = g.coords()
        lim = np.array([0.5 * n for n in N])
        wrapped = np.where(x > lim - 1e-9, 0.0, x)
        u = np.stack([0.05 * np.sin(37.0 * wrapped @ np.arange(1, D + 1) + d) for d in range(D)])
        g.init_equilibrium(np.ones(g.n), u)
        g.collide()
    return g


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("stencil,N,p,tiles", [
    ("D2Q9", [11, 9], 2, (1, 2)),
    ("D2Q9", [5, 6], 3, (1,)),
    ("D2Q9", [9, 5], 4, (1, 2)),
    ("D3Q19", [9, 5, 3], 2, (1, 2)),
    ("D3Q27", [10, 6, 5], 2, (1, 2)),
    ("D3Q19", [5, 3, 3], 3, (1, 2)),
    ("D3Q27", [6, 5, 2], 3, (1, 2)),
    ("D3Q19", [5, 3, 2], 4, (1, 2)),
    ("D3Q27", [3, 3, 3], 4, (1, 2)),
    ("D3Q27", [2, 2, 3], 4, (1, 2)),
])
def test_every_tile_equals_the_fused_kernel(stencil, N, p, tiles, precision):
    if precision == "fp64" and stencil != "D2Q9":
        tiles = (1,)
    if precision == "fp64" and p == 4:
        tiles = (1,)
    stab = stencil == "D3Q19"
    ref = _solver(stencil, N, p, precision, stabilizer=stab)
    ref.set_step_form(0)
    runs = (2, 35, 3)
    want = []
    for n in runs:
        assert ref.step_form(n) == 0
        ref.step(n)
        want.append((ref.download_f(),) + ref.macro()[:2])
    assert np.isfinite(want[-1][0]).all()
    for tile in tiles:
        g = _solver(stencil, N, p, precision, stabilizer=stab)
        g.set_step_form(tile)
        for n, w in zip(runs, want):
            assert g.step_form(n) == tile and g.step_form(1) == 0
            g.step(n)
            for a, b in zip((g.download_f(),) + g.macro()[:2], w):
                np.testing.assert_array_equal(a, b)
        assert g.time == ref.time
    for form in sorted({1, 2, 3} - set(tiles)):
        with pytest.raises(nat.NatError):
            ref.set_step_form(form)


@pytest.mark.parametrize("stencil,N,p,precision,lines", [
    # (steps, form): the form up to that many steps of a run
    ("D2Q9", [8, 8], 4, "fp64", [(1, 0), (1000, 1)]),
    ("D2Q9", [103, 101], 4, "fp32", [(15, 0), (1000, 2)]),    # 6 MB
    ("D2Q9", [103, 101], 4, "fp64", [(1000, 0)]),
    ("D2Q9", [100, 100], 4, "fp64", [(15, 0), (1000, 1)]),
    ("D2Q9", [150, 140], 2, "fp32", [(5, 0), (1000, 2)]),     # 3.02 MB
    ("D2Q9", [140, 145], 2, "fp32", [(1, 0), (1000, 2)]),     # 2.92 MB
    ("D3Q19", [21, 21, 20], 3, "fp32", [(2, 0), (1000, 2)]),
    ("D3Q19", [21, 21, 20], 3, "fp64", [(2, 0), (1000, 1)]),
    ("D3Q19", [12, 12, 12], 4, "fp32", [(7, 0), (1000, 2)]),
    ("D3Q27", [2, 32, 25], 4, "fp32", [(7, 0), (1000, 1)]),   # half of a large tile would be empty
    ("D3Q27", [16, 16, 16], 4, "fp32", [(95, 0), (1000, 2)]),  # one round of the fused kernel's tiles
    ("D3Q27", [16, 16, 16], 4, "fp64", [(1000, 0)]),
    ("D3Q19", [16, 16, 16], 4, "fp32", [(1000, 0)]),
    ("D3Q19", [17, 14, 17], 4, "fp32", [(7, 0), (1000, 2)]),  # fewer cells, but 315 of those tiles
    ("D3Q27", [32, 32, 32], 2, "fp32", [(95, 0), (1000, 2)]),
    ("D3Q27", [32, 32, 32], 2, "fp64", [(1000, 0)]),
    ("D3Q27", [33, 31, 30], 2, "fp64", [(7, 0), (1000, 1)]),
    ("D2Q9", [6, 6], 6, "fp64", [(1000, 0)]),
    ("D3Q19", [6, 6, 6], 1, "fp32", [(1000, 0)]),
])
def test_rule(stencil, N, p, precision, lines):
    g = _solver(stencil, N, p, precision, init=False)
    at = 1
    for steps, form in lines:
        assert g.step_form(at) == form and g.step_form(steps) == form, (at, steps, form)
        at = steps + 1
    for form in (0, -1):
        g.set_step_form(form)
        assert g.step_form(1000) == (0 if form == 0 else lines[-1][1])


def test_autotuned_form_is_what_a_run_takes():
    """A box on which the rule keeps the fused kernel and the other form is 30% faster: the tuner
    moves its runs, a second context of the size gets the choice without timing, and neither the
    state at the time nor the results depend on it."""
    N, p = [44, 44, 44], 2
    a, b, c = (_solver("D3Q19", N, p, "fp64", init=init) for init in (True, True, False))
    assert a.step_form(1000) == 0
    f0, t0 = a.download_f(), a.time
    tile = a.autotune(10)
    assert tile == a.struct_tile()
    np.testing.assert_array_equal(a.download_f(), f0)
    assert a.time == t0
    assert a.step_form(1000) == 1 and a.step_form(1) == 0 and b.step_form(1000) == 0
    assert c.autotune(10) == tile and c.step_form(1000) == 1
    a.step(9)
    b.step(9)
    np.testing.assert_array_equal(a.download_f(), b.download_f())
    a.set_step_form(0)  # a pinned form stands above the tuned one
    assert a.step_form(1000) == 0
    a.set_step_form(-1)
    assert a.step_form(1000) == 1
