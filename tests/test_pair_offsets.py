"""The bound under which a kernel may read a direction and its opposite at 32-bit byte offsets from
the lower one's array (natrium_amd/csrc/nat_offsets.hpp), compiled with g++ from the kernels' header.

A load of 16 bytes that ends with the last byte of the farther array must keep its offset below
2^32 - 16 (the kernels' out-of-range offset is 2^32 - 1). The stencils' opposite directions are two
arrays apart: three arrays, 178,956,970 FP64 DoFs; one more wraps.
"""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "nat_offsets.hpp"
int main(int argc, char** argv) {
  for (int i = 1; i + 2 < argc; i += 3)
    std::printf("%d\n", (int)nat::pair_offsets_fit(atoll(argv[i]), atoll(argv[i + 1]), atoll(argv[i + 2])));
}
"""


def test_bound_is_where_offsets_wrap(tmp_path):
    src = tmp_path / "po.cpp"
    src.write_text(SRC)
    exe = tmp_path / "po"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "natrium_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    q = []
    for apart in (1, 2, 4):
        for es in (4, 8):
            edge = 2 ** 32 // ((apart + 1) * es)
            q += [(apart, s, es) for s in (1, 128, edge // 2, edge - 8, edge - 4, edge - 2, edge, edge + 1, 2 * edge)]
    q += [(2, 178956969, 8), (2, 178956970, 8), (2, 178956971, 8), (2, 2 ** 28 - 1, 8)]
    out = subprocess.run([str(exe)] + [str(v) for t in q for v in t], check=True, capture_output=True, text=True).stdout
    got = [int(v) for v in out.split()]
    assert len(got) == len(q)
    for (apart, stride, es), fit in zip(q, got):
        end = (apart + 1) * stride * es  # offset just behind the farther array
        assert fit == (end <= 2 ** 32 - 16), (apart, stride, es)
    assert got[-4:] == [1, 1, 0, 0]


@pytest.mark.gpu
@pytest.mark.parametrize("N,p,precision,perturb,closed,prandtl", [
    ([5, 3], 1, "fp32", True, True, 0.0),
    ([9, 7], 2, "fp64", False, True, 0.0),   # cut-off terms, reflected rows
    ([40, 33], 2, "fp32", True, False, 0.71),
    ([67, 65], 2, "fp64", True, True, 0.0),  # 4 waves per block either way
    ([11, 6], 3, "fp64", False, True, 0.71),
    ([8, 9], 4, "fp32", True, True, 0.0),
])
def test_far_form_gives_the_same_bits(N, p, precision, perturb, closed, prandtl):
    """The form with 64-bit addresses, which serves arrays beyond the bound, pinned on small meshes."""
    import natrium_amd as nat
    from natrium_amd.problems import box_vertices, perturbed_vertices

    ext = [n / max(N) for n in N]
    v = perturbed_vertices(2, N, [0, 0], ext, amplitude=0.1, seed=5) if perturb else box_vertices(2, N, [0, 0], ext)
    out = []
    for form in (0, 1):
        g = nat.Solver("D2Q25H", p, N, v, precision=precision, cartesian=not perturb,
                       periodic=[1, 0] if closed else [1, 1], scaling=2.0, viscosity=1e-2, cfl=0.4, compressible=True,
                       gamma=1.4, prandtl=prandtl, wall_velocity={3: [0.2, 0.0]} if closed else {})
        assert g.step_form() == 1
        g.set_step_form(form)
        assert g.step_form(3) == form
        x = g.coords()
        rho = 1 + 0.2 * np.cos(2 * np.pi * x[:, 0]) * np.cos(np.pi * x[:, 1])
        T = 1 + 0.1 * np.sin(2 * np.pi * x[:, 0]) * np.sin(np.pi * x[:, 1])
        u = np.stack([0.1 * np.sin(np.pi * x[:, 1]), 0.05 * np.sin(2 * np.pi * x[:, 0])])
        g.init_equilibrium(rho, u, T)
        g.collide()
        g.step(3)
        g.stream()
        out.append((g.download_f(), g.download_g()) + g.macro())
        with pytest.raises(nat.NatError):
            g.set_step_form(2)
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
