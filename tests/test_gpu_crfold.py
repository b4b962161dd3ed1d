"""Dot products folded where they are read, at the edges of their chunk counts (GPU).

rho = s.y and tmp = q.u of a CR iteration are sums over chunks of 256 particles.  Scenes
of up to 1024 chunks fold them in the kernels that read them, larger ones reduce them in
a launch: one full chunk, two, 257 (a lane's second partial), 1024 full, and one more.
The fold keeps the dot-product tree, so a step is bit-identical to the oracle's.
"""
import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import scenes
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import L0

pytestmark = pytest.mark.gpu


def pool(nx, ny):
    fluid = scenes.lattice([0] * 3, [nx, ny, 0], L0, 2)
    walls = scenes.box_walls([0] * 2, [nx, ny + 6], 4, L0, 2, open_top=True)
    lo = [-9 * L0] * 2 + [-0.05]
    hi = [(nx + 9.5) * L0, (ny + 15.5) * L0, 0.05]
    g = scenes.assemble(fluid, walls, 0.0, L0, lo, hi, 5, 2)
    p = scenes.base_params(2, 0.1, (0.0, -9.8, 0.0), 5.0e-4, 4)
    p.cr_tolerance = 1e-4
    return p, g


@pytest.mark.parametrize("n", [(16, 16), (16, 17), (257, 256), (512, 512), (512, 513)], ids=lambda n: "%dx%d" % n)
def test_folded_dots_bitwise(n):
    p, g = pool(*n)
    print("[crfold] %dx%d np=%d" % (n + (g.np,)), flush=True)
    orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
    with Scene(p, g) as s:
        a, b = s.step(1), orc.step(1)
        assert a.cr_iterations == b.cr_iterations >= 3
        assert (a.rr0, a.rr, a.rs0, a.rs) == (b.rr0, b.rr, b.rs0, b.rs)
        v = s.read("Velocity")
    assert np.array_equal(v.view(np.int64), orc.read("Velocity").view(np.int64))
