"""The one-workgroup coarse V-cycle at the edges of its row counts (GPU).

The V-cycle's small levels run in one workgroup, one thread per row: up to 512 rows in
3D (a variant for 256 threads, one for 512), up to 1024 in 2D, from level 0 on when the
whole hierarchy fits.  Each fluid box below puts the fused rows at another place of
that range (cells per axis in the comments); a step solved to 1e-8 must be bit-identical
to the oracle's with the same dot-product tree.  The FP32 stencils of mixed precision
take the same kernels: there the solve must meet its stop rule in as many iterations as
the tolerance of the FP64 one needs, and its velocity lie within 1e-6 of it (the bound
of the mixed-precision tests).
"""
import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene

pytestmark = pytest.mark.gpu

L0 = 0.01
BOXES = [
    (5, 4, 5),       # 2 cells per axis and less: stencils narrower than 3
    (24, 6, 4),      # long and thin: one cell deep in z, level 0 fused
    (14, 14, 14),    # about 4 per axis: whole hierarchy within 256 threads
    (17, 17, 17),    # about 5 per axis: within 512 threads
    (19, 21, 17),    # level 0 launched on its own, coarser levels fused
    (29, 8, 33),
    (9, 7),          # 2D: 2-3 cells
    (41, 61),        # 2D: level 0 of about 12 x 18 cells fused (648 rows and more)
    (75, 47),        # 2D: level 0 beyond 1024 rows with its coarser levels
    (3, 120),        # 2D: one cell wide
]


def pool(n):
    dim = len(n)
    inner = list(n)
    inner[-1] += 6
    fluid = scenes.lattice([0] * 3, list(n) + [0] * (3 - dim), L0, dim)
    walls = scenes.box_walls([0] * dim, inner, 4, L0, dim, open_top=True)
    lo = [-9 * L0] * dim + [-0.05] * (3 - dim)
    hi = [(m + 9) * L0 for m in inner] + [0.05] * (3 - dim)
    for d in range(dim):
        w = hi[d] - lo[d]
        if np.ceil(3.5 * L0 / (w / np.floor(w / (3.5 * L0)))) > 1:
            hi[d] += 0.5 * L0
    g = scenes.assemble(fluid, walls, 0.0, L0, lo, hi, 77, dim)
    p = scenes.base_params(dim, 0.1, (0.0, -9.8, 0.0) if dim == 2 else (0.0, 0.0, -9.8), 5.0e-4, 4)
    p.cr_tolerance = 1e-16
    return p, g


@pytest.mark.parametrize("n", BOXES, ids=lambda n: "x".join(map(str, n)))
def test_coarse_cycle_bitwise(n):
    p, g = pool(n)
    print("[coarse] %s np=%d" % (n, g.np), flush=True)
    orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
    with Scene(p, g) as s:
        for _ in range(2):
            a, b = s.step(1), orc.step(1)
            assert a.cr_iterations == b.cr_iterations
            assert (a.rr0, a.rr, a.rs0, a.rs) == (b.rr0, b.rr, b.rs0, b.rs)
        v = s.read("Velocity")
    assert np.array_equal(v.view(np.int64), orc.read("Velocity").view(np.int64))
    p.precision = abi.PRECISION_MIXED
    with Scene(p, g) as m:
        st = m.step(1)
        m.step(1)
        vm = m.read("Velocity")
    assert st.rr / st.rr0 < p.cr_tolerance
    assert np.abs(vm - v).max() <= 1e-6 * np.abs(v).max()
