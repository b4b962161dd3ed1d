"""Restriction and prolongation inside the sweeps of a level launched on its own (GPU).

Where two levels or more lie above the one-workgroup cycle, the lane-split residual also
restricts and the first sweep after a prolongation forms the prolonged iterate as it reads
it.  The boxes give such levels full stencils (3D, 2D) and stencils narrower than 3 along
an axis, with clipped children on both ends (odd and even first cells).  The assembled
form is bit-identical to the oracle; the factored one, whose sums are associated
differently, to the same solve with a thread per row and launches of their own for the
transfers (LaneRowsMax 0), FP64 and mixed.
"""
import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import abi
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu

BOXES = [
    (44, 40, 42),   # 13 x 12 x 13 cells or so: levels 0 and 1 on their own
    (190, 4, 90),   # 2 cells or fewer along y
    (151, 149),     # 2D: levels 0 and 1
    (3, 5000),      # 2D: one or two cells wide
]


@pytest.mark.parametrize("n", BOXES, ids=lambda n: "x".join(map(str, n)))
def test_fused_transfers(n):
    p, g = pool(n)
    p.cr_tolerance = 1e-12
    print("[mgfused] %s np=%d" % (n, g.np), flush=True)
    orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
    with Scene(p, g) as s:
        a, b = s.step(1), orc.step(1)
        assert a.cr_iterations == b.cr_iterations
        assert (a.rr0, a.rr, a.rs0, a.rs) == (b.rr0, b.rr, b.rs0, b.rs)
        v = s.read("Velocity")
    assert np.array_equal(v.view(np.int64), orc.read("Velocity").view(np.int64))
    for precision in (abi.PRECISION_FP64, abi.PRECISION_MIXED):
        q = p.copy()
        q.operator_form = abi.OPERATOR_FACTORED
        q.precision = precision
        got = []
        for rows in (None, 0):
            with Scene(q, g) as f:
                if rows is not None:
                    f.set_option("LaneRowsMax", rows)
                st = f.step(1)
                got.append((st.cr_iterations, st.rr, f.read("Velocity").view(np.int64)))
        assert got[0][:2] == got[1][:2]
        assert np.array_equal(got[0][2], got[1][2])
