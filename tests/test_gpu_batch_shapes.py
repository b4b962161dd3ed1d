"""Batches whose members take different routes through one iteration (GPU).

Members of up to 262,144 fluid particles (1024 chunks) fold rho and tmp where they are read,
larger ones reduce them.  The cell-staged pass launches once per shape: 3D cells, 3D cells
of more records than two workgroups of a CU hold, 2D cells, and 2D cells of a large radius
in the first of these shapes.  Every member has the bits of its scene alone.
"""
import numpy as np
import pytest

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Batch, Scene
from test_gpu_coarse import pool
from test_gpu_faccells import wide

pytestmark = pytest.mark.gpu

MEMBERS = {
    "fold": [lambda: pool((520, 510)), lambda: pool((40, 41)), lambda: pool((10, 9, 11))],
    "shapes": [lambda: pool((13, 11, 9)), lambda: scenes.periodic_3d(n=13, depth=12), lambda: pool((23, 17)),
               lambda: wide((60, 50), 8.0)],
}


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED])
@pytest.mark.parametrize("name", list(MEMBERS))
def test_members_as_alone(name, precision):
    steps = 2
    made = []
    for make in MEMBERS[name]:
        p, g = make()
        p.operator_form = abi.OPERATOR_FACTORED
        p.precision = precision
        p.cr_tolerance = 1e-12
        p.end_time = 1.0e9
        made.append((p, g))
    print("[batch shapes] %s precision %d: np %s" % (name, precision, [g.np for _, g in made]), flush=True)
    members = [Scene(p, g) for p, g in made]
    with Batch() as b:
        for s in members:
            b.add(s)
        hist = [b.step() for _ in range(steps)]
    for k, (p, g) in enumerate(made):
        with Scene(p, g) as s:
            for t in range(steps):
                st = s.step(1)
                assert (st.cr_iterations, st.rr) == (hist[t][k].cr_iterations, hist[t][k].rr), (k, t)
            assert s.scalar("FactoredCellsUsed") == members[k].scalar("FactoredCellsUsed") == 1
            for n in ("Velocity", "Position"):
                assert np.array_equal(s.read(n).view(np.int64), members[k].read(n).view(np.int64)), (k, n)
        members[k].close()
