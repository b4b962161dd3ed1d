"""Multigrid levels of more cells than one launch has workgroups for (GPU).

Two drops at opposite corners of the domain span 17.6 million level-0 cells in 3D (43 GB of
level matrices) and 68 million in 2D (its level 1 has 17.0 million).  Every level's matrix
is the sum of the finer one's blocks, so the entries of the coarsest add up to 1^T A 1, with
the product A 1 from the particles (bound 1e-12 of the entries' magnitudes, as in
test_gpu_level0.py).
"""
import numpy as np
import pytest
import torch

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import L0
from test_gpu_faccells import two_drops

pytestmark = pytest.mark.gpu


def two_drops_2d(n):
    side = 3.6 * n
    fluid = np.concatenate([scenes.lattice([a, a, 0], [a + 6, a + 6, 0], L0, 2) for a in (2.0, side - 8.0)])
    walls = scenes.lattice([0, 0, 0], [4, 2, 0], L0, 2)
    g = scenes.assemble(fluid, walls, 0.0, L0, [0.0, 0.0, -0.05], [side * L0, side * L0, 0.05], 5, 2)
    return scenes.base_params(2, 0.1, (0.0, -9.8, 0.0), 5.0e-4, 4), g


@pytest.mark.parametrize("make,gb", [(lambda: two_drops(254), 64), (lambda: two_drops_2d(8020), 128)],
                         ids=["3d", "2d"])
@pytest.mark.parametrize("form", [abi.OPERATOR_FACTORED, abi.OPERATOR_ASSEMBLED])
def test_levels_of_many_cells(make, gb, form):
    if torch.cuda.mem_get_info()[0] < gb << 30:
        pytest.skip("needs %d GB of device memory" % gb)
    p, g = make()
    p.operator_form = form
    p.multigrid = 1
    with Scene(p, g) as s:
        print("[manycells] form %d, %d cells in the domain" % (form, s.scalar("TotalCellCount")), flush=True)
        for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIGRID + 1):
            s.run_phase(ph)
        a = s.read("MGCofA_L%d" % (int(s.scalar("MultiGridDepth")) - 1))
        total = float(s.apply_matrix(np.ones(3 * int(s.scalar("FluidCount")))).sum())
    entries, most = float(a.sum()), float(np.abs(a).sum())
    assert abs(entries - total) <= 1e-12 * most, (entries, total)
