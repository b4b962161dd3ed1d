"""More cells than one launch has workgroups for (GPU).

Two drops at opposite corners of the domain span 17.6 million level-0 cells in 3D (43 GB of
level matrices) and 68 million in 2D (its level 1 has 17.0 million).  Every level's matrix
is the sum of the finer one's blocks, so the entries of the coarsest add up to 1^T A 1, with
the product A 1 from the particles (bound 1e-12 of the entries' magnitudes, as in
test_gpu_level0.py).

The cell-staged second pass runs a workgroup of 512 threads per cell of the bounding box.  A
block of fluid and one drop far from it make that more than a launch holds, alone or as
two members of a batch: the chunk kernel takes over, with the same bits.
"""
import numpy as np
import pytest
import torch

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Batch, Scene
from test_gpu_coarse import L0
from test_gpu_faccells import assembled, two_drops

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


def block_and_drop(block, n):
    """block^3 particles in one corner of a domain of n cells per axis, 27 in the other."""
    side = 3.6 * n
    fluid = np.concatenate([scenes.lattice([2.0] * 3, [2.0 + block] * 3, L0, 3),
                            scenes.lattice([side - 5.0] * 3, [side - 2.0] * 3, L0, 3)])
    walls = scenes.lattice([0, 0, 0], [4, 4, 2], L0, 3)
    g = scenes.assemble(fluid, walls, 0.0, L0, [0.0] * 3, [side * L0] * 3, 5, 3)
    p = scenes.base_params(3, 0.1, (0.0, 0.0, -9.8), 5.0e-4, 4)
    p.operator_form = abi.OPERATOR_FACTORED
    p.multigrid = 0
    p.cr_tolerance = 1e-4
    p.end_time = 1.0e9
    return p, g


def test_product_of_many_cells():
    p, g = block_and_drop(162, 199)
    print("[manycells] np=%d" % g.np, flush=True)
    out = []
    for cells in (0, 1):
        s, y = assembled(p, g, cells)
        with s:
            assert s.scalar("FactoredCellsUsed") == 0
        out.append(y)
    assert np.array_equal(*out)


def test_batch_of_many_cells():
    p, g = block_and_drop(129, 158)
    print("[manycells] 2 members of np=%d" % g.np, flush=True)
    with Scene(p, g) as s:
        st = s.step(1)
        assert s.scalar("FactoredCellsUsed") == 1
        v = s.read("Velocity").view(np.int64)
    members = [Scene(p, g) for _ in range(2)]
    with Batch() as b:
        for m in members:
            b.add(m)
        for m, t in zip(members, b.step()):
            assert (t.cr_iterations, t.rr) == (st.cr_iterations, st.rr)
            assert np.array_equal(m.read("Velocity").view(np.int64), v)
    for m in members:
        m.close()


def test_batch_level0_of_90_million_cells():
    """The batch's P2G takes 8 lanes for each of 270 million level-0 rows."""
    if torch.cuda.mem_get_info()[0] < 160 << 30:
        pytest.skip("needs 160 GB of device memory")
    p, g = two_drops_2d(9230)
    p.operator_form = abi.OPERATOR_FACTORED
    p.cr_tolerance = 1e-4
    p.end_time = 1.0e9
    print("[manycells] np=%d" % g.np, flush=True)
    out = []
    for batch in (False, True):
        with Scene(p, g) as s:
            if batch:
                with Batch() as b:
                    b.add(s)
                    st = b.step()[0]
            else:
                st = s.step(1)
            out.append((st.cr_iterations, st.rr, s.read("Velocity").tobytes()))
    assert out[0] == out[1]
