"""The factored form's level-0 build over its workgroup sizes (GPU).

A level-0 row cell takes 64 threads in 2D, 512 in 3D and 256 in 3D levels of 4096 cells
and more.  The scenes put the cells on both sides of that line, with stencils of exactly
three cells and cells whose candidate lists are longer than the LDS list.  The level
matrices equal those summed from the assembled blocks within 1e-12 of the largest entry
(the bound of the factored tests).
"""
import numpy as np
import pytest

from mphimplicit_amd import abi
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu


def wide(n):  # P lists that reach far into the neighbouring cells
    p, g = pool(n)
    p.radius_ratio_a = p.radius_ratio_v = p.radius_ratio_p = 3.5
    return p, g


CASES = {"2d": lambda: pool((41, 61)), "2d_wide": lambda: wide((23, 19)), "3d_narrow": lambda: pool((11, 9, 10)),
         "3d": lambda: pool((17, 14, 15)), "3d_wide": lambda: wide((25, 23, 26)),
         "3d_4096_cells": lambda: pool((57, 56, 57))}


@pytest.mark.parametrize("name", list(CASES))
def test_level0(name):
    levels = []
    for form in (abi.OPERATOR_ASSEMBLED, abi.OPERATOR_FACTORED):
        p, g = CASES[name]()
        p.operator_form = form
        print("[level0] %s form %d np=%d" % (name, form, g.np), flush=True)
        with Scene(p, g) as s:
            for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIGRID + 1):
                s.run_phase(ph)
            if form == abi.OPERATOR_FACTORED:
                assert not s.scalar("AssembledBlocks")
            levels.append([s.read("MGCofA_L%d" % l) for l in range(int(s.scalar("MultiGridDepth")))])
    for a, f in zip(*levels):
        assert a.shape == f.shape and np.abs(a - f).max() <= 1e-12 * np.abs(a).max()
