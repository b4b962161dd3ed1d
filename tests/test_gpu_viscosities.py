"""Fluids of several viscosities in the factored form (GPU).

Matrix A leaves two flags for the product: a pair interacts through the periodic boundary;
a fluid pair's viscosity is not the scene's one.  Nearly every wavefront finds the second
in a scene of two fluids.  Raising it must not cost the pass its time: entry by entry it
took five times that of one fluid, the bound here is two.  Both flags together are checked
by the product against that of the assembled matrix (1e-11 of max |A| |x|, as in
test_gpu_factored.py).
"""
import numpy as np
import pytest

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu


def two_fluids(p, g):
    f = g.type == 0
    g.type[f & (g.pos[:, 0] < np.median(g.pos[f, 0]))] = 1
    p.shear_viscosity[1] = 0.7
    p.density[1] = 800.0
    p.end_time = 1.0e9
    return p, g


def test_time_of_matrix_a():
    ms = []
    for fluids in (1, 2):
        p, g = pool((40, 40, 40))
        if fluids == 2:
            two_fluids(p, g)
        p.operator_form = abi.OPERATOR_FACTORED
        p.end_time = 1.0e9
        print("[viscosities] %d, np=%d" % (fluids, g.np), flush=True)
        with Scene(p, g) as s:
            s.step(1)
            s.set_timing(1)
            ms.append(min(s.step(1).ms_phase[abi.PHASE_MATRIX_A] for _ in range(5)))
    print("[viscosities] matrix A %.3f ms with one, %.3f ms with two" % tuple(ms), flush=True)
    assert ms[1] <= 2.0 * ms[0]


def test_both_flags():
    out = {}
    for form, cells in ((abi.OPERATOR_ASSEMBLED, 1), (abi.OPERATOR_FACTORED, 1), (abi.OPERATOR_FACTORED, 0)):
        p, g = two_fluids(*scenes.periodic_3d())
        p.operator_form = form
        print("[viscosities] periodic, form %d, np=%d" % (form, g.np), flush=True)
        with Scene(p, g) as s:
            s.set_option("FactoredCells", cells)
            for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
                s.run_phase(ph)
            x = np.random.default_rng(3).standard_normal(3 * int(s.scalar("FluidCount")))
            out[form, cells] = s.apply_matrix(x)
            if form == abi.OPERATOR_ASSEMBLED:
                scale = np.abs(s.apply_matrix(np.abs(x))).max()
    a, f, c = out.values()
    assert np.array_equal(f.view(np.int64), c.view(np.int64))
    assert np.abs(f - a).max() <= 1e-11 * scale
