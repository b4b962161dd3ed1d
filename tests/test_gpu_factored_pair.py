"""The factored product's recomputed scalars at their edges (GPU).

The FP64 passes recompute alpha and beta from a pair's distance where one viscosity fills
the scene, and read the stored alpha where fluids of several viscosities meet; the
cell-staged pass has launch shapes for 2D, 3D and domains of few, wide cells, and rows
longer than one block of 64 places.  Each scene's product must agree with the product of
the assembled matrix of the same particles (bound 1e-11 of max(|A| |x|) as in
test_gpu_factored.py; |A| |x| from the assembled blocks' product with |x|, which bounds it
from below), and the chunk kernel must give the same bits as the cells.  Two particles at
the same place and a pair exactly one radius apart contribute nothing.
"""
import numpy as np
import pytest

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu


def two_fluids(n):
    p, g = pool(n)
    g.type[(g.type == 0) & (g.pos[:, 0] < 0.5 * n[0] * g.spacing)] = 1
    p.shear_viscosity[1] = 0.7
    p.density[1] = 800.0
    return p, g


def coincident(n):
    p, g = pool(n)
    g.pos[1] = g.pos[0]                               # the same place
    g.pos[3] = g.pos[2] + [1.7 * g.spacing, 0.0, 0.0]  # one RadiusP apart, up to rounding
    return p, g


def wide(n):
    p, g = pool(n)
    p.radius_ratio_a = p.radius_ratio_v = 4.6  # rows of several blocks, wide cells
    return p, g


MAKE = {
    "2d": lambda: pool((23, 17)), "2d_one_row": lambda: pool((2, 40)), "3d": lambda: pool((13, 11, 9)),
    "3d_small": lambda: pool((6, 5, 4)), "two_fluids_2d": lambda: two_fluids((21, 18)),
    "two_fluids_3d": lambda: two_fluids((11, 12, 10)), "coincident_2d": lambda: coincident((12, 9)),
    "coincident_3d": lambda: coincident((9, 8, 7)), "wide_3d": lambda: wide((12, 11, 10)),
}


@pytest.mark.parametrize("name", list(MAKE))
def test_recomputed_scalars(name):
    print("[pair] %s" % name, flush=True)
    out = {}
    for form, cells in ((abi.OPERATOR_ASSEMBLED, 1), (abi.OPERATOR_FACTORED, 1), (abi.OPERATOR_FACTORED, 0)):
        p, g = MAKE[name]()
        p.operator_form = form
        with Scene(p, g) as s:
            s.set_option("FactoredCells", cells)
            for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
                s.run_phase(ph)
            x = np.random.default_rng(3).standard_normal(3 * int(s.scalar("FluidCount")))
            out[form, cells] = s.apply_matrix(x)
            if form == abi.OPERATOR_ASSEMBLED:
                scale = np.abs(s.apply_matrix(np.abs(x))).max()
    a, f, c = out.values()
    assert np.isfinite(f).all()
    assert np.array_equal(f.view(np.int64), c.view(np.int64))
    err = np.abs(f - a).max() / scale
    print("[pair] %s: max|yf-ya| / max|A||x| <= %.3e" % (name, err), flush=True)
    assert err <= 1e-11
