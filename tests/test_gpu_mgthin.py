"""Thin fluid layers in the transfers that are part of a sweep (GPU).

A 3D level one cell deep in z has the stencil 3x3x1 of a 2D level, but its layer may lie
at an odd cell, where it is the second child of its coarse cell.  The layers below lie at
even and odd cells, wide enough (23 x 23 cells and more) that the level's residual and its
restriction are one launch; the last one is two cells deep, so that level 1 is thin.  The
assembled form is bit-identical to the oracle and to the launches of their own for the
transfers (LaneRowsMax 0) and to the same scene in a batch, the factored one to the
latter two.
"""
import math

import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Batch, Scene

pytestmark = pytest.mark.gpu

L0 = 0.01
CELL = 3.6  # spacings: the height of a cell (13 cells of 3.6 spacings for a radius of 3.5)


def layer(nx, nz, cell):
    """nx x nx x nz fluid particles from cell `cell` in z upwards on two layers of walls."""
    z0 = math.ceil(CELL * cell)
    fluid = scenes.lattice([8, 8, z0], [8 + nx, 8 + nx, z0 + nz], L0, 3)
    walls = scenes.lattice([8, 8, z0 - 2], [8 + nx, 8 + nx, z0], L0, 3)
    width = CELL * math.ceil((nx + 16) / CELL) * L0
    g = scenes.assemble(fluid, walls, 0.0, L0, [0.0] * 3, [width, width, 13 * CELL * L0], 31, 3)
    p = scenes.base_params(3, 0.1, (0.0, 0.0, -9.8), 5.0e-4, 4)
    p.cr_tolerance = 1e-12
    p.end_time = 1.0e9
    return p, g


def solve(p, g, rows=None, batch=False):
    with Scene(p, g) as s:
        if rows is not None:
            s.set_option("LaneRowsMax", rows)
        if batch:
            with Batch() as b:
                b.add(s)
                st = b.step()[0]
        else:
            st = s.step(1)
        return st.cr_iterations, st.rr, s.read("Velocity").view(np.int64)


# (particles across, deep, first cell, compared with the oracle)
LAYERS = [(94, 2, 3, True), (94, 2, 4, True), (94, 3, 1, True), (186, 6, 2, False)]


@pytest.mark.parametrize("nx,nz,cell,oracle", LAYERS, ids=lambda v: str(v))
def test_thin_layer(nx, nz, cell, oracle):
    for form in (abi.OPERATOR_ASSEMBLED, abi.OPERATOR_FACTORED):
        p, g = layer(nx, nz, cell)
        p.operator_form = form
        print("[mgthin] %d x %d x %d at cell %d, form %d, np=%d" % (nx, nx, nz, cell, form, g.np), flush=True)
        it, rr, v = solve(p, g)
        for other in (solve(p, g, rows=0), solve(p, g, batch=True)):
            assert (it, rr) == other[:2]
            assert np.array_equal(v, other[2])
        if oracle and form == abi.OPERATOR_ASSEMBLED:
            orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
            b = orc.step(1)
            assert (it, rr) == (b.cr_iterations, b.rr)
            assert np.array_equal(v, orc.read("Velocity").view(np.int64))
