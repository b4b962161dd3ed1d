"""The neighbour search's wavefront scan at its edges (GPU).

A wavefront scans the candidates of one particle, or of four consecutive ones in scenes
of 32768 particles and more, 64 candidates at a time.  The scenes below have particle
counts that leave a wavefront of four partly filled, cells of less than 64 and of more
than 128 candidates per range, windows that wrap around the periodic box, and particles
of several cells in one wavefront (walls, 2D).  The lists of both ways to build them
(count and fill; one scan into scratch) are whole numbers and equal the oracle's.
"""
import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene
from parity import compare_phase
from test_gpu_coarse import L0, pool

pytestmark = pytest.mark.gpu


def wide(n):
    p, g = pool(n)
    p.radius_ratio_a = p.radius_ratio_v = 4.6
    return p, g


def periodic(n):
    """Fluid that fills a periodic box: every border cell's window wraps."""
    dim = len(n)
    fluid = scenes.lattice([0] * 3, list(n) + [0] * (3 - dim), L0, dim)
    lo = [-0.5 * L0] * dim + [-0.05] * (3 - dim)
    hi = [(m - 0.5) * L0 for m in n] + [0.05] * (3 - dim)
    g = scenes.assemble(fluid, fluid[:0], 0.0, L0, lo, hi, 77, dim)
    p = scenes.base_params(dim, 0.1, (0.0, 0.0, 0.0), 5.0e-4, 4)
    return p, g


CASES = {
    "2d_small": (lambda: pool((9, 7)), None), "3d_wide": (lambda: wide((12, 11, 10)), None),
    "2d_periodic": (lambda: periodic((23, 38)), None), "3d_periodic": (lambda: periodic((12, 15, 19)), None),
    "2d_shared": (lambda: pool((251, 133)), True), "3d_shared": (lambda: pool((31, 24, 27)), True),
    "3d_shared_wide": (lambda: wide((27, 25, 29)), True), "3d_shared_periodic": (lambda: periodic((31, 33, 35)), True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_lists(name):
    make, shared = CASES[name]
    p, g = make()
    print("[neighbors] %s np=%d" % (name, g.np), flush=True)
    assert (g.np >= 32768) == bool(shared)
    rng = np.random.default_rng(3)
    with Scene(p, g) as s:
        orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
        x = s.read("Position").reshape(-1, 3).copy()
        x[:, :p.dim] += rng.uniform(-0.2, 0.2, (len(x), p.dim)) * L0
        for scan in range(2):
            for sc in (s, orc):
                if scan == 0:
                    sc.write("Position", x.reshape(-1))
                for ph in (abi.PHASE_CELLS, abi.PHASE_NEIGHBOR):
                    sc.run_phase(ph)
            bad = compare_phase(s, orc, abi.PHASE_CELLS) + compare_phase(s, orc, abi.PHASE_NEIGHBOR)
            assert not bad, "\n".join(bad)
            for ph in range(abi.PHASE_EXPLICIT, abi.PHASE_MULTIGRID + 1):  # the run starts
                s.run_phase(ph), orc.run_phase(ph)
            bad = compare_phase(s, orc, abi.PHASE_MULTIGRID)
            assert not bad, "\n".join(bad)
