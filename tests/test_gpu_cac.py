"""C Lambda C^T by hashed lists at the edges of its tables (GPU).

A particle's P-neighbour list goes into 32 buckets of four entries; lists of up to 64
entries take that way, longer ones are merged.  The radius ratios below give lists from
a handful to just below and above 64, with buckets that run over, and the fluid counts a
last slice of one row, of a part and a full one.  The blocks are bit-identical to the
oracle's.
"""
import pytest

import pyoracle
from mphimplicit_amd import abi
from mphimplicit_amd.scene import Scene
from parity import compare_phase
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu

CASES = [((13, 5), 1.2, 9), ((8, 8), 1.7, 13), ((21, 15), 3.3, 37), ((21, 15), 4.2, 64), ((21, 15), 4.5, 80),
         ((16, 8, 5), 1.7, 27), ((7, 8, 8), 2.3, 64), ((7, 8, 8), 2.6, 99)]


@pytest.mark.parametrize("n,ratio,most", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_blocks(n, ratio, most):
    p, g = pool(n)
    p.radius_ratio_p = ratio
    h = 2.0 * ratio * g.spacing
    dim = len(n)
    for d in range(dim):  # at least four cells of the largest radius per axis
        grow = max(0.0, 4.2 * h - (g.domain_max[d] - g.domain_min[d]))
        g.domain_max[d] += grow
    with Scene(p, g) as s:
        orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
        for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
            s.run_phase(ph), orc.run_phase(ph)
        longest = int(s.read("NeighborCountP")[:s.read("CsrPtrA").size // 3].max())
        print("[cac] %s ratio %g: lists of up to %d" % (n, ratio, longest), flush=True)
        assert (longest <= 64) == (most <= 64)
        bad = compare_phase(s, orc, abi.PHASE_MATRIX_A) + compare_phase(s, orc, abi.PHASE_MULTIPLY_C)
        assert not bad, "\n".join(bad)
