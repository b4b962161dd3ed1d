"""The bitonic network at the edges of its block sizes (GPU).

Keys are padded to a power of two; blocks of up to 8192 keys are sorted in the registers of
one workgroup (eight per thread), wider passes go through memory.  The pools below give 128
to 65,536 keys: less than a wavefront's share, one wavefront, less than a block, one block,
and several.  Particle order, with its ties, and fields are the oracle's bit for bit over
steps that move particles between cells.
"""
import numpy as np
import pytest

import pyoracle
from mphimplicit_amd import scenes
from mphimplicit_amd.scene import Scene
from test_gpu_crfold import L0

pytestmark = pytest.mark.gpu


def pool(nx, ny):
    fluid = scenes.lattice([0] * 3, [nx, ny, 0], L0, 2)
    walls = scenes.box_walls([0] * 2, [nx, ny + 2], 1, L0, 2, open_top=True)
    lo = [-9 * L0] * 2 + [-0.05]
    hi = [(nx + 9.5) * L0, (ny + 11.5) * L0, 0.05]
    g = scenes.assemble(fluid, walls, 0.0, L0, lo, hi, 5, 2)
    u = scenes.splitmix64_uniform(3, 2 * g.np).reshape(-1, 2)
    fl = np.asarray(g.type) < 2
    g.vel[fl, :2] = 2.0 * u[fl] - 1.0
    p = scenes.base_params(2, 0.1, (0.0, -9.8, 0.0), 5.0e-4, 4)
    p.cr_tolerance = 1e-6
    return p, g


@pytest.mark.parametrize("n", [(9, 7), (20, 18), (35, 25), (44, 40), (60, 58), (80, 70), (110, 90), (230, 220)], ids=lambda n: "%dx%d" % n)
def test_order_bitwise(n):
    p, g = pool(*n)
    print("[sort] %dx%d np=%d keys=%d" % (n + (g.np, 1 << int(g.np).bit_length())), flush=True)
    orc = pyoracle.OracleScene(p, g, pyoracle.DOT_TREE)
    with Scene(p, g) as s:
        for _ in range(2):
            s.step(1)
            orc.step(1)
        for name in ("ParticleIndex", "Position", "Velocity"):
            a, b = s.read(name), orc.read(name)
            assert np.array_equal(a.view(np.int64) if a.dtype == np.float64 else a,
                                  b.view(np.int64) if b.dtype == np.float64 else b), name
