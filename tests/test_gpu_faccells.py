"""When the factored product's second pass runs staged per cell (GPU).

FactoredCellsUsed tells which kernel the last assembled matrix has its FP64 second pass
run as; either gives the same bits.  The cells take part only once the rows' staged
places have been built, so switching the option on afterwards leaves the chunk kernel in
place until the next step.  A cell whose visited cells hold more records than the staging
does has its rows gathered inside the cell kernel.
"""
import numpy as np
import pytest

from mphimplicit_amd import abi, scenes
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import L0, pool

pytestmark = pytest.mark.gpu


def assembled(p, g, cells):
    """The scene with its matrix assembled, and a product."""
    p.operator_form = abi.OPERATOR_FACTORED
    s = Scene(p, g)
    s.set_option("FactoredCells", cells)
    for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
        s.run_phase(ph)
    return s, product(s)


def product(s):
    x = np.random.default_rng(3).standard_normal(3 * int(s.scalar("FluidCount")))
    return s.apply_matrix(x).view(np.int64)


@pytest.mark.parametrize("n", [(23, 17), (13, 11, 9)], ids=lambda n: "x".join(map(str, n)))
def test_cells_used(n):
    print("[faccells] %s" % (n,), flush=True)
    p, g = pool(n)
    p.operator_form = abi.OPERATOR_FACTORED
    p.end_time = 1.0e9
    with Scene(p, g) as s:
        assert s.scalar("FactoredCellsUsed") == 0  # no matrix yet
        s.step(1)
        assert s.scalar("FactoredCellsUsed") == 1
        y = product(s)
        s.set_option("FactoredCells", 0)
        assert s.scalar("FactoredCellsUsed") == 0
        assert np.array_equal(product(s), y)
        s.step(1)
        s.set_option("FactoredCells", 1)  # this matrix has no staged places
        assert s.scalar("FactoredCellsUsed") == 0
        y = product(s)
        s.step(1)
        assert s.scalar("FactoredCellsUsed") == 1
    p.operator_form = abi.OPERATOR_ASSEMBLED
    with Scene(p, g) as s:
        s.step(1)
        assert s.scalar("FactoredCellsUsed") == 0


def wide(n, radius):
    """A pool with a larger MaxRadius, in spacings, in a domain to match."""
    p, g = pool(n)
    p.radius_ratio_a = p.radius_ratio_v = radius
    for d in range(len(n)):  # cells a little wider than the radius
        w = g.domain_max[d] - g.domain_min[d]
        g.domain_max[d] = g.domain_min[d] + np.ceil(w / (radius * L0)) * (radius + 0.1) * L0
    return p, g


# The launch shape follows the particles that a lattice has in the visited cells: up to 256
# in 2D, up to 1456, and beyond.  9 cells of 5.5 spacings hold 273 and more, of 8 spacings
# 576; of 18 spacings 2916, and 27 of 5.5 hold 4492, more than the largest staging (2816).
# A pool 3 deep has cells of 3.86 spacings in z: 11 x 11 x 12 of a lattice
@pytest.mark.parametrize("n,radius", [((30, 31), 5.0), ((60, 50), 5.5), ((60, 50), 8.0), ((70, 60), 13.0),
                                      ((70, 60), 18.0), ((20, 19, 18), 5.5), ((38, 32, 3), 3.5)], ids=str)
def test_large_radii(n, radius):
    print("[faccells] %s radius %g" % (n, radius), flush=True)
    out = []
    for cells in (0, 1):
        s, y = assembled(*(wide(n, radius) if radius > 3.5 else pool(n)), cells)
        with s:
            assert s.scalar("FactoredCellsUsed") == cells
        out.append(y)
    assert np.array_equal(*out)


def two_drops(n):
    """Two drops at opposite corners of a domain of n cells per axis."""
    side = 3.6 * n
    at = [2.0, side - 8.0]
    fluid = np.concatenate([scenes.lattice([a] * 3, [a + 6] * 3, L0, 3) for a in at])
    walls = scenes.lattice([0, 0, 0], [4, 4, 2], L0, 3)
    g = scenes.assemble(fluid, walls, 0.0, L0, [0.0] * 3, [side * L0] * 3, 5, 3)
    p = scenes.base_params(3, 0.1, (0.0, 0.0, -9.8), 5.0e-4, 4)
    p.multigrid = 0
    return p, g


def clump(n):
    """n^3 particles two spacings apart, and 384 in one place."""
    grid = scenes.lattice([0] * 3, [n] * 3, 2 * L0, 3)
    u = np.stack(np.meshgrid(np.arange(8), np.arange(8), np.arange(6), indexing="ij"), axis=-1).reshape(-1, 3)
    fluid = np.concatenate([grid, (n + 0.13 + 0.25 * u) * L0])
    walls = scenes.lattice([0, 0, -4], [4, 4, -2], L0, 3)
    g = scenes.assemble(fluid, walls, 0.0, L0, [-0.09] * 3, [(2 * n + 9.5) * L0] * 3, 5, 3, jitter=0)
    return scenes.base_params(3, 0.1, (0.0, 0.0, -9.8), 5.0e-4, 4), g


@pytest.mark.parametrize("make", [lambda: two_drops(100), lambda: clump(28)], ids=["two_drops", "clump"])
def test_places_not_worth_their_memory(make):
    """A million cells for 432 particles, one long row among 22 thousand: the chunk kernel,
    and no buffers for the cells."""
    p, g = make()
    print("[faccells] np=%d" % g.np, flush=True)
    out = []
    for cells in (0, 1):
        s, y = assembled(p, g, cells)
        with s:
            assert s.scalar("FactoredCellsUsed") == 0
            out.append((y, s.device_bytes()))
    assert np.array_equal(out[0][0], out[1][0])
    assert np.isfinite(out[0][0].view(np.float64)).all()
    assert out[0][1] == out[1][1]
