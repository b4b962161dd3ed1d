"""The product of small scenes, split over the components of a row (GPU).

Scenes of up to 400 slices of 64 rows take it, larger ones the kernel with a row per
lane.  Rows are summed in the order of the CSR in both, so the products equal a sum in
that order bit for bit: in FP64 of the stored values, in FP32 of the values rounded to
float.  The scenes put the last row at the edges of a slice and the row lengths at those
of a round of 8 blocks, and lie on both sides of the rule.
"""
import numpy as np
import pytest

from mphimplicit_amd import abi
from mphimplicit_amd.scene import Scene
from test_gpu_coarse import pool

pytestmark = pytest.mark.gpu

BOXES = [(3, 2), (9, 7), (8, 8), (13, 5), (5, 5, 5), (4, 4, 4), (16, 8, 5), (159, 161), (161, 160)]


def in_order(s, x, f32):
    ptr, ind, cof = s.read("CsrPtrA"), s.read("CsrIndA"), s.read("CsrCofA")
    if f32:
        cof = cof.astype(np.float32).astype(np.float64)
    n = np.diff(ptr)
    y = np.zeros(len(n))
    for k in range(int(n.max())):
        at = np.where(k < n, ptr[:-1] + k, 0)
        y = np.where(k < n, y + cof[at] * x[ind[at]], y)
    return y


@pytest.mark.parametrize("precision", [abi.PRECISION_FP64, abi.PRECISION_MIXED], ids=["fp64", "fp32"])
@pytest.mark.parametrize("n", BOXES, ids=lambda n: "x".join(map(str, n)))
def test_product_in_order(n, precision):
    p, g = pool(n)
    p.precision = precision
    print("[split] %s np=%d" % (n, g.np), flush=True)
    with Scene(p, g) as s:
        for ph in range(abi.PHASE_KINEMATICS, abi.PHASE_MULTIPLY_C + 1):
            s.run_phase(ph)
        x = np.random.default_rng(5).standard_normal(3 * int(np.prod(n)))
        y = s.apply_matrix(x, precision)
        assert y.tobytes() == in_order(s, x, precision == abi.PRECISION_MIXED).tobytes()
