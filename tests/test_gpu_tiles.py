"""Operator tiles picked from the grid (walsh_tile_rule in
chfem_amd/csrc/walsh.hip): whole solves on the grids where the pick changes
(one layer per block, partial rows, columns and layers, a single layer,
several rounds of blocks), against the oracle."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
@pytest.mark.parametrize("shape", [(3, 2, 4), (1, 9, 8), (24, 24, 24), (10, 65, 50), (37, 41, 56), (70, 8, 130)],
                         ids=lambda s: "x".join(map(str, s)))
def test_rule_tile_solves(shape, which, precision):
    """FP64 stops at 1e-9 of the initial residual: C agrees to 1e-7 (its error
    is the residual's times the condition of these two-phase problems, under
    100).  Mixed precision meets the same FP64 stop rule."""
    rng = np.random.default_rng(sum(shape))
    img = np.where(rng.random(shape) < 0.4, 255, 0).astype(np.uint8)
    img[0, 0, 0] = 0
    img[-1, -1, -1] = 255
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 10.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 10.0])
    s = H.GpuSolver(m, precision=precision, tol=1e-9)
    try:
        x, ok, st = s.solve(m.rhs(1))
        tile = np.zeros(3, dtype=np.int32)
        assert s.L.cudapcgGetOperatorTile(precision, s.ptr(tile)) == 1
        xr, okr, itr, _ = m.solve(1, tol=1e-9)
        assert ok and okr
        assert tile[2] in (1, 2, 4, 8, 16, 32)
        if m.N <= 24 ** 3:  # few blocks: at most 2 layers each
            assert tile[2] <= 2
        assert rel(m.update_c(1, x), m.update_c(1, xr)) < 1e-7
        if precision == 0:
            assert abs(int(st.iterations) - itr) <= 2
    finally:
        s.close()
