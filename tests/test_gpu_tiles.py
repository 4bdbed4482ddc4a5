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


@pytest.mark.parametrize("which,precision,shape,tile", [
    ("elastic", 1, (71, 64, 85), (65, 15, 2)),
    ("elastic", 1, (113, 32, 29), (32, 16, 2)),
    ("thermal", 1, (67, 31, 50), (32, 16, 2)),
    ("thermal", 0, (41, 49, 89), (32, 16, 2)),
    ("elastic", 0, (41, 49, 89), (32, 16, 2)),
    ("thermal", 1, (38, 33, 48), (16, 16, 2)),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_rule_picks(which, precision, shape, tile, monkeypatch):
    """Grids on which the rule takes 65x15, 32x16 and, in FP32, 16x16 tiles: the
    pick, and the iterate after 20 steps against a 32x8x16 tile's.  Sums grouped otherwise and the
    layers of a block begun elsewhere change single roundings (6e-8 in FP32,
    1e-16 in FP64), which 20 steps multiply by less than 1000."""
    rng = np.random.default_rng(sum(shape))
    img = rng.choice(np.array([0, 255], np.uint8), size=shape)
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 5.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 5.0])
    monkeypatch.setenv("CHFEM_RELIABLE_DROP", "1e-30")
    got = []
    for env in (None, "32x8x16"):
        if env:
            monkeypatch.setenv("CHFEM_WALSH_TILE", env)
        s = H.GpuSolver(m, precision=precision, tol=1e-30, maxit=20)
        try:
            x, _, st = s.solve(m.rhs(1))
            t = np.zeros(3, dtype=np.int32)
            assert s.L.cudapcgGetOperatorTile(precision, s.ptr(t)) == 1
            assert tuple(t) == (tile if env is None else (32, 8, 16))
            assert int(st.iterations) == 20
            got.append(x)
        finally:
            s.close()
    scale = np.abs(got[1]).max()
    assert scale > 0 and np.abs(got[0] - got[1]).max() < (6e-5 if precision else 1e-10) * scale


@pytest.mark.parametrize("env", [None, "mfma"], ids=["default", "matrix-cores"])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
@pytest.mark.parametrize("shape", [(3, 2, 4), (9, 70, 40), (17, 33, 65)], ids=lambda s: "x".join(map(str, s)))
def test_element_strategy(shape, which, env, monkeypatch):
    """The element-by-element strategy on its default operator and on the
    matrix-core kernel: apply to 1e-12, solves to the FP64 stop rule, then a
    solve of another image set on the same solver (its node keys are
    rebuilt)."""
    if env:
        monkeypatch.setenv("CHFEM_EBE", env)
    rng = np.random.default_rng(sum(shape))
    props = [1.0, 0.3, 10.0, 0.2, 4.0, 0.25] if which == "elastic" else [1.0, 10.0, 3.5]
    images = [rng.choice(np.array([0, 100, 255], np.uint8), size=shape, p=[.5, .3, .2]) for _ in range(2)]
    ms = [H.model(H.ELASTIC if which == "elastic" else H.THERMAL, i, props, colors=(0, 100, 255)) for i in images]
    s = H.GpuSolver(ms[0], strategy=1, tol=1e-9)
    try:
        for m in ms:
            elem = m.elem.copy()
            assert s.L.cudapcgSetImage(s.ptr(elem)) == 1
            v = rng.standard_normal(m.ndof)
            assert rel(s.apply(v), m.apply(v, strategy=1)) < 1e-12
            x, ok, st = s.solve(m.rhs(0))
            xr, okr, itr, _ = m.solve(0, tol=1e-9, strategy=1)
            assert ok and okr and abs(int(st.iterations) - itr) <= 2
            assert rel(m.update_c(0, x), m.update_c(0, xr)) < 1e-7
    finally:
        s.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("solver", [0, 1, 2], ids=["cg", "minres", "cg3"])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
@pytest.mark.parametrize("shape", [(3, 2, 4), (9, 70, 40), (24, 24, 24)], ids=lambda s: "x".join(map(str, s)))
def test_density_solves(shape, which, solver, precision):
    """Scalar density field (densities down to 1 % of the largest) with every
    kind of loop, against the oracle's solve of the same scaled elements;
    residual 1e-9 and a condition of the field below 1000 give 1e-6 in C."""
    rng = np.random.default_rng(sum(shape) + solver)
    img = rng.choice(np.array([0, 255], np.uint8), size=shape)
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 1.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 2.0])
    d = rng.integers(0, 65536, size=m.N).astype(np.uint16)
    lo, hi = 0.01, 1.0
    m.set_element_scale(d.astype(np.float64) * (1.0 / 65535.0) * (hi - lo) + lo)
    s = H.GpuSolver(m, strategy=1, solver=solver, precision=precision, tol=1e-9)
    try:
        assert s.L.cudapcgSetParametricDensityField(s.ptr(d), lo, hi) == 1
        v = rng.standard_normal(m.ndof) if solver < 2 else None
        if v is not None:
            assert rel(s.apply(v), m.apply(v, strategy=1)) < 1e-12
        x, ok, st = s.solve(m.rhs(0))
        xr, okr, itr, _ = m.solve(0, tol=1e-9, strategy=1)
        assert ok and okr
        assert rel(m.update_c(0, x), m.update_c(0, xr)) < 1e-6
    finally:
        s.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("tile", ["32x8x5", "65x7x5"])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
def test_density_tiles(which, tile, precision, monkeypatch):
    """Both tile shapes of the density kernels with several layers per block,
    on a grid ragged in every direction (two tiles along the rows, a last
    chunk of one layer), densities independent from element to element: the
    operator in the precision of the loop, and a solve (tolerances as in
    test_density_solves; FP32 rounds sums over 8 elements)."""
    monkeypatch.setenv("CHFEM_WALSH_TILE", tile)
    rng = np.random.default_rng(70)
    img = rng.choice(np.array([0, 255], np.uint8), size=(11, 70, 23))
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 1.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 2.0])
    d = rng.integers(0, 65536, size=m.N).astype(np.uint16)
    lo, hi = 0.01, 1.0
    m.set_element_scale(d.astype(np.float64) * (1.0 / 65535.0) * (hi - lo) + lo)
    s = H.GpuSolver(m, strategy=1, precision=precision, tol=1e-9)
    try:
        assert s.L.cudapcgSetParametricDensityField(s.ptr(d), lo, hi) == 1
        v = rng.standard_normal(m.ndof).astype(np.float32)
        q = m.apply(v.astype(np.float64), strategy=1)
        if precision:
            assert np.abs(s.apply32(v) - q).max() < 1e-5 * np.abs(q).max()
        else:
            assert rel(s.apply(v.astype(np.float64)), q) < 1e-12
        x, ok, _ = s.solve(m.rhs(0))
        xr, okr, _, _ = m.solve(0, tol=1e-9, strategy=1)
        assert ok and okr
        assert rel(m.update_c(0, x), m.update_c(0, xr)) < 1e-6
    finally:
        s.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(2, 5, 9), (3, 33, 16), (7, 62, 30), (10, 100, 63), (16, 14, 31)],
                         ids=lambda s: "x".join(map(str, s)))
def test_stokes_layer_groups(shape, precision, monkeypatch):
    """On grids of few tiles two groups of work-items share a tile's layers,
    with the sums of one group: after 30 MINRES steps the solution has the same
    bits as with one group (tiles of 32 layers: one chunk either way)."""
    rng = np.random.default_rng(sum(shape))
    img = np.where(rng.random(shape) < 0.3, 255, 0).astype(np.uint8)
    img[:2, :2, :2] = 0  # the elements around one node: it is fully fluid
    m = H.model(H.FLUID, img, [0.0], colors=(0, 255))
    got = []
    for tile in (None, "32x8x32"):
        if tile:
            monkeypatch.setenv("CHFEM_WALSH_TILE", tile)
        s = H.GpuSolver(m, solver=1, precision=precision, tol=1e-30, maxit=30)
        try:
            x, _, st = s.solve(m.rhs(0))
            got.append((x, st.iterations))
        finally:
            s.close()
    assert got[0][1] == got[1][1] and np.abs(got[0][0]).max() > 0
    assert np.array_equal(got[0][0], got[1][0])


@pytest.mark.parametrize("nz", [17, 33])
def test_stokes_layer_groups_solve(nz):
    """Layer chunks shorter than a group: a whole solve against the oracle's."""
    rng = np.random.default_rng(nz)
    img = np.where(rng.random((nz, 20, 14)) < 0.1, 255, 0).astype(np.uint8)
    m = H.model(H.FLUID, img, [0.0], colors=(0, 255))
    s = H.GpuSolver(m, solver=1, tol=1e-9)
    try:
        x, ok, st = s.solve(m.rhs(2))
        xr, okr, _, _ = m.solve(2, solver=1, tol=1e-9)
        assert ok and okr
        assert rel(m.update_c(2, x), m.update_c(2, xr)) < 1e-6
    finally:
        s.close()


@pytest.mark.parametrize("maxit", [1, 2, 16, 17, 37])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
@pytest.mark.parametrize("shape", [(4, 5, 3), (24, 24, 24), (33, 64, 50), (48, 90, 61)],
                         ids=lambda s: "x".join(map(str, s)))
def test_chained_iterations(shape, which, maxit):
    """On small grids a CG iteration finishes the one before it, in chains that
    end with the queued batch (16) and with each ring flush.  The iterate after
    a given number of steps is the oracle's: rounding (1e-16 per step, times a
    condition below 1e4 and 37 steps) stays below 1e-8; the last shape runs on
    more blocks than are chained."""
    rng = np.random.default_rng(sum(shape))
    img = rng.choice(np.array([0, 255], np.uint8), size=shape)
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 5.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 5.0])
    if maxit > m.ndof // 2:
        # 60 unknowns are solved to rounding at step 17 (residual 5e-12); after
        # that the recurrences divide rounding by rounding, here and in the
        # oracle, and the iterate drifts along the constants
        pytest.skip("no more directions left to search")
    s = H.GpuSolver(m, tol=1e-30, maxit=maxit)
    try:
        x, _, st = s.solve(m.rhs(1))
        xr, _, itr, _ = m.solve(1, tol=1e-30, maxit=maxit)
        assert int(st.iterations) == itr == maxit
        assert np.abs(x - xr).max() < 1e-8 * np.abs(xr).max()
    finally:
        s.close()


@pytest.mark.parametrize("solver", [0, 1], ids=["cg", "minres"])
def test_block_count_of_the_launched_tile(solver, monkeypatch):
    """A fixed tile that FP64 runs as a smaller one (65x15 as 65x7: 3 tiles of
    each layer instead of 1): the layers per block keep the launched blocks
    within the reduction partials.  One layer per block would be 196608 blocks
    of 4 partials.  The iterate after 20 steps is the default tile's: sums of
    9e5 terms grouped otherwise differ by less than 1e-12, which 20 steps
    multiply by less than 1000."""
    rng = np.random.default_rng(3)
    m = H.model(H.THERMAL, rng.choice(np.array([0, 255], np.uint8), size=(65536, 1, 14)), [1.0, 5.0])
    got = []
    for tile in (None, "65x15x1"):
        if tile:
            monkeypatch.setenv("CHFEM_WALSH_TILE", tile)
        s = H.GpuSolver(m, solver=solver, tol=1e-30, maxit=20)
        try:
            x, _, st = s.solve(m.rhs(0))
            got.append(x)
            assert int(st.iterations) == 20
        finally:
            s.close()
    assert np.abs(got[0]).max() > 0
    assert np.abs(got[1] - got[0]).max() < 1e-9 * np.abs(got[0]).max()


@pytest.mark.parametrize("solver", [0, 1], ids=["cg", "minres"])
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("which", ["elastic", "thermal"])
def test_timed_tiles(which, precision, solver, monkeypatch):
    """CHFEM_WALSH_TILE=auto: the timed choice of tile and loop form, and the
    solve that follows (residual 1e-9, condition below 100: 1e-7 in C).  The
    rule's tile is a candidate: on this grid tiles of 16 layers take over
    twice as long per FP64 elastic iteration."""
    monkeypatch.setenv("CHFEM_WALSH_TILE", "auto")
    rng = np.random.default_rng(24)
    img = rng.choice(np.array([0, 255], np.uint8), size=(24, 24, 24))
    m = H.model(H.ELASTIC, img, [1.0, 0.3, 5.0, 0.2]) if which == "elastic" else H.model(H.THERMAL, img, [1.0, 5.0])
    s = H.GpuSolver(m, solver=solver, precision=precision, tol=1e-9)
    try:
        x, ok, _ = s.solve(m.rhs(0))
        xr, okr, _, _ = m.solve(0, tol=1e-9)
        t = np.zeros(3, dtype=np.int32)
        assert s.L.cudapcgGetOperatorTile(precision, s.ptr(t)) == 1
        assert ok and okr and rel(m.update_c(0, x), m.update_c(0, xr)) < 1e-7
        assert s.L.cudapcgGetLoopForm(precision) in (1, 2)
        if which == "elastic" and precision == 0 and solver == 0:
            assert t[2] <= 4, t
    finally:
        s.close()
