"""Tile shapes of the batched operators (64 x 7 with the halo wavefront, 32 x 8
and 64 x 8): batches whose sizes make the rule choose each of them, with whole
tiles, remainders of one node and chunks of one layer, in every step form,
against the oracle."""
import numpy as np
import pytest

from chfem_amd import batch, synthetic
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["2", "1"], ids=["single-kernel", "dir-fused"])
@pytest.mark.parametrize("prop", ["conductivity", "elasticity"])
@pytest.mark.parametrize("shapes", [
    [(9, 64, 12), (5, 128, 7)],   # 64 rows owned per tile
    [(9, 63, 14), (5, 126, 8)],   # 63 rows
    [(9, 31, 15), (33, 33, 7)],   # 31 rows
    [(2, 2, 2), (3, 65, 3)],
], ids=lambda s: "x".join(map(str, s[0])))
def test_batch_tile_shapes(shapes, prop, form, monkeypatch):
    """A CG residual of 1e-8 leaves the effective matrix within 1e-6 of the
    oracle's (the error is quadratic in the residual, times the contrast)."""
    monkeypatch.setenv("CHFEM_BATCH_FORM", form)
    el = prop == "elasticity"
    mats = {0: (1.0, 0.3), 255: (6.0, 0.2)} if el else {0: 1.0, 255: 6.0}
    rng = np.random.default_rng(12)
    samples = [(255 * rng.integers(0, 2, s).astype(np.uint8), mats) for s in shapes]
    Cs, info = batch.batch_homogenize(samples, prop, tol=1e-8)
    assert info["converged"], info
    for (img, _), C in zip(samples, Cs):
        R, _ = H.model(H.ELASTIC if el else H.THERMAL, img,
                       [*mats[0], *mats[255]] if el else [mats[0], mats[255]]).homogenize(tol=1e-10)
        R = np.asarray(R)
        assert np.abs(np.asarray(C) - R).max() < 1e-6 * np.abs(R).max()
