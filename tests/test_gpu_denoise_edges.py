"""The denoise filter at the image's edges (needs an MI355X): taps outside the image weigh nothing whatever the albedo is.
A constant image stays constant, radiance and albedo of any size.  Tolerance: 25 products and sums in float32 per level
and a product and a quotient with the albedo: 5 * 26 + 2 roundings of 6e-8, below 1e-5."""
import numpy as np
import pytest

from vviewer_amd import RendererPathTracing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("albedo", [0.5, 1e15, 3e30])
@pytest.mark.parametrize("surface", [True, False])
def test_constant_image(albedo, surface):
    h, w = 37, 50
    rad = np.full((h, w, 4), albedo * 1.5, np.float32)
    alb = np.full((h, w, 4), albedo, np.float32)
    nrm = np.full((h, w, 4), 0.5, np.float32)
    if surface:
        nrm[..., 2] = 1.0
    r = RendererPathTracing()
    out = r.denoise(rad, alb, nrm)
    r.close()
    assert np.max(np.abs(out[..., :3] / rad[..., :3] - 1.0)) < 1e-5
