"""The denoise filter at sizes where its tiling can go wrong (needs an MI355X): one pixel, images smaller than a tap
spacing or a tile, exact tiles, one past a tile, and strips, against a float64 restatement of the filter with whole-
image shifts.  Tolerance: five levels of 25 products and sums in float32 over weights from exp() (a few ulp at
arguments up to about 100, so up to 1e-5 relative in small weights) stay below 1e-4 of a pixel's value."""
import numpy as np
import pytest

from vviewer_amd import RendererPathTracing

pytestmark = pytest.mark.gpu

H5 = (1 / 16, 1 / 4, 3 / 8, 1 / 4, 1 / 16)


def _ref(rad, alb, nrm):
    H, W = rad.shape[:2]
    alb3 = alb[..., :3]
    a = np.where(alb3 > np.float64(np.float32(1e-3)), alb3, 1.0)
    c = rad[..., :3] / a
    n = nrm[..., :3] * 2.0 - 1.0
    l2 = (n * n).sum(-1)
    surf = l2 > 0.25
    n = n / np.sqrt(np.where(surf, l2, 1.0))[..., None]
    sc = 0.5
    for lev in range(5):
        step = 1 << lev
        t = np.log1p(np.maximum(c, 0.0))
        acc, ws = np.zeros_like(c), np.zeros((H, W))
        for j in range(5):
            for i in range(5):
                dy, dx = (j - 2) * step, (i - 2) * step
                y0, y1, x0, x1 = max(0, -dy), min(H, H - dy), max(0, -dx), min(W, W - dx)
                if y0 >= y1 or x0 >= x1:
                    continue
                p = (slice(y0, y1), slice(x0, x1))
                q = (slice(y0 + dy, y1 + dy), slice(x0 + dx, x1 + dx))
                wn = np.where(surf[p] & surf[q], np.maximum((n[p] * n[q]).sum(-1), 0.0) ** 64,
                              (surf[p] == surf[q]).astype(np.float64))
                w = H5[i] * H5[j] * wn * np.exp(-((t[q] - t[p]) ** 2).sum(-1) / sc ** 2
                                                - ((alb3[q] - alb3[p]) ** 2).sum(-1) / 0.02 ** 2)
                acc[p] += w[..., None] * c[q]
                ws[p] += w
        c = acc / ws[..., None]
        sc *= 0.5
    return c * a


@pytest.fixture(scope="module")
def r():
    rr = RendererPathTracing()
    yield rr
    rr.close()


@pytest.mark.parametrize("w,h", [(1, 1), (2, 5), (15, 16), (16, 16), (17, 33), (31, 3), (1, 70), (130, 67), (257, 19)])
def test_filter_at_tile_edges(r, w, h):
    rng = np.random.default_rng(1000 * w + h)
    k = rng.integers(0, 3, (h, w))
    alb = np.ones((h, w, 4), np.float32)
    alb[..., :3] = np.array([[0.3, 0.5, 0.7], [0.31, 0.5, 0.7], [0.0, 0.9, 0.2]], np.float32)[k]
    nv = np.array([0.1, 0.2, 1.0]) + 0.1 * rng.normal(size=(h, w, 3))
    nrm = np.ones((h, w, 4), np.float32)
    nrm[..., :3] = nv / np.linalg.norm(nv, axis=-1, keepdims=True) * 0.5 + 0.5
    nrm[rng.random((h, w)) < 0.1, :3] = 0.5  # pixels that saw no surface
    rad = np.ones((h, w, 4), np.float32)
    rad[..., :3] = rng.gamma(4.0, 0.25, (h, w, 3))
    got = r.denoise(rad, alb, nrm)
    ref = _ref(*(x.astype(np.float64) for x in (rad, alb, nrm)))
    assert np.all(got[..., 3] == 1.0)
    assert np.max(np.abs(got[..., :3] - ref) / np.maximum(np.abs(ref), 1e-3)) < 1e-4
