"""Where the denoise filter may write (needs an MI355X): over each of its inputs, with the same bits as into a buffer of its
own, from both device entry points.  The image spans several of the filter's tiles, so a block that wrote over an image
other blocks still read would change them."""
import numpy as np
import pytest
import torch

from vviewer_amd import RendererPathTracing
from vviewer_amd import _ffi as F

pytestmark = pytest.mark.gpu

W, H = 259, 131


def _inputs():
    rng = np.random.default_rng(11)
    k = rng.integers(0, 3, (H, W))
    alb, nrm, rad = (np.ones((H, W, 4), np.float32) for _ in range(3))
    alb[..., :3] = np.array([[0.3, 0.5, 0.7], [0.31, 0.5, 0.7], [0.9, 0.9, 0.2]], np.float32)[k]
    nv = np.array([0.1, 0.2, 1.0]) + 0.1 * rng.normal(size=(H, W, 3))
    nrm[..., :3] = nv / np.linalg.norm(nv, axis=-1, keepdims=True) * 0.5 + 0.5
    rad[..., :3] = rng.gamma(4.0, 0.25, (H, W, 3))
    return [torch.from_numpy(a).cuda() for a in (rad, alb, nrm)]


@pytest.mark.parametrize("entry", ["vvpt_denoise_device", "vvpt_denoise_device_noalloc"])
@pytest.mark.parametrize("target", [0, 1, 2])
def test_output_over_an_input(target, entry):
    r = RendererPathTracing()
    stream = torch.cuda.current_stream().cuda_stream

    def call(imgs, out):
        p = [t.data_ptr() for t in imgs]
        F.check(getattr(r._lib, entry)(r._ctx, p[0], p[1], p[2], W, H, out.data_ptr(), stream), r._lib, r._ctx)
        torch.cuda.synchronize()
        return out.cpu().numpy()

    imgs = _inputs()
    ref = call(imgs, torch.zeros_like(imgs[0]))
    assert np.isfinite(ref).all()
    assert np.array_equal(call(imgs, imgs[target]), ref)
    # overlapping an input in part: half an image into it
    imgs = _inputs()
    both = torch.cat([imgs[target], torch.zeros_like(imgs[target])])
    part = list(imgs)
    part[target] = both[:H]
    assert np.array_equal(call(part, both[H // 2:H // 2 + H]), ref)
    r.close()
