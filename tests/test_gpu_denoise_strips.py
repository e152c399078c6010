"""Images of one row or one column through the denoise filter (needs an MI355X): as long as the filter's widest step has
more tiles than a launch of 256-thread rows of blocks may hold if every residue class of both axes got its own (2^24
blocks).  A pixel depends on the 62 pixels to each side of it, so the last part of a long strip equals the same pixels
denoised as a strip of their own, beyond those 62."""
import pytest
import torch

from vviewer_amd import RendererPathTracing
from vviewer_amd import _ffi as F

pytestmark = pytest.mark.gpu


def _denoise(r, imgs, w, h):
    out = torch.full_like(imgs[0], float("nan"))
    p = [t.data_ptr() for t in imgs]
    F.check(r._lib.vvpt_denoise_device(r._ctx, p[0], p[1], p[2], w, h, out.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), r._lib, r._ctx)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("n", [70, (1 << 24) + 5])
@pytest.mark.parametrize("row", [True, False])
def test_strip(row, n):
    g = torch.Generator(device="cuda").manual_seed(n)
    rad, alb, nrm = (torch.rand((n, 4), generator=g, device="cuda") for _ in range(3))
    alb = torch.round(alb * 3) / 3
    nrm[:, :2] = 0.5 + 0.1 * nrm[:, :2]
    nrm[:, 2] = 1.0
    r = RendererPathTracing()
    out = _denoise(r, [rad, alb, nrm], n if row else 1, 1 if row else n)
    assert torch.isfinite(out).all()
    # positions keep their residue class modulo the widest step, 16
    k = min(n - 1, 4096) // 16 * 16
    at = (n - k) // 16 * 16
    part = _denoise(r, [t[at:].contiguous() for t in (rad, alb, nrm)], n - at if row else 1, 1 if row else n - at)
    skip = 62 if at else 0
    assert torch.equal(out[at + skip:], part[skip:])
    r.close()
