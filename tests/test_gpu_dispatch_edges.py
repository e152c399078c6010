"""The branches that pick a kernel by scene and size (needs an MI355X): k_shade compiled with and without texture
sampling gives the same image where every texture is white, and the LBVH build's block scans and sort-row scans agree
with the host build byte for byte at the edges of their blocks (128 wide nodes, 2048 keys a tile, 256 tiles a round)."""
import ctypes as C

import numpy as np
import pytest

from vviewer_amd import RenderInfo, RendererPathTracing, TextureData, configs
from vviewer_amd import _ffi as F

pytestmark = pytest.mark.gpu


def _render(scene, extended, slots):
    r = RendererPathTracing(scene)
    r.set_tuning(slots=slots)
    r.renderInfo().__dict__.update(RenderInfo(samples=6, depth=9, batchSize=3, width=70, height=45, seed=3, aovs=True,
                                              extended=extended).__dict__)
    out = np.stack([r.render(), r.albedo, r.normal])
    r.close()
    return out


@pytest.mark.parametrize("extended", [False, True])
@pytest.mark.parametrize("make", [configs.cornell_box, configs.cornell_glass, lambda: configs.furnace(True),
                                  configs.mesh_light_scene, lambda: configs.volume_cube_scene(2, "mesh")])
def test_white_textures_do_not_change_the_image(make, extended):
    plain = make()
    textured = make()
    white = textured.add_texture(TextureData(np.full((1, 1, 4), 255, np.uint8), F.TEXTURE_RGBA8_UNORM))
    for m in textured.materials:
        if m.kind != F.MATERIAL_VOLUME:
            m.tex["albedo"] = white
    a, b = _render(plain, extended, 1 << 25), _render(textured, extended, 192)
    # a white texel multiplies by exactly 1 and the other slots hold the same default texels: the same bits
    assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("n", [1, 2, 3, 127, 129, 1023, 2047, 2048, 2049, 256 * 2048, 256 * 2048 + 1])
def test_lbvh_at_block_edges(n):
    rng = np.random.default_rng(n)
    c = rng.normal(size=(n, 3)).astype(np.float32)
    h = rng.uniform(0.001, 0.05, (n, 3)).astype(np.float32)
    boxes = np.concatenate([c - h, c + h], 1).astype(np.float32)
    lib = F.load_library()
    ctx = C.c_void_p()
    F.check(lib.vvpt_create(C.byref(ctx), 0))
    dev, host = F.build_lbvh(boxes, 3, ctx), F.build_lbvh(boxes, 3)
    lib.vvpt_destroy(ctx)
    for k in ("morton", "order", "inner", "leaf_refs", "nodes"):
        assert np.array_equal(dev[k], host[k]), k
    assert dev["depth"] == host["depth"]
