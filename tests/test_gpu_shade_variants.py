"""The k_shade variants that the other tests do not reach (needs an MI355X): batches whose scenes and jobs hold no medium,
with and without textures, plain and extended, several jobs and one, eager and through the captured graph; and the cached
estimator with textures.

A job's image is bit-identical to a single render of its scene.  White textures multiply by exactly 1, so the cached
estimator (untrained, hence deterministic) makes the same image with them as without, up to samples whose threshold
comparisons fall within a rounding of their threshold: fewer than one pixel in a thousand."""
import numpy as np
import pytest
import torch

from vviewer_amd import RenderInfo, RendererPathTracing, TextureData, configs
from vviewer_amd import _ffi as F

pytestmark = pytest.mark.gpu


def _textured(scene, texels):
    t = scene.add_texture(TextureData(texels, F.TEXTURE_RGBA8_UNORM))
    for m in scene.materials:
        if m.kind != F.MATERIAL_VOLUME:
            m.tex["albedo"] = t
    return scene


def _pool(textures):
    scenes = [configs.cornell_box(), configs.cornell_glass(), configs.mesh_light_scene()]
    for s in scenes:  # a batch lights every scene with the environment of scene 0
        s.env_type, s.background, s.env_intensity, s.env_texture = (scenes[0].env_type, scenes[0].background,
                                                                    scenes[0].env_intensity, -1)
    if textures:
        rng = np.random.default_rng(5)
        for s in scenes:
            _textured(s, rng.integers(40, 256, (8, 8, 4), dtype=np.uint8))
    return scenes


JOBS = [(0, 70, 45, 8, 9, 4, 3), (1, 64, 64, 6, 8, 3, 1), (2, 33, 17, 12, 5, 4, 7), (0, 16, 16, 1, 12, 1, 0)]


def _info(w, h, spp, depth, batch, seed, extended):
    return RenderInfo(samples=spp, depth=depth, batchSize=batch, width=w, height=h, seed=seed, extended=extended)


def _batch(r, jobs, extended, graph):
    outs = [torch.full((j[2], j[1], 4), float("nan"), dtype=torch.float32, device="cuda") for j in jobs]
    r.render_jobs([(j[0], _info(*j[1:], extended)) for j in jobs], [o.data_ptr() for o in outs], extended=extended,
                  graph=graph)
    torch.cuda.synchronize()
    return [o.cpu().numpy() for o in outs]


@pytest.mark.parametrize("extended", [False, True])
@pytest.mark.parametrize("textures", [False, True])
def test_batch_without_media_equals_single_renders(textures, extended):
    scenes = _pool(textures)
    ref = []
    for sc, *rest in JOBS:
        r = RendererPathTracing(scenes[sc])
        r.renderInfo().__dict__.update(_info(*rest, extended).__dict__)
        ref.append(r.render())
        r.close()
    r = RendererPathTracing()
    r.set_scenes(scenes)
    for graph in (False, True):
        print(f"textures={textures} extended={extended} graph={graph}", flush=True)
        imgs = _batch(r, JOBS, extended, graph)
        for k, job in enumerate(JOBS):
            assert np.isfinite(imgs[k]).all() and np.array_equal(imgs[k], ref[k]), f"job {k}"
        for k, job in enumerate(JOBS):  # one job per launch
            assert np.array_equal(_batch(r, [job], extended, graph)[0], ref[k]), f"job {k} alone"
    r.close()


@pytest.mark.parametrize("make", [configs.cornell_box, configs.cornell_medium])
def test_white_textures_under_the_cached_estimator(make):
    imgs = []
    for white in (False, True):
        scene = make(160, 90)
        if white:
            _textured(scene, np.full((1, 1, 4), 255, np.uint8))
        r = RendererPathTracing(scene)
        info = r.renderInfo()
        info.samples, info.depth, info.batchSize, info.width, info.height, info.seed = 32, 8, 4, 160, 90, 5
        info.extended, info.nrc, info.nrc_untrained = True, True, True
        imgs.append(r.render())
        assert r.last_stats["nrc_queries"] > 0
        r.close()
    a, b = imgs
    assert np.isfinite(a).all() and np.isfinite(b).all()
    assert np.mean(np.any(a != b, axis=-1)) < 1e-3
