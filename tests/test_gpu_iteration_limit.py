"""vvpt_options.max_iterations is the limit itself (needs an MI355X): the message of a render that runs into it names the
caller's number, whatever the depth, and a limit of as many iterations as the render takes lets it finish."""
import pytest

from vviewer_amd import RenderInfo, RendererPathTracing, configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [1, 2, 8])
def test_limit_is_taken_as_given(depth):
    r = RendererPathTracing(configs.cornell_box())
    r.renderInfo().__dict__.update(RenderInfo(samples=64, depth=depth, batchSize=64, width=64, height=64).__dict__)
    ref = r.render()
    n = r.last_stats["iterations"]
    for limit in (4, 8):
        assert limit < n
        r.set_options(max_iterations=limit)
        with pytest.raises(RuntimeError, match=f"VVPT_TIMEOUT.*within {limit} wavefront iterations"):
            r.render()
    r.set_options(max_iterations=n)
    assert (r.render() == ref).all() and r.last_stats["iterations"] == n
    r.close()


def test_limit_of_a_batch_with_a_shallow_job():
    r = RendererPathTracing()
    r.set_scenes([configs.cornell_box()])
    import torch
    infos = [RenderInfo(samples=32, depth=d, batchSize=32, width=32, height=32) for d in (1, 8)]
    outs = [torch.zeros((32, 32, 4), dtype=torch.float32, device="cuda") for _ in infos]
    r.set_options(max_iterations=8)
    with pytest.raises(RuntimeError, match="VVPT_TIMEOUT.*within 8 wavefront iterations"):
        r.render_jobs([(0, i) for i in infos], [o.data_ptr() for o in outs])
    r.close()
