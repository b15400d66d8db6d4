"""Layers of few units run on the narrow convolution kernel, the same layers of a large batch on the
persistent one (launch_conv's rule): an item's results must not depend on which, bit for bit, at the
edges of both kernels' tiles (32, 64, 128 and 256 columns) and at the smallest sizes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300]


@pytest.mark.parametrize("block,c", [("noise_res.0", 256), ("resblocks.0", 256), ("resblocks.2", 256),
                                     ("noise_res.1", 128), ("resblocks.3", 128), ("resblocks.4", 128)])
def test_snake_block_alone_equals_batch(gpu_ctx, block, c):
    """Each edge length alone (a few units) and in one call with 24,000 rows of other items."""
    from kokoro_hip import api
    rng = np.random.default_rng(c + len(block))
    xs = [rng.standard_normal((c, t)).astype(np.float32) for t in EDGES + [8000, 8000, 8000]]
    styles = [rng.standard_normal(128).astype(np.float32) for _ in xs]
    prefix = "decoder.generator." + block
    with api.Plan.snake(gpu_ctx, prefix, xs, styles, gap=40) as plan:
        plan.run()
        batch = plan.fetch()
    for b, t in enumerate(EDGES):
        with api.Plan.snake(gpu_ctx, prefix, [xs[b]], [styles[b]], gap=40) as plan:
            plan.run()
            alone = plan.fetch()[0]
        assert np.isfinite(alone).all() and np.array_equal(alone, batch[b]), f"{block} t={t}"


def test_decoder_items_alone_equal_batch(gpu_ctx):
    """The decoder's, the ConvTs' and the generator's layers: item lengths around the tiles' edges."""
    from kokoro_hip import workloads
    items = workloads.small_items(81, [1, 3, 31, 32, 33, 64, 65, 127, 129, 260] + [700] * 12)
    batch = gpu_ctx.forward_decoder_batch(items)
    for b in range(10):
        alone = gpu_ctx.forward_decoder_batch([items[b]])[0]
        assert np.array_equal(alone, batch[b]), f"N={items[b].n_frames}"


def test_ids_items_alone_equal_batch():
    """The linear layers and the prosody convolutions: text lengths around the tiles' edges."""
    from kokoro_hip import api, model_spec, workloads
    ctx = api.Context(0)
    ctx.upload_model(model_spec.random_model_weights(seed=0))
    items = workloads.small_ids_items(82, [1, 6, 30, 62, 63, 126, 127] + [480] * 16)
    batch = ctx.forward_batch(items)
    for b in range(7):
        audio, dur = ctx.forward_batch([items[b]])[0]
        assert np.array_equal(dur, batch[b][1]) and np.array_equal(audio, batch[b][0]), f"{len(items[b].ids)} ids"
    ctx.close()
