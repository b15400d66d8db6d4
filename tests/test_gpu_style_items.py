"""The style projections pick their split by the number of items and of rows (launch_style_fc): an
item's results must not depend on how many items share its call, bit for bit, at the edges of the
passes (1, 4 and 16 items) for one block's rows and for the whole table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 4, 5, 16, 17, 33])
def test_snake_block_styles(gpu_ctx, n):
    """Rows of one block: passes of four items beside each other."""
    from kokoro_hip import api
    rng = np.random.default_rng(n)
    xs = [rng.standard_normal((128, 20)).astype(np.float32) for _ in range(n)]
    styles = [rng.standard_normal(128).astype(np.float32) for _ in range(n)]
    prefix = "decoder.generator.resblocks.4"
    with api.Plan.snake(gpu_ctx, prefix, xs, styles, gap=40) as plan:
        plan.run()
        batch = plan.fetch()
    for b in (0, n // 2, n - 1):
        with api.Plan.snake(gpu_ctx, prefix, [xs[b]], [styles[b]], gap=40) as plan:
            plan.run()
            alone = plan.fetch()[0]
        assert np.isfinite(alone).all() and np.array_equal(alone, batch[b]), f"item {b} of {n}"


@pytest.mark.parametrize("n", [2, 4, 5, 16, 17])
def test_decoder_styles(gpu_ctx, n):
    """The whole table."""
    from kokoro_hip import workloads
    items = workloads.small_items(83, [5] * n)
    batch = gpu_ctx.forward_decoder_batch(items)
    for b in (0, n // 2, n - 1):
        alone = gpu_ctx.forward_decoder_batch([items[b]])[0]
        assert np.array_equal(alone, batch[b]), f"item {b} of {n}"
