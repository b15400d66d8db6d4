"""The statistics of items of at most four 256-row tiles go to AdaIN coefficients in one launch
(launch_stats_fin), those of longer items in two: an item's results must not depend on which, bit for
bit, at the edges of the tiles and of the kernel's one-, two- and four-tile forms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [1, 3, 255, 256, 257, 511, 512, 513, 768, 769, 1023, 1024, 1025]


@pytest.mark.parametrize("block,c", [("resblocks.0", 256), ("resblocks.3", 128)])
def test_alone_equals_batch(gpu_ctx, block, c):
    from kokoro_hip import api
    rng = np.random.default_rng(c)
    xs = [rng.standard_normal((c, t)).astype(np.float32) for t in EDGES]
    styles = [rng.standard_normal(128).astype(np.float32) for _ in xs]
    prefix = "decoder.generator." + block

    def run(idx):
        with api.Plan.snake(gpu_ctx, prefix, [xs[i] for i in idx], [styles[i] for i in idx], gap=40) as plan:
            plan.run()
            return plan.fetch()

    batch = run(range(len(EDGES)))  # its longest item has five tiles: two launches
    for b, t in enumerate(EDGES):
        alone = run([b])[0]
        assert np.isfinite(alone).all() and np.array_equal(alone, batch[b]), f"{block} t={t}"
    up_to = {1: [0, 1, 2, 3], 2: [1, 4, 5, 6], 4: [0, 6, 7, 8, 9, 10, 11]}
    for n, idx in up_to.items():  # ragged batches of each form
        for i, got in zip(idx, run(idx)):
            assert np.array_equal(got, batch[i]), f"{block} {n} tiles, t={EDGES[i]}"
