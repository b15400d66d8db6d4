"""The three resblocks of a generator stage in grouped launches (small calls) against the separate
ones: per-launch profiling runs every layer by itself, so a profiled plan must give the same audio bit
for bit; sizes on either side of the grouped path's limit for stage 0 (64 tiles of 128 columns: 410
frames) and stage 1 (64 tiles of 256: 136 frames), and of the launch order's (409, 1,200 and 2,048 frames, 8 items)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ns", [[1], [17, 40], [136], [137], [100, 100, 200], [409], [410, 3], [60] * 8, [60] * 9, [700, 500], [700, 501], [700, 700, 648], [700, 700, 649]])
def test_grouped_equals_separate(gpu_ctx, ns):
    from kokoro_hip import api, workloads
    items = workloads.small_items(200 + len(ns), ns)
    outs = []
    for prof in (False, True, False):
        gpu_ctx.set_profiling(prof)
        try:
            with api.Plan.decoder(gpu_ctx, items) as plan:
                plan.run()
                outs.append(plan.fetch())
        finally:
            gpu_ctx.set_profiling(False)
            gpu_ctx.profile_read()
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.isfinite(a).all() and np.array_equal(a, b)
