"""The BiLSTM recurrences on 16, 8 and 4 CUs per sequence (chosen by the number of sequences), against the
two-CU kernel (KOKORO_HIP_LSTM_QUAD=0): each row's sums are in the same order, so durations and audio
must be equal bit for bit; batch sizes on either side of every boundary (2 nb = 16, 32, 64 sequences)
and past the last, where groups run lists of sequences."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_context_stays_on_pairs_after_a_give_up():
    """Groups whose bounded wait runs out (KOKORO_HIP_TEST_LSTM_SILENT=2: a part of every group, but no
    pair, publishes nothing, 10 us limit) fall back to the one-CU kernel in the call; the context's
    next calls take pairs, whose results differ from the one-CU kernel's in the last bits."""
    from kokoro_hip import api, model_spec, workloads
    items = workloads.small_ids_items(95, [40, 12])
    ctx = api.Context(0)
    ctx.upload_model(model_spec.random_model_weights(seed=0))
    groups = ctx.forward_batch(items)
    os.environ["KOKORO_HIP_TEST_LSTM_SILENT"] = "2"
    try:
        single = ctx.forward_batch(items)
        after = ctx.forward_batch(items)
    finally:
        del os.environ["KOKORO_HIP_TEST_LSTM_SILENT"]
    assert any(not np.array_equal(a, a2) for (a, _), (a2, _) in zip(single, groups))
    for (a, d), (a2, d2) in zip(after, groups):
        assert np.array_equal(d, d2) and np.array_equal(a, a2)
    ctx.close()


@pytest.mark.parametrize("nb", [1, 8, 9, 16, 17, 32, 33])
def test_split_matches_pair(nb):
    from kokoro_hip import api, model_spec, workloads
    ctx = api.Context(0)
    ctx.upload_model(model_spec.random_model_weights(seed=0))
    rng = np.random.default_rng(nb)
    items = workloads.small_ids_items(90 + nb, [int(n) for n in rng.integers(1, 24, nb)])
    res = {}
    for sel in ("1", "0", None):
        if sel is None:
            os.environ.pop("KOKORO_HIP_LSTM_QUAD", None)
        else:
            os.environ["KOKORO_HIP_LSTM_QUAD"] = sel
        try:
            res[sel] = ctx.forward_batch(items)
        finally:
            os.environ.pop("KOKORO_HIP_LSTM_QUAD", None)
    for sel in ("1", None):
        for b, ((a, d), (a2, d2)) in enumerate(zip(res[sel], res["0"])):
            assert np.array_equal(d, d2) and np.array_equal(a, a2), (sel, b)
    ctx.close()


@pytest.mark.parametrize("nb", [9, 17, 33])
def test_split_wait_falls_back(nb):
    """The bounded wait of groups of 8, of 4, and of 4 with lists, forced from the host: the call runs
    again on the one-CU kernel, so its results are those of pairs that gave up, bit for bit."""
    from kokoro_hip import api, model_spec, workloads
    ctx = api.Context(0)
    ctx.upload_model(model_spec.random_model_weights(seed=0))
    rng = np.random.default_rng(nb)
    items = workloads.small_ids_items(97, [int(n) for n in rng.integers(1, 24, nb)])
    res = {}
    try:
        for sel, hook in (("1", "0"), ("1", "2"), ("0", "1")):
            os.environ["KOKORO_HIP_LSTM_QUAD"], os.environ["KOKORO_HIP_TEST_LSTM_SILENT"] = sel, hook
            res[sel, hook] = ctx.forward_batch(items)
    finally:
        os.environ.pop("KOKORO_HIP_LSTM_QUAD", None)
        os.environ.pop("KOKORO_HIP_TEST_LSTM_SILENT", None)
    assert any(not np.array_equal(a, a2) for (a, _), (a2, _) in zip(res["1", "2"], res["1", "0"]))
    for (a, d), (a2, d2) in zip(res["1", "2"], res["0", "1"]):
        assert np.array_equal(d, d2) and np.array_equal(a, a2)
    ctx.close()
