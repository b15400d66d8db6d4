"""kk_encode_pcm16 keeps its device buffer between calls up to a bound: calls of other lengths before
and after, beyond the bound, and from two threads at once encode as the oracle does; a one-shot call
that fails gives it back."""
import ctypes as C
import threading

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def wave(n, seed):
    return (np.random.default_rng(seed).standard_normal(n) * 0.5).astype(np.float32)


def same(ctx, a):
    got, clipped = ctx.encode_pcm16(a)
    want, wclip = O.encode_pcm16(a)
    return np.array_equal(got, want) and clipped == wclip


@pytest.mark.parametrize("sizes", [[1, 0, 5, 1], [24000, 100, 24001, 0, 240000, 3],
                                   [10, 2_796_000, 2_800_000, 3_000_000, 10]])
def test_lengths_in_turn(gpu_ctx, sizes):
    for i, n in enumerate(sizes):
        assert same(gpu_ctx, wave(n, i)), f"call {i}: {n} samples"


def test_two_threads(gpu_ctx):
    ok = []
    def work(seed):
        ok.append(all(same(gpu_ctx, wave(n, seed)) for n in (50000, 7, 120001, 50000)))
    ts = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert ok == [True, True]


def test_failed_one_shot_call_releases_the_buffer(gpu_ctx, monkeypatch):
    """A caller that splits its batch after KK_ERR_OOM has the whole device: no 16 MB stay behind."""
    from kokoro_hip import api, workloads
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library is bound to
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    items = workloads.small_items(5, [3])

    def fail():
        with pytest.raises(api.KKError) as e:
            gpu_ctx.forward_decoder_batch(items)
        assert e.value.code == -3

    def free():
        f, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(total)) == 0
        return f.value

    monkeypatch.setenv("KOKORO_HIP_TEST_OOM_ABOVE", "0")
    fail()  # what earlier calls kept
    before = free()
    a = wave(2_700_000, 3)  # 16.2 MB
    assert same(gpu_ctx, a)
    kept = free()
    assert before - kept >= 16_000_000
    fail()
    assert free() - kept >= 16_000_000
    assert same(gpu_ctx, a)
