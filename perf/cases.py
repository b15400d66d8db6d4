"""The calls this library's users make, as measurable cases.

- `ids`: kk_forward_batch, phoneme ids to audio (host to host) -- what a synthesis engine calls.
- `decoder`: kk_forward_decoder_batch, durations / text features / F0 / energy to audio (host to
  host) -- the benchmark's call, and an engine's that computes prosody elsewhere.
- `generator`: a generator-only plan kept by the caller, one run and fetch of its audio.
- `snake`: kk_snake_block_noalloc, one AdaIN + Snake resblock in place on device memory.
- `pcm`: kk_encode_pcm16, a host array of samples to PCM_16 (the WAV writer's step).

Weights are random values of the real architecture (one model per process, kept on the device like
a program keeps its model); inputs come from the seed alone.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "kokoro-rust_amd"))

BLOCKS = {  # Snake blocks: (channels, kernel size)
    "noise_res.0": (256, 7), "noise_res.1": (128, 11),
    "resblocks.0": (256, 3), "resblocks.1": (256, 7), "resblocks.2": (256, 11),
    "resblocks.3": (128, 3), "resblocks.4": (128, 7), "resblocks.5": (128, 11),
}
GAP = 40              # rows between packed items of a Snake call (wider than every conv's reach)
FRAMES_PER_ID = 6.04  # what the random duration head predicts on average


def listed():
    return [
        # one word, read out at once: the smallest call of an interactive program
        {"name": "ids_word", "kind": "ids", "items": 1, "lo": 6, "hi": 6, "lengths": 1, "speed": 1.0},
        # one ordinary sentence, the usual interactive request
        {"name": "ids_sentence", "kind": "ids", "items": 1, "lo": 110, "hi": 110, "lengths": 1, "speed": 1.0},
        # a paragraph's sentences as one batch, spoken a little faster
        {"name": "ids_paragraph", "kind": "ids", "items": 6, "lo": 20, "hi": 180, "lengths": 2, "speed": 1.2},
        # a book's chapter: a full batch with lengths over the model's whole range
        {"name": "ids_chapter", "kind": "ids", "items": 32, "lo": 20, "hi": 510, "lengths": 4, "speed": 1.0},
        # the decoder half alone: one second of speech
        {"name": "decoder_second", "kind": "decoder", "items": 1, "lo": 40, "hi": 40, "lengths": 1},
        # the same for a handful of ragged sentences
        {"name": "decoder_few", "kind": "decoder", "items": 5, "lo": 60, "hi": 500, "lengths": 2},
        # the benchmark's batch: 32 ragged items of 100 to 800 frames
        {"name": "decoder_batch", "kind": "decoder", "items": 32, "lo": 100, "hi": 800, "lengths": 3},
        # generator only on a kept plan, 100 decoder frames (2.5 s of audio)
        {"name": "generator_plan", "kind": "generator", "items": 1, "lo": 100, "hi": 100, "lengths": 1},
        # one short Snake block call (a streaming chunk's rows)
        {"name": "snake_chunk", "kind": "snake", "block": "resblocks.3", "items": 1, "lo": 300, "hi": 300, "lengths": 1},
        # the 16 ragged items of 500 to 2000 rows of the one-block benchmark
        {"name": "snake_ragged", "kind": "snake", "block": "resblocks.1", "items": 16, "lo": 500, "hi": 2000, "lengths": 2},
        # the widest kernel over nearly as many rows as the entry takes
        {"name": "snake_long", "kind": "snake", "block": "resblocks.5", "items": 5, "lo": 6000, "hi": 13000, "lengths": 5},
        # ten seconds of finished audio to PCM_16
        {"name": "pcm_ten_seconds", "kind": "pcm", "samples": 240000},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["ids", "ids", "decoder", "decoder", "generator", "snake", "snake", "pcm"])
    lengths = rng.randrange(1, 1 << 20)
    if kind == "pcm":
        return {"kind": kind, "samples": _log_int(rng, 601, 2400001)}
    items = {"ids": _log_int(rng, 1, 32), "decoder": _log_int(rng, 1, 32), "generator": _log_int(rng, 1, 4),
             "snake": _log_int(rng, 1, 24)}[kind]
    top = {"ids": min(510, 9800 // items), "decoder": 800, "generator": 800, "snake": min(13000, 64000 // items - GAP)}[kind]
    hi = _log_int(rng, {"ids": 4, "decoder": 8, "generator": 8, "snake": 60}[kind], top)
    lo = max(1, int(hi * rng.uniform(0.1, 1.0)))
    case = {"kind": kind, "items": items, "lo": lo, "hi": hi, "lengths": lengths}
    if kind == "ids":
        case["speed"] = rng.choice([1.0, 1.0, 0.8, 1.25])
    if kind == "snake":
        case["block"] = rng.choice(sorted(BLOCKS))
    return case


def _lengths(case):
    rng = np.random.default_rng(case["lengths"])
    return [int(v) for v in rng.integers(case["lo"], case["hi"] + 1, case["items"])]


# ------------------------------------------------------------------ the model, kept by the program
_model = {}


def _weights():
    if "w" not in _model:
        from kokoro_hip import model_spec
        _model["w"] = model_spec.random_model_weights(seed=0)
    return _model["w"]


def _context():
    if "ctx" not in _model:
        torch.cuda.init()  # torch's runtime first: the library binds to the one that is loaded
        torch.zeros(1, device="cuda")
        from kokoro_hip import api
        ctx = api.Context(0)
        ctx.upload_model(_weights())
        _model["ctx"] = ctx
    return _model["ctx"]


class _Batch:
    """Marshalled items of a one-shot entry and the outputs of its last call (the library's pinned
    blocks, given back before the next call and when the program drops the batch)."""

    def __init__(self, prepared):
        self.pb, self.live = prepared, False

    def release(self):
        if self.live:
            self.pb.release()
            self.live = False

    def __del__(self):
        self.release()


class _View:
    def __init__(self, ptr, n):
        self.__array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": "<f4", "version": 3}


# ------------------------------------------------------------------ a case's inputs
def prepare(case, seed):
    kind = case["kind"]
    ctx = _context()
    from kokoro_hip import api, workloads
    rng = np.random.default_rng([int(seed), 77])
    if kind == "pcm":
        # speech-like levels with a few samples over full scale, as a loud voice has them
        x = rng.standard_normal(case["samples"]).astype(np.float32) * np.float32(0.25)
        return {"kind": kind, "ctx": ctx, "x": x}
    lens = _lengths(case)
    if kind == "ids":
        # the text and its prosody style are the case's, so that its predicted durations, hence the
        # audio's lengths, are the same for every seed; the voice's timbre (the half of ref_s that the
        # decoder takes) and the noise are the seed's
        text = np.random.default_rng([case["lengths"], 76])
        items = [workloads.make_ids_item(text, n, int(rng.integers(0, 2**63)), case["speed"]) for n in lens]
        for it in items:
            it.ref_s[:128] = rng.standard_normal(128)
        return {"kind": kind, "ctx": ctx, "batch": _Batch(ctx.prepare_ids(items))}
    if kind == "decoder":
        items = [workloads.make_item(rng, n, int(rng.integers(0, 2**63))) for n in lens]
        return {"kind": kind, "ctx": ctx, "batch": _Batch(ctx.prepare(items))}
    if kind == "generator":
        xs = [rng.standard_normal((512, 2 * n)).astype(np.float32) for n in lens]
        f0s = [workloads.smooth_curve(rng, 2 * n, 100.0, 300.0) for n in lens]
        styles = [rng.standard_normal(128).astype(np.float32) for _ in lens]
        seeds = [int(rng.integers(0, 2**63)) for _ in lens]
        return {"kind": kind, "plan": api.Plan.generator(ctx, xs, f0s, styles, seeds)}
    x, styles, starts, rows = _snake_inputs(case, seed)
    return {"kind": kind, "ctx": ctx, "x0": x, "x": torch.empty_like(x), "styles": styles, "starts": starts,
            "lens": lens, "rows": rows, "block": "decoder.generator." + case["block"]}


def _snake_inputs(case, seed):
    lens = _lengths(case)
    c, _ = BLOCKS[case["block"]]
    starts = [0]
    for n in lens[:-1]:
        starts.append(starts[-1] + n + GAP)
    rows = starts[-1] + lens[-1]
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    x = torch.randn(rows, c, device="cuda", generator=g)
    styles = [s for s in np.random.default_rng([int(seed), 78]).standard_normal((len(lens), 128)).astype(np.float32)]
    return x, styles, starts, rows


def run(state):
    kind = state["kind"]
    if kind == "ids":
        b = state["batch"]
        b.release()
        state["ctx"].forward_ids_prepared(b.pb)
        b.live = True
        outs = b.pb.outs
        audio = [np.asarray(_View(_address(o.audio), o.n_samples)) for o in outs]
        durs = [np.asarray(o.pred_dur[: o.n_tok]) for o in outs]
        return {"audio": audio, "pred_dur": durs}
    if kind == "decoder":
        b = state["batch"]
        b.release()
        state["ctx"].forward_prepared(b.pb)
        b.live = True
        return [np.asarray(_View(_address(o.audio), o.n_samples)) for o in b.pb.outs]
    if kind == "generator":
        state["plan"].run()
        return state["plan"].fetch()
    if kind == "snake":
        x = state["x"]
        x.copy_(state["x0"])  # the block's input, left by an earlier layer on the program's stream
        torch.cuda.current_stream().synchronize()  # the library runs on its own stream
        state["ctx"].snake_block_noalloc(state["block"], x.data_ptr(), state["rows"], state["starts"], state["lens"],
                                         state["styles"])
        return x
    pcm, clipped = state["ctx"].encode_pcm16(state["x"])
    return [pcm, clipped]


def _address(p):
    import ctypes
    return ctypes.cast(p, ctypes.c_void_p).value


# ------------------------------------------------------------------ what a pass cannot do without
def _snake_macs(c, k):
    return 6 * c * c * k  # three steps of two convolutions, per column


def _generator_work(frames):
    """(MACs, weight values) of the generator per decoder frame / in all."""
    s0 = sum(_snake_macs(256, k) for k in (3, 7, 11, 7))
    s1 = sum(_snake_macs(128, k) for k in (3, 7, 11, 11))
    ups0, ups1 = 512 * 256 * 20, 256 * 128 * 12
    n0, n1, post = 22 * 256 * 12, 22 * 128, 128 * 22 * 7
    macs = 2 * ups0 + 20 * (s0 + n0 + ups1) + 120 * (s1 + n1 + post)
    return macs * frames, s0 + s1 + ups0 + ups1 + n0 + n1 + post


def _decoder_work(frames):
    enc = 514 * 1024 * 3 + 1024 * 1024 * 3 + 514 * 1024
    dec = 1090 * 1024 * 3 + 1024 * 1024 * 3 + 1090 * 1024
    up, up1 = 1090 * 512 * 3 + 512 * 512 * 3, 1090 * 512
    macs = enc + 3 * dec + 2 * up + up1 + 512 * 64
    return macs * frames, enc + 3 * dec + up + up1 + 512 * 64


def _resblk(din, dout, up):
    return (din * dout * 3 + dout * dout * 3) * (2 if up else 1) + (din * dout if din != dout else 0)


def _upstream_work(ids, pairs, frames):
    """MACs and weight values of the stages before the decoder; pairs = sum of squared lengths."""
    albert = 4 * 768 * 768 + 2 * 768 * 2048
    token = 128 * 768 + 12 * albert + 768 * 512 + 4 * (640 + 256) * 2048 + 512 * 50 + 3 * 512 * 512 * 5
    token += (512 + 256) * 2048 + 640 * 2048
    attention = 12 * 2 * 768 * pairs
    f0n = 2 * (_resblk(512, 512, False) + _resblk(512, 256, True) + 2 * _resblk(256, 256, False))
    frame = 256 * 2048 + f0n
    return token * ids + attention + frame * frames, token - 11 * albert + frame


def work(case):
    kind = case["kind"]
    if kind == "pcm":
        return {"bytes": 6 * case["samples"], "flops": 3 * case["samples"]}
    lens = _lengths(case)
    if kind == "snake":
        c, k = BLOCKS[case["block"]]
        return {"bytes": 8 * c * sum(lens) + 2 * _snake_macs(c, k), "flops": 2 * _snake_macs(c, k) * sum(lens)}
    frames, bytes_ = sum(lens), 0
    macs = weights = 0
    if kind == "ids":
        ids = sum(n + 2 for n in lens)
        frames = int(FRAMES_PER_ID / case["speed"] * ids)
        macs, weights = _upstream_work(ids, sum((n + 2) ** 2 for n in lens), frames)
        bytes_ = 8 * ids + 1024 * len(lens)
    if kind == "decoder":
        bytes_ = 4 * frames * (512 / 5 + 4) + 1024 * len(lens)  # tokens of five frames on average
    if kind == "generator":
        bytes_ = 4 * frames * (1024 + 2) + 512 * len(lens)
    else:
        m, w = _decoder_work(frames)
        macs, weights = macs + m, weights + w
    m, w = _generator_work(frames)
    # the audio is written once; weights are read once, as the 16-bit operands the layers take
    return {"bytes": bytes_ + 2400 * frames + 2 * (weights + w), "flops": 2 * (macs + m)}


# ------------------------------------------------------------------ how far two correct programs lie apart
def tolerance(case):
    kind = case["kind"]
    if kind == "pcm":
        return "exact"
    if kind == "snake":
        # bf16 operands in six convolutions in a row: 5e-3 from 64-bit sums, and 2e-3 from a version
        # whose intermediate rows are rounded at other points
        return {"rel": 8e-3, "max": 0.1}
    # Some 60 such layers in a row and an exponential at the end: one more 16-bit rounding point in
    # the residual streams moves the audio by 5e-3, single samples by up to the signal's own level
    # where a spectrum bin's phase is decided by rounding.  With the stages before the decoder even
    # f32 sums in another order move F0, hence every harmonic's phase: the most that can be stated.
    return {"rel": 0.03 if kind == "ids" else 0.02, "max": 0.9, "differ": 0.01}


# ------------------------------------------------------------------ 64-bit results
def exact(case, seed):
    """Snake blocks in 64-bit torch; PCM_16 by its rule.  The audio has no 64-bit value: the harmonic
    source's phases are defined by a sequence of 32-bit operations on values of up to millions of
    radians, which another precision turns into another signal."""
    kind = case["kind"]
    if kind == "pcm":
        # the rule is stated in 32 bits: round(s * 32767) half to even, clamped
        v = np.rint(prepare(case, seed)["x"] * np.float32(32767.0)).astype(np.float64)
        return [np.clip(v, -32768, 32767).astype(np.int16), int(((v > 32767) | (v < -32768)).sum())]
    if kind != "snake":
        return None
    x, styles, starts, _ = _snake_inputs(case, seed)
    w, p = _weights(), "decoder.generator." + case["block"]
    k = BLOCKS[case["block"]][1]

    def t(name):
        return torch.as_tensor(w[p + name], dtype=torch.float64, device="cuda")

    def adain_snake(v, norm, alpha, style):  # v [rows][channels]
        c = v.shape[1]
        h = t(norm + ".fc.weight") @ style + t(norm + ".fc.bias")
        var, mean = torch.var_mean(v, dim=0, correction=0)
        v = (v - mean) / torch.sqrt(var + 1e-5) * t(norm + ".norm.weight") + t(norm + ".norm.bias")
        v = (1 + h[:c]) * v + h[c:]
        a = t(alpha).reshape(-1)
        return v + torch.sin(a * v) ** 2 / a

    def conv(v, name, dil):
        wt, half = t(name + ".weight"), (k - 1) * dil // 2
        z = torch.zeros(half, v.shape[1], dtype=v.dtype, device=v.device)
        v = torch.cat([z, v, z])
        n = v.shape[0] - 2 * half
        return sum(v[j * dil: j * dil + n] @ wt[:, :, j].t().contiguous() for j in range(k)) + t(name + ".bias")

    out = x.double()
    for s0, n, style in zip(starts, _lengths(case), styles):
        v, st = x[s0: s0 + n].double(), torch.as_tensor(style, dtype=torch.float64, device="cuda")
        for i, dil in enumerate((1, 3, 5)):
            h = conv(adain_snake(v, f".adain1.{i}", f".alpha1.{i}", st), f".convs1.{i}", dil)
            v = v + conv(adain_snake(h, f".adain2.{i}", f".alpha2.{i}", st), f".convs2.{i}", 1)
        out[s0: s0 + n] = v
    return out
