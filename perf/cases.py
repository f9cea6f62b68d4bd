"""The performance cases of this framework: what a program that uses it has it do, through the
package's public entry points, over the sizes that such programs meet.

  live     NemotronEncoder.step for n concurrent streams (Rnnt.nemotron_step): each stream's mel
           chunk through the subsampling front-end, 24 conformer layers and joint.enc, with 70
           frames of left context cached.  80, 160, 560 and 1120 ms chunks (1, 2, 7, 14 frames).
  step     the 24 conformer layers alone (Encoder.encode_stream_step), for a program that has its
           own front-end; also with partly valid chunks (streams that end in this step).
  offline  whole-utterance relative-position attention of one layer (rel_pos_attention_batched).
  decode   the decoder's paged attention: one new token per sequence, or several (draft tokens
           checked in one call), on bf16 or f16 pages; with rope, the whole attention step (rotate q
           and k, append, attend).
  rnnt     joint.enc and greedy RNN-T decoding of one chunk of n streams.
  mel      log-mel features of a batch of clips.

Weights are random and the same for every state (a program opens a model once); inputs follow the
seed.  Linear weights are bf16-valued (half-valued for an f16 encoder), as a checkpoint of that
type holds them, so exact() sees the weights that the encoder computes with.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"


def _package():
    name = "universal_dictator_amd"
    if name not in sys.modules:
        path = os.path.join(ROOT, "universal-dictator_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


ud = _package()

LAYERS, D, HEADS, DK, FF, KC, LEFT = 24, 1024, 8, 128, 4096, 9, 70
SUB_C, MELS, HIDDEN, VOCAB = 256, 128, 640, 1025
DROP = 2                                 # frames of the pre-encode cache, dropped after subsampling


# ---------------------------------------------------------------- the cases

def listed():
    live = lambda name, n, frames: dict(name=name, kind="live", n=n, frames=frames, dtype="bf16")
    gqa = dict(kind="decode", q_heads=32, kv_heads=8, head_dim=128)
    return [
        # one person dictating: the latency of each 160 ms chunk
        live("live_1x2", 1, 2),
        # a server's 64 live streams at 160 ms
        live("live_64x2", 64, 2),
        # many streams with long chunks: the throughput end
        live("live_256x14", 256, 14),
        # a dozen-odd streams at 560 ms from an f16 checkpoint, some ending inside this chunk
        dict(name="step_13x7_f16", kind="step", n=13, frames=7, dtype="f16", ragged=True),
        # the fp32 encoder, for a few streams
        dict(name="step_4x2_f32", kind="step", n=4, frames=2, dtype="f32", ragged=False),
        # one 30 s dictation transcribed after the fact
        dict(name="offline_1x377", kind="offline", batch=1, frames=377, mask="full"),
        # a batch of two-minute recordings of unequal length
        dict(name="offline_8x1500", kind="offline", batch=8, frames=1500, mask="full"),
        # one chat or transcription session: the whole attention step of a token
        dict(gqa, name="decode_1_rope", n=1, queries=1, ctx_min=1131, ctx_max=1131, pages="f16", rope=True),
        # a serving batch, one token each
        dict(gqa, name="decode_64", n=64, queries=1, ctx_min=512, ctx_max=4096, pages="bf16", rope=False),
        # a few sequences with four draft tokens each
        dict(gqa, name="decode_12x4", n=12, queries=4, ctx_min=300, ctx_max=3000, pages="bf16", rope=False),
        # tokens of a 160 ms chunk of 64 streams at the rate of speech
        dict(name="rnnt_64x2", kind="rnnt", n=64, frames=2),
        # features of a batch of half-minute clips
        dict(name="mel_8x30s", kind="mel", n=8, samples=480011),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["live", "live", "step", "offline", "decode", "decode", "rnnt", "mel"])
    if kind in ("live", "step"):
        frames = rng.choice([1, 2, 2, 7, 14])
        dtype = rng.choice(["bf16", "bf16", "f16"]) if kind == "live" else rng.choice(["bf16", "f16", "f32"])
        c = dict(kind=kind, n=_log(rng, 1, 16 if dtype == "f32" else 200), frames=frames, dtype=dtype)
        if kind == "step":
            c["ragged"] = rng.random() < 0.5
        return c
    if kind == "offline":
        frames = _log(rng, 40, 2000)
        return dict(kind=kind, batch=rng.randint(1, max(1, min(8, 4 * 10**6 // frames**2))), frames=frames,
                    mask=rng.choice(["full", "full", "chunked"]))
    if kind == "decode":
        hq, hkv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (16, 2, 64), (8, 8, 64)])
        n, queries = _log(rng, 1, 64), rng.choice([1, 1, rng.randint(2, 8)])
        hi = _log(rng, 64, 4096)
        return dict(kind=kind, n=n, queries=queries, q_heads=hq, kv_heads=hkv, head_dim=hd,
                    ctx_min=max(8, hi // rng.randint(1, 8)), ctx_max=hi, pages=rng.choice(["bf16", "bf16", "f16"]),
                    rope=queries == 1 and rng.random() < 0.5)
    if kind == "rnnt":
        return dict(kind=kind, n=_log(rng, 1, 200), frames=rng.choice([1, 2, 7, 14]))
    return dict(kind=kind, n=_log(rng, 1, 24), samples=_log(rng, 2000, 600000))


# ---------------------------------------------------------------- helpers

class Buf:
    """Device memory of a torch tensor, as the package takes it."""

    def __init__(self, t):
        self.tensor, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _gen(*seed):
    g = torch.Generator(device=DEV)
    h = 0
    for s in seed:
        h = (h * 1000003 + int(s) + 17) % (1 << 60)
    g.manual_seed(h)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _uniform(g, bound, *shape):
    return (torch.rand(*shape, generator=g, device=DEV) * 2 - 1) * bound


def _host_ints(seed, lo, hi, n):
    return np.random.default_rng([int(seed), lo, hi]).integers(lo, hi + 1, n)


def _rounded(t, dtype):
    return t if dtype == "f32" else t.to(torch.bfloat16 if dtype == "bf16" else torch.float16).float()


def _layer_weights(layer, dtype):
    g = _gen(1, layer)
    lin = lambda o, i: _rounded(_uniform(g, math.sqrt(6 / (o + i)), o, i), dtype)
    w = {}
    for n in ("norm_feed_forward1", "norm_self_att", "norm_conv", "conv.batch_norm", "norm_feed_forward2", "norm_out"):
        w[n + ".weight"], w[n + ".bias"] = 1 + _uniform(g, 0.1, D), _uniform(g, 0.1, D)
    for n in ("feed_forward1", "feed_forward2"):
        w[n + ".linear1.weight"], w[n + ".linear2.weight"] = lin(FF, D), lin(D, FF)
    for n in ("q", "k", "v", "out", "pos"):
        w["self_attn.linear_%s.weight" % n] = lin(D, D)
    w["self_attn.pos_bias_u"], w["self_attn.pos_bias_v"] = _normal(g, HEADS, DK) * 0.02, _normal(g, HEADS, DK) * 0.02
    w["conv.pointwise_conv1.weight"], w["conv.pointwise_conv2.weight"] = lin(2 * D, D), lin(D, D)
    w["conv.depthwise_conv.weight"] = _uniform(g, math.sqrt(3 / KC), D, KC)
    return w


def _sub_weights(dtype):
    g = _gen(2)
    f3 = MELS
    for _ in range(3):
        f3 = f3 // 2 + 1
    w = {"conv.0.weight": _uniform(g, math.sqrt(6 / (9 + 9 * SUB_C)), SUB_C, 9), "conv.0.bias": _uniform(g, 1 / 3, SUB_C)}
    for i in (2, 5):
        w["conv.%d.weight" % i], w["conv.%d.bias" % i] = _uniform(g, math.sqrt(3 / 9), SUB_C, 9), _uniform(g, 1 / 3, SUB_C)
    for i in (3, 6):
        w["conv.%d.weight" % i] = _rounded(_uniform(g, math.sqrt(3 / SUB_C), SUB_C, SUB_C), dtype)
        w["conv.%d.bias" % i] = _uniform(g, 1 / 16, SUB_C)
    w["out.weight"] = _rounded(_uniform(g, math.sqrt(6 / (SUB_C * f3 + D)), D, SUB_C * f3), dtype)
    w["out.bias"] = _uniform(g, 0.02, D)
    return w


def _rnnt_weights():
    """Prediction and joint networks in torch's initial ranges; the blank's logit varies from frame
    to frame (a row of larger weights), so that streams emit a few tokens a second, as speech does."""
    g = _gen(3)
    k, p = 1 / math.sqrt(HIDDEN), "decoder.prediction.dec_rnn.lstm."
    w = {"decoder.prediction.embed.weight": _normal(g, VOCAB, HIDDEN)}
    w["decoder.prediction.embed.weight"][VOCAB - 1] = 0
    for l in range(2):
        for n in ("ih", "hh"):
            w[p + "weight_%s_l%d" % (n, l)] = _uniform(g, k, 4 * HIDDEN, HIDDEN)
            w[p + "bias_%s_l%d" % (n, l)] = _uniform(g, k, 4 * HIDDEN)
    w["joint.pred.weight"], w["joint.pred.bias"] = _uniform(g, k, HIDDEN, HIDDEN), _uniform(g, k, HIDDEN)
    w["joint.enc.weight"], w["joint.enc.bias"] = _uniform(g, 1 / 32, HIDDEN, D), _uniform(g, 1 / 32, HIDDEN)
    w["joint.joint_net.2.weight"], w["joint.joint_net.2.bias"] = _uniform(g, k, VOCAB, HIDDEN), _uniform(g, k, VOCAB)
    row = w["joint.joint_net.2.weight"][VOCAB - 1]
    w["joint.joint_net.2.weight"][VOCAB - 1] = 8 * (row - row.mean())
    w["joint.joint_net.2.bias"][VOCAB - 1] = 3.6
    return w


_kept = {}


def _encoder(frames, dtype):
    """The model as a program opens it once: 24 layers, chunks of `frames`, room for several times
    the streams of a case."""
    key = ("encoder", frames, dtype)
    if key not in _kept:
        e = ud.Encoder(ud.EncoderConfig(layers=LAYERS, max_chunk=frames, max_streams=64 if dtype == "f32" else 1024,
                                        dtype=dtype))
        for l in range(LAYERS):
            e.set_layer_weights(l, {n: t.cpu().numpy() for n, t in _layer_weights(l, dtype).items()})
        e.set_subsampling_weights({"encoder.pre_encode." + n: t.cpu().numpy() for n, t in _sub_weights(dtype).items()})
        e.finalize()
        _kept[key] = e
    return _kept[key]


def _decoder():
    if "rnnt" not in _kept:
        r = ud.Rnnt(max_streams=1024)
        r.set_weights({n: t.cpu().numpy() for n, t in _rnnt_weights().items()})
        _kept["rnnt"], _kept["slots"] = r, list(range(1024))
    return _kept["rnnt"]


class Streams:
    """n open streams of an encoder, closed with the object."""

    def __init__(self, encoder, n):
        self.list = [encoder.new_stream() for _ in range(n)]

    def __del__(self):
        for s in self.list:
            s.close()


class Slots:
    """n decoder slots in their initial state, given back with the object."""

    def __init__(self, decoder, n):
        self.free = _kept["slots"]
        self.list = [self.free.pop() for _ in range(n)]
        for s in self.list:
            decoder.reset(s)

    def __del__(self):
        self.free.extend(self.list)


# ---------------------------------------------------------------- inputs

def _history(case, seed, chunk):
    """Encoder input of a stream's earlier chunk, [n, T, D]."""
    return _normal(_gen(10, seed, chunk), case["n"], case["frames"], D) * 0.5


def _mel_rows(case):
    return 8 * (case["frames"] + DROP) - 7


def _mel(case, seed):
    return _normal(_gen(11, seed), case["n"], _mel_rows(case), MELS) * 3 - 6


def _valid(case, seed):
    if not case.get("ragged"):
        return np.full(case["n"], case["frames"], np.int32)
    v = _host_ints(seed, 0, case["frames"], case["n"])
    return np.where(_host_ints(seed + 1, 0, 3, case["n"]) == 0, v, case["frames"]).astype(np.int32)


def _prepare_stream(case, seed):
    n, T = case["n"], case["frames"]
    enc = _encoder(T, case["dtype"])
    streams = Streams(enc, n)
    x, out = torch.empty(n, T, D, device=DEV), torch.zeros(n, T, D, device=DEV)
    s = dict(kind=case["kind"], enc=enc, streams=streams, T=T, x=Buf(x), out=Buf(out))
    for c in range(LEFT // T):
        x.copy_(_history(case, seed, c))
        enc.encode_stream_step(streams.list, s["x"], s["out"], T=T)
    if case["kind"] == "live":
        s.update(rnnt=_decoder(), mel=Buf(_mel(case, seed)), rows=_mel_rows(case), valid=[_mel_rows(case)] * n,
                 keep=[False] * n, proj=Buf(torch.zeros(n, T, HIDDEN, device=DEV)))
    else:
        x.copy_(_history(case, seed, LEFT // T))
        s["valid"] = _valid(case, seed)
    return s


def _offline_inputs(case, seed):
    B, T, g = case["batch"], case["frames"], _gen(20, seed)
    q, k, v = (_normal(g, B, T, D).bfloat16() for _ in range(3))
    p = (_normal(g, 2 * T - 1, D) * 0.5).bfloat16()
    u, vb = _normal(g, HEADS, DK) * 0.02, _normal(g, HEADS, DK) * 0.02
    lens = _host_ints(seed, (3 * T + 4) // 5, T, B)
    i = np.arange(T)
    lo, hi = np.zeros(T, np.int64), np.full(T, T)
    if case["mask"] == "chunked":       # 1120 ms chunks that see 70 earlier frames
        lo, hi = np.maximum(0, i // 14 * 14 - 70), i // 14 * 14 + 14
    r = np.stack([np.broadcast_to(lo, (B, T)), np.minimum(hi[None], lens[:, None])], -1).astype(np.int32)
    return q, k, v, p, u, vb, r


def _decode_inputs(case, seed):
    n, M, hq, hkv, d = (case[k] for k in ("n", "queries", "q_heads", "kv_heads", "head_dim"))
    g, t16 = _gen(30, seed), torch.bfloat16 if case["pages"] == "bf16" else torch.float16
    lens = np.maximum(M, _host_ints(seed, case["ctx_min"], case["ctx_max"], n))
    blocks = (lens + 15) // 16
    perm = np.random.default_rng(seed).permutation(int(blocks.sum())).astype(np.int32)
    table = np.zeros((n, int(blocks.max())), np.int32)
    at = 0
    for i, b in enumerate(blocks):
        table[i, :b] = perm[at:at + b]
        at += b
    kp, vp = (_normal(g, at, hkv, 16, d).to(t16) for _ in range(2))
    q = _normal(g, n, M, hq * d)
    kn, vn = (_normal(g, n, hkv * d).to(t16) for _ in range(2))
    # query m of a sequence of L keys attends to keys 0 .. L - M + m
    ends = lens[:, None] - (M - 1) + np.arange(M)
    ranges = np.stack([np.zeros_like(ends), ends], -1).astype(np.int32)
    return q, kp, vp, kn, vn, table, lens, ranges


def _inv_freq(d):
    return (1 / np.power(1e6, 2 * np.arange(d // 2) / d)).astype(np.float32)


def _clips(case, seed):
    """Voiced sound under a slow envelope over low noise; clips of unequal length."""
    n, m, g = case["n"], case["samples"], _gen(40, seed)
    t = torch.arange(m, device=DEV, dtype=torch.float64) / 16000
    f0 = torch.rand(n, 1, generator=g, device=DEV).double() * 120 + 90
    ph = 2 * math.pi * f0 * t - 40 * torch.cos(2 * math.pi * 0.7 * t)
    x = sum(torch.sin(h * ph) / h for h in range(1, 12)) * (0.2 + 0.15 * torch.sin(2 * math.pi * 1.3 * t))
    lens = _host_ints(seed, max(1, m // 2), m, n)
    lens[0] = m
    return (0.3 * x).float() + 1e-3 * _normal(g, n, m), lens.astype(np.int64)


def _mel_tables():
    """The Slaney filterbank of 128 bins over 257 frequencies and the symmetric Hann window of 400."""
    to_hz = lambda m: m * 200 / 3 if m < 15 else 1000 * math.exp(math.log(6.4) / 27 * (m - 15))
    top = 15 + math.log(8) / (math.log(6.4) / 27)
    f = np.array([to_hz(top * i / (MELS + 1)) for i in range(MELS + 2)])
    r = f[:, None] - np.linspace(0, 8000, 257)[None]
    step = np.diff(f)[:, None]
    fb = np.maximum(0, np.minimum(-r[:-2] / step[:-1], r[2:] / step[1:])) * (2 / (f[2:] - f[:-2]))[:, None]
    return fb.astype(np.float32), (0.5 - 0.5 * np.cos(2 * np.pi * np.arange(400) / 399)).astype(np.float32)


def prepare(case, seed):
    kind, dev = case["kind"], lambda a: Buf(torch.from_numpy(np.ascontiguousarray(a)).to(DEV))
    if kind in ("live", "step"):
        return _prepare_stream(case, seed)
    if kind == "offline":
        q, k, v, p, u, vb, r = _offline_inputs(case, seed)
        return dict(kind=kind, q=Buf(q), k=Buf(k), v=Buf(v), p=Buf(p), u=Buf(u), vb=Buf(vb), r=dev(r),
                    out=Buf(torch.zeros_like(q)), B=case["batch"], T=case["frames"])
    if kind == "decode":
        q, kp, vp, kn, vn, table, lens, ranges = _decode_inputs(case, seed)
        n, M, d = case["n"], case["queries"], case["head_dim"]
        max_keys = int(lens.max())
        return dict(kind=kind, c=case, q=Buf(q), kp=Buf(kp), vp=Buf(vp), kn=Buf(kn), vn=Buf(vn), table=dev(table),
                    blocks=table.shape[1], ranges=dev(ranges), max_keys=max_keys, out=Buf(torch.zeros_like(q)),
                    pos=dev((lens - 1).astype(np.int32)), inv=dev(_inv_freq(d)),
                    ws=Buf(torch.empty(ud.gqa_workspace_bytes(n * M, case["q_heads"], d, max_keys), device=DEV,
                                       dtype=torch.uint8)))
    if kind == "rnnt":
        n, T, dec = case["n"], case["frames"], _decoder()
        return dict(kind=kind, dec=dec, slots=Slots(dec, n), n=n, T=T, enc=Buf(_normal(_gen(50, seed), n * T, D)),
                    proj=Buf(torch.zeros(n * T, HIDDEN, device=DEV)), frames=[T] * n)
    if "mel" not in _kept:
        _kept["mel"] = ud.MelFrontend(*_mel_tables())
    audio, lens = _clips(case, seed)
    rows = case["samples"] // 160 + 1
    return dict(kind=kind, mel=_kept["mel"], audio=Buf(audio), lens=lens, rows=rows, n=case["n"], stride=case["samples"],
                out=Buf(torch.zeros(case["n"], rows, MELS, device=DEV)))


# ---------------------------------------------------------------- one pass

def run(s):
    kind = s["kind"]
    if kind == "live":
        s["rnnt"].nemotron_step(s["enc"], s["streams"].list, s["mel"], s["rows"], s["valid"], s["keep"], DROP, s["T"],
                                s["proj"], s["T"])
        return s["proj"].tensor
    if kind == "step":
        s["enc"].encode_stream_step(s["streams"].list, s["x"], s["out"], valid=s["valid"], T=s["T"])
        return s["out"].tensor
    if kind == "offline":
        ud.rel_pos_attention_batched(s["q"], s["k"], s["v"], s["p"], s["T"] - 1, s["u"], s["vb"], s["r"], s["out"],
                                     s["B"], s["T"], HEADS, 2 * s["T"] - 1)
        return s["out"].tensor
    if kind == "decode":
        c = s["c"]
        n, hq, hkv, d, pages = c["n"], c["q_heads"], c["kv_heads"], c["head_dim"], c["pages"]
        if c["rope"]:
            ud.rope_rotate_half(s["q"], n, hq, d, hq * d, s["inv"], positions=s["pos"])
            ud.rope_rotate_half(s["kn"], n, hkv, d, hkv * d, s["inv"], positions=s["pos"], dtype=pages)
            ud.paged_kv_append(s["kn"], s["vn"], s["kp"], s["vp"], s["table"], s["blocks"], s["pos"], n, hkv, d,
                               kv_dtype=pages)
        if c["queries"] == 1:
            ud.gqa_attention_paged(s["q"], s["kp"], s["vp"], s["table"], s["blocks"], s["ranges"], s["out"], n, hq, hkv,
                                   d, s["max_keys"], s["ws"], kv_dtype=pages)
        else:
            ud.gqa_attention_paged_mq(s["q"], s["kp"], s["vp"], s["table"], s["blocks"], s["ranges"], s["out"], n,
                                      c["queries"], hq, hkv, d, s["max_keys"], s["ws"], kv_dtype=pages)
        return [s["out"].tensor, s["q"].tensor, s["kn"].tensor] if c["rope"] else [s["out"].tensor]
    if kind == "rnnt":
        s["dec"].project(s["n"] * s["T"], s["enc"], s["proj"])
        tokens, counts = s["dec"].greedy(s["slots"].list, s["proj"], s["T"], s["frames"], cap=10 * s["T"])
        padded = np.full((s["n"], 10 * s["T"]), -1, np.int32)
        for row, t in zip(padded, tokens):
            row[:len(t)] = t
        return [s["proj"].tensor, padded, counts]
    s["mel"].features_device(s["n"], s["audio"], s["stride"], s["lens"], s["out"], s["rows"])
    return s["out"].tensor


# ---------------------------------------------------------------- what a pass cannot do without

def _attended(case, seed=0):
    """Keys of all query rows of an offline case (the lengths follow the seed; their mean here)."""
    B, T = case["batch"], case["frames"]
    i, valid = np.arange(T), int(round(0.8 * T))
    lo, hi = np.zeros(T, np.int64), np.full(T, T)
    if case["mask"] == "chunked":
        lo, hi = np.maximum(0, i // 14 * 14 - 70), i // 14 * 14 + 14
    return B * int(np.maximum(0, np.minimum(hi, valid) - lo).sum())


def work(case):
    kind = case["kind"]
    if kind in ("live", "step"):
        n, T, size = case["n"], case["frames"], 4 if case["dtype"] == "f32" else 2
        rows, keys = n * T, LEFT + T
        layer = 4 * D * FF + 4 * D * D + 3 * D * D
        per_layer = layer * size + n * keys * D * 2 * size + n * 8 * D * 4 + (LEFT + 2 * T - 1) * D * size
        b = LAYERS * per_layer + 2 * rows * D * 4
        f = LAYERS * (2 * rows * layer + 6 * rows * keys * D + 2 * rows * KC * D)
        if kind == "live":
            m, f1, f2, f3 = _mel_rows(case), 65, 33, 17
            t1 = m // 2 + 1
            t2 = t1 // 2 + 1
            t3 = t2 // 2 + 1
            b += n * m * MELS * 4 + (2 * SUB_C * SUB_C + SUB_C * f3 * D) * size + D * HIDDEN * 4 \
                + rows * (HIDDEN - D) * 4 - rows * D * 4
            f += 2 * n * (9 * SUB_C * (t1 * f1 + t2 * f2 + t3 * f3) + SUB_C * SUB_C * (t2 * f2 + t3 * f3)) \
                + 2 * rows * SUB_C * f3 * D + 2 * rows * D * HIDDEN
        return {"bytes": b, "flops": f}
    if kind == "offline":
        B, T = case["batch"], case["frames"]
        return {"bytes": (4 * B * T + 2 * T - 1) * D * 2, "flops": 6 * _attended(case) * D}
    if kind == "decode":
        n, M, hq, hkv, d = (case[k] for k in ("n", "queries", "q_heads", "kv_heads", "head_dim"))
        keys = n * (case["ctx_min"] + case["ctx_max"]) // 2
        return {"bytes": keys * hkv * d * 4 + n * M * hq * d * 8 + keys // 16 * 4, "flops": 4 * keys * M * hq * d}
    if kind == "rnnt":
        # every frame's joint; about 0.4 predictions a frame; all weights once
        rows = case["n"] * case["frames"]
        net = 2 * 8 * HIDDEN * HIDDEN + HIDDEN * HIDDEN
        return {"bytes": 4 * (net + D * HIDDEN + VOCAB * HIDDEN + rows * (D + HIDDEN)),
                "flops": 2 * rows * (D * HIDDEN + int(1.4 * VOCAB * HIDDEN) + int(0.4 * net))}
    # a 512-point real transform of each frame and the filterbank's non-zero weights
    frames = case["n"] * (0.75 * case["samples"] // 160 + 1)
    return {"bytes": int(case["n"] * 0.75 * case["samples"] * 4 + frames * MELS * 4),
            "flops": int(frames * (2.5 * 512 * 9 + 3 * 257 + 2 * 2 * 257))}


def tolerance(case):
    """About four times the distance from exact() (24 layers: 1e-3 with 16-bit operands, 3e-6 in
    fp32; attention with bf16 probabilities: 3e-3; fp32 sums: 2e-7 to 5e-7; f16-rounded q and k:
    their last bit)."""
    kind = case["kind"]
    if kind in ("live", "step"):
        return {"rel": 1.5e-5} if case["dtype"] == "f32" else {"rel": 4e-3}
    if kind == "offline":
        return {"rel": 1.2e-2}
    if kind == "decode":
        return {"rel": 1e-2} if case["pages"] == "bf16" else {"rel": 2e-4} if case["rope"] else {"rel": 2e-6}
    if kind == "rnnt":
        return {"rel": 2e-6, "differ": 0.01}
    return {"rel": 2e-6}


# ---------------------------------------------------------------- the same in 64 bits

def _ln(x, w, name):
    return torch.nn.functional.layer_norm(x, (D,), w[name + ".weight"], w[name + ".bias"], 1e-5)


def _exact_layers(x, frames, valid, dtype):
    """All frames of n streams [n, F, D] through the layers: chunks of `frames` that see every
    earlier frame; the last chunk's rows past `valid` are not seen as keys and leave the conv."""
    n, F, _ = x.shape
    i = torch.arange(F, device=DEV)
    seen = (i[None] < (i // frames * frames + frames)[:, None])[None].repeat(n, 1, 1)
    real = i[None] < F - frames + valid[:, None]
    last = F - frames
    seen[:, last:] &= real[:, None]
    rel = torch.arange(-(F - 1), F, device=DEV).double()[:, None]
    div = torch.exp(torch.arange(0, D, 2, device=DEV).double() * -(math.log(10000.0) / D))
    pe = torch.stack([torch.sin(rel * div), torch.cos(rel * div)], -1).reshape(2 * F - 1, D)
    at = (i[:, None] - i[None] + F - 1).expand(n, HEADS, F, F)
    for l in range(LAYERS):
        w = {k: v.double() for k, v in _layer_weights(l, dtype).items()}
        ff = lambda y, m: 0.5 * torch.nn.functional.silu(_ln(y, w, "norm_" + m) @ w[m + ".linear1.weight"].T) \
            @ w[m + ".linear2.weight"].T
        x = x + ff(x, "feed_forward1")
        z = _ln(x, w, "norm_self_att")
        q, k, v = ((z @ w["self_attn.linear_%s.weight" % m].T).view(n, F, HEADS, DK).transpose(1, 2).contiguous()
                   for m in "qkv")
        p = (pe @ w["self_attn.linear_pos.weight"].T).view(2 * F - 1, HEADS, DK).permute(1, 2, 0).contiguous()
        qu, qv = q + w["self_attn.pos_bias_u"][:, None], q + w["self_attn.pos_bias_v"][:, None]
        a = qu @ k.transpose(2, 3).contiguous() + torch.gather(qv @ p, 3, at)
        a = torch.softmax((a / math.sqrt(DK)).masked_fill(~seen[:, None], -math.inf), -1)
        x = x + (a @ v).transpose(1, 2).reshape(n, F, D) @ w["self_attn.linear_out.weight"].T
        g = torch.nn.functional.glu(_ln(x, w, "norm_conv") @ w["conv.pointwise_conv1.weight"].T, -1) * real[..., None]
        g = torch.nn.functional.pad(g, (0, 0, KC - 1, 0))
        c = sum(g[:, t:t + F] * w["conv.depthwise_conv.weight"][:, t] for t in range(KC))
        x = x + torch.nn.functional.silu(_ln(c, w, "conv.batch_norm")) @ w["conv.pointwise_conv2.weight"].T
        x = _ln(x + ff(x, "feed_forward2"), w, "norm_out")
    return x


def _exact_subsample(mel, dtype):
    w = {k: v.double() for k, v in _sub_weights(dtype).items()}
    relu = torch.relu

    def conv(y, i):                       # 3x3, stride 2, two rows and columns before and one after
        y = torch.nn.functional.pad(y, (0, 0, 2, 1, 2, 1))
        t, f = (y.shape[1] - 3) // 2 + 1, (y.shape[2] - 3) // 2 + 1
        k = w["conv.%d.weight" % i]
        return sum(y[:, a:a + 2 * t - 1:2, b:b + 2 * f - 1:2] * k[:, 3 * a + b] for a in range(3) for b in range(3)) \
            + w["conv.%d.bias" % i]

    y = relu(conv(mel.double()[..., None], 0))
    y = relu(conv(y, 2) @ w["conv.3.weight"].T + w["conv.3.bias"])
    y = relu(conv(y, 5) @ w["conv.6.weight"].T + w["conv.6.bias"])
    y = y.transpose(2, 3).reshape(y.shape[0], y.shape[1], -1)
    return y @ w["out.weight"].T + w["out.bias"]


def _exact_joint_enc(y):
    w = _rnnt_weights()
    return y @ w["joint.enc.weight"].double().T + w["joint.enc.bias"].double()


def _exact_offline(case, seed):
    q, k, v, p, u, vb, r = _offline_inputs(case, seed)
    B, T = case["batch"], case["frames"]
    heads = lambda t: t.double().view(-1, HEADS, DK).transpose(0, 1).contiguous()
    out, pt = torch.empty(B, T, D, dtype=torch.float64, device=DEV), heads(p).transpose(1, 2).contiguous()
    i = torch.arange(T, device=DEV)
    at = (i[:, None] - i[None] + T - 1).expand(HEADS, T, T)
    for b in range(B):
        qb, lim = heads(q[b]), torch.from_numpy(r[b]).to(DEV)
        seen = (i[None] >= lim[:, :1]) & (i[None] < lim[:, 1:])
        a = (qb + u.double()[:, None]) @ heads(k[b]).transpose(1, 2).contiguous() \
            + torch.gather((qb + vb.double()[:, None]) @ pt, 2, at)
        a = torch.softmax((a / math.sqrt(DK)).masked_fill(~seen, -1e300), -1) * seen
        out[b] = (a @ heads(v[b])).transpose(0, 1).reshape(T, D)
    return out


def _exact_rope(x, heads, d, pos):
    a = torch.from_numpy(pos.astype(np.float32)[:, None] * _inv_freq(d)[None]).to(DEV).double()[:, None]
    lo, hi = x.double().view(len(pos), heads, 2, d // 2).unbind(2)
    return torch.cat([lo * torch.cos(a) - hi * torch.sin(a), hi * torch.cos(a) + lo * torch.sin(a)], -1).flatten(1)


def _exact_decode(case, seed):
    q, kp, vp, kn, vn, table, lens, ranges = _decode_inputs(case, seed)
    n, M, hq, hkv, d = (case[k] for k in ("n", "queries", "q_heads", "kv_heads", "head_dim"))
    rq, rk = q, kn
    if case["rope"]:
        pos = (lens - 1).astype(np.int32)
        rq, rk = _exact_rope(q[:, 0], hq, d, pos)[:, None], _exact_rope(kn, hkv, d, pos)
    out = torch.zeros(n, M, hq * d, dtype=torch.float64, device=DEV)
    for i in range(n):
        L = int(lens[i])
        pages = torch.from_numpy(table[i, :(L + 15) // 16].astype(np.int64)).to(DEV)
        k, v = (t[pages].double().transpose(1, 2).reshape(-1, hkv, d)[:L] for t in (kp, vp))
        if case["rope"]:
            k[L - 1], v[L - 1] = rk[i].view(hkv, d), vn[i].double().view(hkv, d)
        k, v = (t.repeat_interleave(hq // hkv, 1).transpose(0, 1).contiguous() for t in (k, v))
        a = rq[i].double().view(M, hq, d).transpose(0, 1) @ k.transpose(1, 2).contiguous() / math.sqrt(d)
        ends = torch.from_numpy(ranges[i, :, 1].astype(np.int64)).to(DEV)
        a = a.masked_fill(torch.arange(L, device=DEV)[None] >= ends[:, None], -math.inf)
        out[i] = (torch.softmax(a, -1) @ v).transpose(0, 1).reshape(M, hq * d)
    return [out, rq, rk] if case["rope"] else [out]


def _exact_mel(case, seed):
    audio, lens = _clips(case, seed)
    fb, window = (torch.from_numpy(a).to(DEV).double() for a in _mel_tables())
    rows = case["samples"] // 160 + 1
    out = torch.zeros(case["n"], rows, MELS, dtype=torch.float64, device=DEV)
    for b, m in enumerate(lens):
        a = audio[b, :int(m)]
        x = torch.cat([a[:1], a[1:] - 0.97 * a[:-1]]).double()
        f = torch.nn.functional.pad(x, (256, 256)).unfold(0, 512, 160)[:int(m) // 160]
        f = f * torch.nn.functional.pad(window, (56, 56))
        out[b, :f.shape[0]] = torch.log(torch.fft.rfft(f).abs().square() @ fb.T + 2.0 ** -24)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("live", "step"):
        T, n = case["frames"], case["n"]
        x = [_history(case, seed, c).double() for c in range(LEFT // T)]
        if kind == "live":
            x.append(_exact_subsample(_mel(case, seed), case["dtype"])[:, DROP:])
            valid = np.full(n, T)
        else:
            x.append(_history(case, seed, LEFT // T).double())
            valid = _valid(case, seed)
        y = _exact_layers(torch.cat(x, 1), T, torch.from_numpy(valid).to(DEV), case["dtype"])[:, LEFT:]
        return _exact_joint_enc(y) if kind == "live" else y
    if kind == "offline":
        return _exact_offline(case, seed)
    if kind == "decode":
        return _exact_decode(case, seed)
    if kind == "rnnt":
        return [_exact_joint_enc(_normal(_gen(50, seed), case["n"] * case["frames"], D).double()), None, None]
    return _exact_mel(case, seed)
