"""The performance cases of the engine: what a program that speaks with it has
it do, through the public entry points of the q3h binding.

Six kinds of case, each one of the library's jobs:

- "frame": whole sentences, started from prompt embeddings and continued frame
  by frame (Frame.start_batch / step / state) on the full model, 28 talker
  layers and 5 code-predictor layers, for 1 to 32 streams; f32 or Q8_0
  weights, f32 activations or the int8 products, greedy or sampled.
- "start_text": the time to the first frame of a sentence given as token ids.
- "layers": one context of a stack of a few layers: a prompt, then rows one by
  one (Context.forward, the stack adapter's only call).
- "batch": several contexts of one stack: their prompts, then steps of one row
  per context (forward_batch).
- "codec": the decoder's back part, frame rows in and samples out, a sentence
  in one call or streamed in chunks.
- "text": the text projection of a prompt.

Every pass starts from a reset (or a start), so it can be repeated. Inputs and
outputs are host arrays, as the library takes and returns them. exact() is the
same computation in float64 torch, apart from the library and its oracle.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "mormot2-qwen-tts_amd"))

import q3h  # noqa: E402
import synth  # noqa: E402

H, HEADS, KVH, HD, FFN = 1024, 16, 8, 128, 3072
QKV = (HEADS + 2 * KVH) * HD
LAYER_WEIGHTS = QKV * H + H * HEADS * HD + 3 * FFN * H
VOCAB, CP_VOCAB, GROUPS = synth.VOCAB, synth.CP_VOCAB, synth.GROUPS
TALKER_LAYERS, CP_LAYERS = synth.TALKER["layers"], synth.PREDICTOR["layers"]
PENALTY = 1.05
TEXT_VOCAB, TEXT_HIDDEN = 16384, synth.TEXT_HIDDEN  # the gather reads one row per token
CODEC_RATES, CODEC_DILS = synth.CODEC_RATES, (1, 3, 9)
CODEC_PASS = 16  # frames per device pass, the reference's CHUNK_FRAMES


def listed():
    return [
        # one row through the 5-layer stack: the smallest call, all latency
        dict(name="row", kind="layers", dtype="q8", act_q8=False, kv_f16=False, layers=5,
             rows=1, decode=0),
        # one sentence at batch 1, the reference's own use: a 48-row prompt, a
        # second of frames
        dict(name="frame_b1", kind="frame", dtype="q8", act_q8=False, streams=1, rows_min=48,
             rows_max=48, frames=12, sample=False),
        # a few sampled speakers on one card (qwen_tts default sampling)
        dict(name="frame_b4_sampled", kind="frame", dtype="q8", act_q8=False, streams=4,
             rows_min=40, rows_max=200, frames=6, sample=True),
        # a server's batch: 32 ragged prompts, int8 activations
        dict(name="frame_b32_int8", kind="frame", dtype="q8", act_q8=True, streams=32,
             rows_min=16, rows_max=256, frames=12, sample=False),
        # time to the first frame of a 40-token sentence, non-streaming
        dict(name="start_text", kind="start_text", tokens=40, streaming=False),
        # the prompt of a cloned voice or a long text, Q8_0 weights
        dict(name="prefill_q8", kind="layers", dtype="q8", act_q8=False, kv_f16=False, layers=4,
             rows=203, decode=0),
        # long form: a 2048-row context with a half-float cache, then decoding
        dict(name="long_f16", kind="layers", dtype="q8", act_q8=False, kv_f16=True, layers=4,
             rows=2048, decode=48),
        # f32 weights, 8 contexts of 512-row prompts, then batched rows
        dict(name="batch_f32", kind="batch", dtype="f32", act_q8=False, kv_f16=False, layers=4,
             contexts=8, rows=512, steps=8),
        # int8 products over 20 contexts at ordinary prompt lengths
        dict(name="batch_int8", kind="batch", dtype="q8", act_q8=True, kv_f16=False, layers=4,
             contexts=20, rows=70, steps=16),
        # sound as it is spoken: one frame per call
        dict(name="codec_stream", kind="codec", frames=12, per_call=1),
        # the sound of a whole 12.5 s sentence in one call
        dict(name="codec_sentence", kind="codec", frames=156, per_call=156),
        # the text projection of a 48-id prompt
        dict(name="text", kind="text", ids=48),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("layers", "layers", "layers", "batch", "batch", "codec", "codec", "text",
                       "frame", "start_text"))
    if kind == "layers":
        form = rng.choice(("q8", "q8", "f32", "int8"))
        return dict(kind=kind, dtype="f32" if form == "f32" else "q8", act_q8=form == "int8",
                    kv_f16=rng.random() < 0.4, layers=rng.randint(1, 5),
                    rows=_spread(rng, 1, 320 if form == "int8" else 2300),
                    decode=rng.choice((0, 0, 1, rng.randint(2, 40))))
    if kind == "batch":
        form = rng.choice(("q8", "f32", "int8", "int8"))
        return dict(kind=kind, dtype="f32" if form == "f32" else "q8", act_q8=form == "int8",
                    kv_f16=rng.random() < 0.3, layers=rng.randint(1, 4),
                    contexts=_spread(rng, 2, 40), rows=_spread(rng, 1, 300),
                    steps=rng.randint(1, 16))
    if kind == "codec":
        per_call = _spread(rng, 1, 64)
        return dict(kind=kind, frames=per_call * max(1, rng.randint(1, 96) // per_call) +
                    rng.randint(0, 5), per_call=per_call)
    if kind == "text":
        return dict(kind=kind, ids=_spread(rng, 1, 520))
    if kind == "frame":
        form = rng.choice(("q8", "q8", "int8", "f32"))
        lo = rng.randint(8, 60)
        return dict(kind=kind, dtype="f32" if form == "f32" else "q8", act_q8=form == "int8",
                    streams=_spread(rng, 1, 16 if form != "int8" else 32), rows_min=lo,
                    rows_max=lo + rng.randint(0, 100), frames=rng.randint(2, 8),
                    sample=rng.random() < 0.4)
    return dict(kind=kind, tokens=_spread(rng, 2, 200), streaming=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# tensors, made on the card from the seed


def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + part) % (1 << 62))
    return g


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


class _Matrix:
    """A weight matrix [rows][cols] as a checkpoint holds it: f32, or Q8_0
    blocks (a half-float scale and 32 quants)."""

    def __init__(self, g, rows, cols, dtype, std=0.02):
        w = _normal(g, (rows, cols), std)
        self.q = None
        if dtype == "f32":
            self.f = w
            return
        w = w.view(rows, cols // 32, 32)
        self.d = (w.abs().amax(dim=2, keepdim=True) / 127).half()
        self.q = torch.round(w / self.d.float()).clamp(-127, 127).to(torch.int8)

    def host(self):
        if self.q is None:
            return self.f.cpu().numpy()
        b = torch.cat([self.d.view(torch.uint8), self.q.view(torch.uint8)], dim=2)
        return b.flatten(1).cpu().numpy()

    def value(self):
        if self.q is None:
            return self.f.double()
        return (self.q.double() * self.d.double()).flatten(1)


def _layer(g, dtype):
    m = {"wq": (HEADS * HD, H), "wk": (KVH * HD, H), "wv": (KVH * HD, H), "wo": (H, HEADS * HD),
         "wgate": (FFN, H), "wup": (FFN, H), "wdown": (H, FFN)}
    L = {k: _Matrix(g, r, c, dtype) for k, (r, c) in m.items()}
    for k, n in (("input_norm", H), ("post_norm", H), ("q_norm", HD), ("k_norm", HD)):
        L[k] = 1 + _normal(g, (n,), 0.1)
    return L


def _stack_tensors(seed, part, layers, dtype):
    """(layers one at a time, then the final norm): a generator, so that one
    layer is held at once."""
    g = _gen(seed, part)
    for _ in range(layers):
        yield _layer(g, dtype)
    yield 1 + _normal(g, (H,), 0.1)


def _heads(seed, part, n, rows, dtype):
    g = _gen(seed, part)
    for _ in range(n):
        yield _Matrix(g, rows, H, dtype)


def _tables(seed):
    """codec_emb [3072][1024], pred_emb [15][2048][1024], tts_pad [1024]."""
    g = _gen(seed, 5)
    return (_normal(g, (VOCAB, H), 0.02), _normal(g, (GROUPS - 1, CP_VOCAB, H), 0.02),
            _normal(g, (H,), 0.02))


def _rows(seed, part, shape):
    return _normal(_gen(seed, part), shape)


def _prompt_rows(case, seed):
    """The prompt lengths of a frame case's streams."""
    r = np.random.default_rng([int(seed), 7])
    return r.integers(case["rows_min"], case["rows_max"] + 1, case["streams"]).tolist()


def _codec_tensors(seed):
    """The decoder's back part in its checkpoint layouts (synth.codec_weights'
    names and scales)."""
    g = _gen(seed, 11)
    L, D = synth.CODEC_LATENT, synth.CODEC_DIM

    def n(shape, std):
        return _normal(g, shape, std)

    w = {k: [] for k in ("up_w", "up_b", "dw_w", "dw_b", "norm_w", "norm_b", "pw1_w", "pw1_b",
                         "pw2_w", "pw2_b", "gamma")}
    for _ in range(2):
        w["up_w"].append(n((L, L, 2), L ** -0.5))
        w["up_b"].append(n((L,), 0.01))
        w["dw_w"].append(n((L, 1, 7), 0.5 * 7 ** -0.5))
        w["dw_b"].append(n((L,), 0.01))
        w["norm_w"].append(1 + n((L,), 0.1))
        w["norm_b"].append(n((L,), 0.1))
        w["pw1_w"].append(n((4 * L, L), L ** -0.5))
        w["pw1_b"].append(n((4 * L,), 0.01))
        w["pw2_w"].append(n((L, 4 * L), (4 * L) ** -0.5))
        w["pw2_b"].append(n((L,), 0.01))
        w["gamma"].append(0.1 + n((L,), 0.02))
    w["conv0_w"], w["conv0_b"] = n((D, L, 7), (7 * L) ** -0.5), n((D,), 0.01)
    w["block"] = []
    for i, rate in enumerate(CODEC_RATES):
        cin, c = D >> i, D >> (i + 1)
        b = dict(act_alpha=n((cin,), 0.1), act_beta=n((cin,), 0.1),
                 up_w=n((cin, c, 2 * rate), (2 * cin) ** -0.5), up_b=n((c,), 0.01), res=[])
        for _ in range(3):
            b["res"].append(dict(
                a1_alpha=n((c,), 0.1), a1_beta=n((c,), 0.1),
                c1_w=n((c, c, 7), 0.5 * (7 * c) ** -0.5), c1_b=n((c,), 0.01),
                a2_alpha=n((c,), 0.1), a2_beta=n((c,), 0.1),
                c2_w=n((c, c, 1), 0.5 * c ** -0.5), c2_b=n((c,), 0.01)))
        w["block"].append(b)
    w["out_alpha"], w["out_beta"] = n((D >> 4,), 0.1), n((D >> 4,), 0.1)
    w["out_w"], w["out_b"] = n((1, D >> 4, 7), 0.05 * (7 * (D >> 4)) ** -0.5), n((1,), 0.01)
    return w


def _text_tensors(seed):
    g = _gen(seed, 13)
    TH = TEXT_HIDDEN
    return (_normal(g, (TEXT_VOCAB, TH)).bfloat16(), _normal(g, (TH, TH), 0.02),
            _normal(g, (TH,), 0.02), _normal(g, (H, TH), 0.02), _normal(g, (H,), 0.02))


def _start_ids(case, seed):
    """A prompt's ids (role, text, end), its codec ids and the special ids."""
    r = np.random.default_rng([int(seed), 17])
    text = r.integers(0, TEXT_VOCAB - 16, case["tokens"]).tolist()
    im_start, im_end, assistant, nl = TEXT_VOCAB - 1, TEXT_VOCAB - 2, 77, 198
    ids = [im_start, assistant, nl] + text + [im_end, nl, im_start, assistant, nl]
    special = dict(tts_bos=TEXT_VOCAB - 5, tts_eos=TEXT_VOCAB - 4, tts_pad=TEXT_VOCAB - 3,
                   codec_pad=2148, codec_bos=2149)
    return ids, [2155, 2156, 2157, 2148, 2149], special


# ---------------------------------------------------------------------------
# prepare: the handles a program keeps


class _Session:
    """The library objects of one state, destroyed in order with it."""

    def __init__(self):
        self.dev = q3h.Device(0)
        self.keep = []

    def own(self, o):
        self.keep.append(o)
        return o

    def __del__(self):
        for o in reversed(self.keep):
            o.destroy()
        self.dev.close()


def _host(t):
    return t.cpu().numpy()


def _make_stack(ses, case, seed, part, layers, positions, heads, head_rows, kv_f16):
    dims = dict(synth.TALKER, layers=layers)
    parts = list(_stack_tensors(seed, part, layers, case["dtype"]))
    lw = [{k: v.host() if isinstance(v, _Matrix) else _host(v) for k, v in L.items()}
          for L in parts[:-1]]
    dt = q3h.F32 if case["dtype"] == "f32" else q3h.Q8_0
    s = ses.own(q3h.Stack(ses.dev, dict(dims, dtype=dt, kv_f16=int(kv_f16),
                                        act_q8=int(case["act_q8"]), max_positions=positions),
                          lw, _host(parts[-1]), dt))
    for m in _heads(seed, part + 1, heads, head_rows, case["dtype"]):
        s.add_head(m.host(), dt)
    return s


def _make_frame(ses, case, seed, streams, positions, frames):
    ts = _make_stack(ses, case, seed, 1, TALKER_LAYERS, positions, 1, VOCAB, False)
    cs = _make_stack(ses, case, seed, 3, CP_LAYERS, 16, GROUPS - 1, CP_VOCAB, False)
    ce, pe, pad = (_host(t) for t in _tables(seed))
    return ses.own(q3h.Frame(ts, cs, ce, list(pe), pad, n_streams=streams, penalty=PENALTY,
                             max_frames=frames, max_positions=positions))


def prepare(case, seed):
    kind, ses = case["kind"], _Session()
    s = dict(case=case, ses=ses)
    if kind == "layers":
        n = case["rows"] + case["decode"]
        st = _make_stack(ses, case, seed, 1, case["layers"], n, 1, VOCAB, case["kv_f16"])
        s["ctx"] = ses.own(q3h.Context(st, n))
        s["x"] = _host(_rows(seed, 7, (n, H)))
    elif kind == "batch":
        n, m = case["rows"] + case["steps"], case["contexts"]
        st = _make_stack(ses, case, seed, 1, case["layers"], n, 1, VOCAB, case["kv_f16"])
        s["ctxs"] = [ses.own(q3h.Context(st, n)) for _ in range(m)]
        s["x"] = _host(_rows(seed, 7, (n, m, H)))
        s["prompts"] = [np.ascontiguousarray(s["x"][:case["rows"], i]) for i in range(m)]
    elif kind == "frame":
        lens = _prompt_rows(case, seed)
        s["frame"] = _make_frame(ses, case, seed, case["streams"], max(lens) + case["frames"],
                                 case["frames"])
        if case["sample"]:
            s["frame"].set_sampling(do_sample=True, temperature=0.9, top_k=50, top_p=1.0,
                                    sub_do_sample=True, sub_temperature=0.9, sub_top_k=50,
                                    sub_top_p=1.0, seed=int(seed) + 1)
        s["prompts"] = [_host(_rows(seed, 100 + i, (n, H))) for i, n in enumerate(lens)]
    elif kind == "start_text":
        q8 = dict(dtype="q8", act_q8=False)
        s["frame"] = _make_frame(ses, q8, seed, 1, case["tokens"] + 32, max(64, case["tokens"]))
        emb, *rest = _text_tensors(seed)
        s["proj"] = ses.own(q3h.TextProj(ses.dev, _host(emb.view(torch.int16)).view(np.uint16),
                                         *[_host(t) for t in rest]))
        s["ids"], s["codec"], s["special"] = _start_ids(case, seed)
    elif kind == "codec":
        def host(v):
            if isinstance(v, dict):
                return {k: host(x) for k, x in v.items()}
            return [host(x) for x in v] if isinstance(v, list) else _host(v)

        s["codec"] = ses.own(q3h.Codec(ses.dev, host(_codec_tensors(seed)), CODEC_PASS))
        s["x"] = _host(_rows(seed, 7, (case["frames"], synth.CODEC_LATENT)))
    else:
        emb, *rest = _text_tensors(seed)
        s["proj"] = ses.own(q3h.TextProj(ses.dev, _host(emb.view(torch.int16)).view(np.uint16),
                                         *[_host(t) for t in rest]))
        s["ids"] = np.random.default_rng([int(seed), 19]).integers(
            0, TEXT_VOCAB, case["ids"]).astype(np.int32)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "layers":
        ctx, x, p = s["ctx"], s["x"], case["rows"]
        ctx.reset()
        out = [ctx.forward(x[:p], 0)] + [ctx.forward(x[i], 0) for i in range(p, len(x))]
        return dict(logits=np.stack([o[0] for o in out]), normed=np.stack([o[1] for o in out]))
    if kind == "batch":
        ctxs, x = s["ctxs"], s["x"]
        for c, p in zip(ctxs, s["prompts"]):
            c.reset()
            c.forward(p)
        heads = [0] * len(ctxs)
        out = [q3h.forward_batch(ctxs, x[i], heads) for i in range(case["rows"], len(x))]
        return dict(logits=np.stack([o[0] for o in out]), normed=np.stack([o[1] for o in out]))
    if kind == "frame":
        fr, n = s["frame"], case["streams"]
        fr.start_batch(list(range(n)), s["prompts"])
        codes = [fr.step()[0] for _ in range(case["frames"])]
        state = [fr.state(i) for i in range(n)]
        return dict(codes=np.stack(codes), logits=np.stack([t[0] for t in state]),
                    past=np.stack([t[1] for t in state]))
    if kind == "start_text":
        fr = s["frame"]
        fr.start_text(0, s["proj"], s["ids"], s["codec"], non_streaming=not case["streaming"],
                      **s["special"])
        codes, _ = fr.step()
        logits, past = fr.state(0)
        return dict(codes=codes, logits=logits, past=past)
    if kind == "codec":
        s["codec"].reset()
        n = case["per_call"]
        return np.concatenate([s["codec"].back(s["x"][i:i + n])
                               for i in range(0, case["frames"], n)])
    return s["proj"].project(s["ids"])


# ---------------------------------------------------------------------------
# what a pass cannot do without


def _forward_work(layers, rows, before, weight_bytes, kv_bytes, head):
    """(bytes, flops) of one forward of `rows` rows after `before` positions."""
    w = layers * LAYER_WEIGHTS + head * H
    kv = layers * 2 * KVH * HD * kv_bytes
    pairs = rows * before + rows * (rows + 1) / 2
    return (w * weight_bytes + kv * (before + rows) + rows * H * 4 + (head + H) * 4,
            2 * rows * layers * LAYER_WEIGHTS + 2 * head * H + layers * 4 * HEADS * HD * pairs)


def _frame_step_work(streams, before, weight_bytes):
    """One frame of streams at `before` talker positions each."""
    b = (TALKER_LAYERS + (GROUPS - 1) * CP_LAYERS) * LAYER_WEIGHTS
    b += VOCAB * H + (GROUPS - 1) * CP_VOCAB * H
    kv = (TALKER_LAYERS * (before + 1) + CP_LAYERS * sum(range(2, GROUPS + 1))) * 2 * KVH * HD * 4
    att = (TALKER_LAYERS * (before + 1) + CP_LAYERS * sum(range(1, GROUPS + 1))) * 4 * HEADS * HD
    rows = b + CP_LAYERS * LAYER_WEIGHTS  # the first code-predictor forward has two rows
    return b * weight_bytes + streams * (kv + 32 * H * 4), streams * (2 * rows + att)


def _codec_macs():
    L, D = synth.CODEC_LATENT, synth.CODEC_DIM
    macs, rows = 0, 1
    for _ in range(2):
        macs += rows * L * L * 2
        rows *= 2
        macs += rows * (L * 7 + 2 * 4 * L * L)
    macs += rows * D * L * 7
    for i, rate in enumerate(CODEC_RATES):
        cin, c = D >> i, D >> (i + 1)
        macs += rows * cin * c * 2 * rate
        rows *= rate
        macs += 3 * rows * c * c * 8
    return macs + rows * (D >> 4) * 7


def _codec_weight_count():
    L, D = synth.CODEC_LATENT, synth.CODEC_DIM
    n = 2 * (2 * L * L + 7 * L + 8 * L * L) + 7 * D * L + 7 * (D >> 4)
    for i, rate in enumerate(CODEC_RATES):
        cin, c = D >> i, D >> (i + 1)
        n += cin * c * 2 * rate + 3 * 8 * c * c
    return n


def work(case):
    kind = case["kind"]
    wb = 4 if case.get("dtype") == "f32" else 34 / 32
    kb = 2 if case.get("kv_f16") else 4
    parts = []
    if kind == "layers":
        parts.append(_forward_work(case["layers"], case["rows"], 0, wb, kb, VOCAB))
        parts += [_forward_work(case["layers"], 1, case["rows"] + i, wb, kb, VOCAB)
                  for i in range(case["decode"])]
    elif kind == "batch":
        # the weights once for all prompts, then once a step
        b, f = _forward_work(case["layers"], case["rows"], 0, wb, kb, 0)
        n = case["contexts"]
        once = case["layers"] * LAYER_WEIGHTS * wb
        parts.append((once + n * (b - once), n * f))
        for i in range(case["steps"]):
            b, f = _forward_work(case["layers"], 1, case["rows"] + i, wb, kb, VOCAB)
            once = (case["layers"] * LAYER_WEIGHTS + VOCAB * H) * wb
            parts.append((once + n * (b - once), n * f))
    elif kind == "frame":
        n = case["streams"]
        mean = (case["rows_min"] + case["rows_max"]) / 2
        b, f = _forward_work(TALKER_LAYERS, mean, 0, wb, kb, VOCAB)
        once = (TALKER_LAYERS * LAYER_WEIGHTS + VOCAB * H) * wb
        parts.append((once + n * (b - once), n * f))
        parts += [_frame_step_work(n, mean + i, wb) for i in range(case["frames"])]
    elif kind == "start_text":
        rows = 8 if case["streaming"] else case["tokens"] + 9
        ids = case["tokens"] + 8
        parts.append((TEXT_HIDDEN * (TEXT_HIDDEN + H) * 4 + ids * TEXT_HIDDEN * 2,
                      2 * ids * TEXT_HIDDEN * (TEXT_HIDDEN + H)))
        parts.append(_forward_work(TALKER_LAYERS, rows, 0, wb, kb, VOCAB))
        parts.append(_frame_step_work(1, rows, wb))
    elif kind == "codec":
        # the weights once for each call
        calls = -(-case["frames"] // case["per_call"])
        parts.append((calls * _codec_weight_count() * 4 + case["frames"] * (1024 + 1920) * 4,
                      2 * _codec_macs() * case["frames"]))
    else:
        parts.append((TEXT_HIDDEN * (TEXT_HIDDEN + H) * 4 + case["ids"] * (TEXT_HIDDEN * 2 + H * 4),
                      2 * case["ids"] * TEXT_HIDDEN * (TEXT_HIDDEN + H)))
    return dict(bytes=float(sum(p[0] for p in parts)), flops=float(sum(p[1] for p in parts)))


def tolerance(case):
    if case.get("act_q8"):
        # quantized activations: one documented order of every sum, the same bits
        return "exact"
    if case.get("kv_f16"):
        # a cached value next to a rounding boundary may fall to either half
        return dict(rel=1e-4, max=1e-3)
    if case["kind"] in ("frame", "start_text"):
        return dict(rel=2e-5, max=2e-4, differ=0.005)
    return dict(rel=1e-5, max=1e-4)


# ---------------------------------------------------------------------------
# the same in float64


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


class _Exact:
    """A stack in float64 with the caches of n sequences."""

    def __init__(self, seed, part, layers, dtype, kv_f16=False):
        *self.layers, self.norm = _stack_tensors(seed, part, layers, dtype)
        self.kv_f16 = kv_f16
        self.inv = (1.0 / 1e6 ** (torch.arange(64, dtype=torch.float64, device="cuda") / 64)).float()

    def _rope(self, x, pos):
        a = (pos.float()[:, None] * self.inv[None]).double()  # the fp32 angle
        c, s = a.cos()[:, None], a.sin()[:, None]
        u, v = x[..., :64], x[..., 64:]
        return torch.cat([u * c - v * s, v * c + u * s], dim=-1)

    def forward(self, xs, caches):
        """xs: per sequence [rows][H]; caches: per sequence a list of (k, v) by
        layer (changed in place). The final-normed states."""
        hs = list(xs)
        for l, L in enumerate(self.layers):
            W = {k: v.value() for k, v in L.items() if isinstance(v, _Matrix)}
            for i, h in enumerate(hs):
                n, cache = h.shape[0], caches[i]
                y = _rms(h, L["input_norm"])
                old = cache[l][0].shape[1] if l < len(cache) else 0
                pos = torch.arange(old, old + n, device="cuda")
                q = self._rope(_rms((y @ W["wq"].T).view(n, HEADS, HD), L["q_norm"]), pos)
                k = self._rope(_rms((y @ W["wk"].T).view(n, KVH, HD), L["k_norm"]), pos)
                v = (y @ W["wv"].T).view(n, KVH, HD)
                if self.kv_f16:
                    k, v = k.half().double(), v.half().double()
                k, v = k.transpose(0, 1), v.transpose(0, 1)
                if old:
                    k = torch.cat([cache[l][0], k], dim=1)
                    v = torch.cat([cache[l][1], v], dim=1)
                    cache[l] = (k, v)
                else:
                    cache.append((k, v))
                mask = torch.arange(old + n, device="cuda")[None] > pos[:, None]
                out = []
                for head in range(HEADS):
                    s = q[:, head] @ k[head * KVH // HEADS].T / math.sqrt(HD)
                    s = s.masked_fill(mask, -math.inf).softmax(-1)
                    out.append(s @ v[head * KVH // HEADS])
                h = h + torch.cat(out, dim=1) @ W["wo"].T
                y = _rms(h, L["post_norm"])
                g = y @ W["wgate"].T
                hs[i] = h + (g * torch.sigmoid(g) * (y @ W["wup"].T)) @ W["wdown"].T
        return [_rms(h, self.norm) for h in hs]


def _exact_frames(case, seed, prompts, trailing, frames):
    """Greedy frames of every stream: (talker logits, normed states)."""
    talker = _Exact(seed, 1, TALKER_LAYERS, case["dtype"])
    cp = _Exact(seed, 3, CP_LAYERS, case["dtype"])
    head = next(_heads(seed, 2, 1, VOCAB, case["dtype"])).value()
    cheads = [m.value() for m in _heads(seed, 4, GROUPS - 1, CP_VOCAB, case["dtype"])]
    ce, pe, pad = _tables(seed)
    n = len(prompts)
    caches = [[] for _ in range(n)]
    past = [y[-1] for y in talker.forward(prompts, caches)]
    logits = [head @ y for y in past]
    history = [[] for _ in range(n)]
    for f in range(frames):
        codes = []
        for i in range(n):
            s = logits[i].clone()
            s[VOCAB - 1024:] = -math.inf
            for c in set(history[i]):
                s[c] = s[c] / PENALTY if s[c] > 0 else s[c] * PENALTY
            codes.append([int(s.argmax())])
            history[i].append(codes[i][0])
        cc = [[] for _ in range(n)]
        xs = [torch.stack([past[i], ce[codes[i][0]].double()]) for i in range(n)]
        for g in range(GROUPS - 1):
            for i, y in enumerate(cp.forward(xs, cc)):
                codes[i].append(int((cheads[g] @ y[-1]).argmax()))
                xs[i] = pe[g][codes[i][-1]].double()[None]
        xs = []
        for i in range(n):
            x = ce[codes[i][0]].double()
            for g in range(GROUPS - 1):
                x = x + pe[g][codes[i][g + 1]].double()
            xs.append((x + (trailing[f] if f < len(trailing) else pad.double()))[None])
        past = [y[-1] for y in talker.forward(xs, caches)]
        logits = [head @ y for y in past]
    return torch.stack(logits).cpu().numpy(), torch.stack(past).cpu().numpy()


def _exact_project(seed, ids):
    emb, w1, b1, w2, b2 = _text_tensors(seed)
    x = emb[torch.tensor(ids, device="cuda")].double()
    x = torch.nn.functional.silu(x @ w1.double().T + b1.double())
    return x @ w2.double().T + b2.double()


def _conv(x, w, b, dil=1):
    """Causal convolution of x [T][in] with w [out][in][k]."""
    k = w.shape[2]
    x = torch.cat([x.new_zeros(((k - 1) * dil, x.shape[1])), x])
    T = x.shape[0] - (k - 1) * dil
    return sum(x[j * dil:j * dil + T] @ w[:, :, j].double().T for j in range(k)) + b.double()


def _tconv(x, w, b, stride):
    """Transposed convolution of x [T][in] with w [in][out][k], the first T
    stride samples."""
    taps, T = w.shape[2] // stride, x.shape[0]
    x = torch.cat([x.new_zeros((taps - 1, x.shape[1])), x])
    y = [sum(x[taps - 1 - i:taps - 1 - i + T] @ w[:, :, j + i * stride].double()
             for i in range(taps)) + b.double() for j in range(stride)]
    return torch.stack(y, dim=1).reshape(T * stride, w.shape[1])


def _snake(x, alpha, beta):
    a = alpha.double().exp()
    return x + (x * a).sin() ** 2 / (beta.double().exp() + 1e-9)


def _exact_codec(seed, x):
    w, F = _codec_tensors(seed), torch.nn.functional
    for i in range(2):
        x = _tconv(x, w["up_w"][i], w["up_b"][i], 2)
        p = torch.cat([x.new_zeros((6, x.shape[1])), x])
        h = sum(p[k:k + x.shape[0]] * w["dw_w"][i][:, 0, k].double() for k in range(7))
        h = F.layer_norm(h + w["dw_b"][i].double(), (x.shape[1],), w["norm_w"][i].double(),
                         w["norm_b"][i].double(), eps=1e-6)
        h = F.gelu(h @ w["pw1_w"][i].double().T + w["pw1_b"][i].double())
        x = x + w["gamma"][i].double() * (h @ w["pw2_w"][i].double().T + w["pw2_b"][i].double())
    x = _conv(x, w["conv0_w"], w["conv0_b"])
    for b, rate in zip(w["block"], CODEC_RATES):
        x = _tconv(_snake(x, b["act_alpha"], b["act_beta"]), b["up_w"], b["up_b"], rate)
        for r, dil in zip(b["res"], CODEC_DILS):
            h = _conv(_snake(x, r["a1_alpha"], r["a1_beta"]), r["c1_w"], r["c1_b"], dil)
            x = x + _conv(_snake(h, r["a2_alpha"], r["a2_beta"]), r["c2_w"], r["c2_b"])
    x = _conv(_snake(x, w["out_alpha"], w["out_beta"]), w["out_w"], w["out_b"])
    return x[:, 0].clamp(-1, 1)


def exact(case, seed):
    """None for the int8 path (its values are its rounding steps, compared bit
    for bit), for sampled frames (the draw is the library's own) and where
    float64 would take long (many streams of the full model)."""
    kind = case["kind"]
    if case.get("act_q8"):
        return None
    if kind == "layers":
        m = _Exact(seed, 1, case["layers"], case["dtype"], case["kv_f16"])
        x, p, cache = _rows(seed, 7, (case["rows"] + case["decode"], H)).double(), case["rows"], []
        y = [m.forward([x[:p]], [cache])[0][-1]]
        y += [m.forward([x[i:i + 1]], [cache])[0][-1] for i in range(p, x.shape[0])]
        y = torch.stack(y)
        head = next(_heads(seed, 2, 1, VOCAB, case["dtype"])).value()
        return dict(logits=(y @ head.T).cpu().numpy(), normed=y.cpu().numpy())
    if kind == "batch":
        m = _Exact(seed, 1, case["layers"], case["dtype"], case["kv_f16"])
        n, p = case["contexts"], case["rows"]
        x = _rows(seed, 7, (p + case["steps"], n, H)).double()
        caches = [[] for _ in range(n)]
        m.forward([x[:p, i] for i in range(n)], caches)
        y = torch.stack([torch.stack([t[0] for t in m.forward([x[j, i:i + 1] for i in range(n)],
                                                              caches)])
                         for j in range(p, p + case["steps"])])
        head = next(_heads(seed, 2, 1, VOCAB, case["dtype"])).value()
        return dict(logits=(y @ head.T).cpu().numpy(), normed=y.cpu().numpy())
    if kind == "frame":
        if case["sample"] or case["streams"] * case["frames"] > 16:
            return None
        prompts = [_rows(seed, 100 + i, (n, H)).double()
                   for i, n in enumerate(_prompt_rows(case, seed))]
        logits, past = _exact_frames(case, seed, prompts, [], case["frames"])
        return dict(codes=None, logits=logits, past=past)
    if kind == "start_text":
        ids, codec, sp = _start_ids(case, seed)
        ce = _tables(seed)[0].double()
        text = _exact_project(seed, ids[:-5])
        bos, eos, pad = _exact_project(seed, [sp["tts_bos"], sp["tts_eos"], sp["tts_pad"]])
        rows = list(text[:3]) + [(bos if i == len(codec) - 2 else pad) + ce[c]
                                 for i, c in enumerate(codec[:-1])]
        if case["streaming"]:
            rows.append(text[3] + ce[sp["codec_bos"]])
            trailing = list(text[4:]) + [eos]
        else:
            rows += [t + ce[sp["codec_pad"]] for t in text[3:]]
            rows += [eos + ce[sp["codec_pad"]], pad + ce[sp["codec_bos"]]]
            trailing = [pad]
        logits, past = _exact_frames(dict(dtype="q8"), seed, [torch.stack(rows)], trailing, 1)
        return dict(codes=None, logits=logits[0], past=past[0])
    if kind == "codec":
        return _exact_codec(seed, _rows(seed, 7, (case["frames"], synth.CODEC_LATENT)).double()) \
            .cpu().numpy()
    ids = np.random.default_rng([int(seed), 19]).integers(0, TEXT_VOCAB, case["ids"])
    return _exact_project(seed, ids.tolist()).cpu().numpy()
