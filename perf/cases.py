"""The work a user of this library has it do, as measurable cases.

Every case is one pass through the public entry points of the Python binding
(`qtts.py`, one C entry point each): the Q4 row and row-block products, the
text projection, the prompt prefills, single steps, the frame loop, the
batched loop and the speech decoder, at the 1.7B shapes with random-init
weights.  Models are made once per process and kept, as a program does that
serves more than one request; inputs, buffers and caches belong to a state.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "qora-tts-12hz-1.7b_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import qtts  # noqa: E402

TALKER, PREDICTOR, GROUPS = qtts.TALKER_1P7B, qtts.PREDICTOR_1P7B, qtts.NUM_GROUPS
SAMPLES_PER_FRAME = 1920
WEIGHT_SEED = 1


def listed():
    return [
        # The smallest call: `gemv` of one row from and to host memory, as the
        # crate calls it for one projection (o_proj's shape).
        {"name": "row_host", "kind": "gemv_host", "k": 2048, "n": 2048},
        # One row through the fused gate|up weight of every talker layer, on
        # device buffers: what a caller with its own decode loop enqueues.
        {"name": "row_layers", "kind": "gemv", "k": 2048, "n": 12288, "weights": 28},
        # 64 rows through 20 different gate|up weights: a short prompt's
        # projections, weights coming from memory as in a whole prefill.
        {"name": "rows_64", "kind": "gemm", "rows": 64, "k": 2048, "n": 12288, "weights": 20},
        # 1000 rows (no multiple of a tile) through one down projection.
        {"name": "rows_1000", "kind": "gemm", "rows": 1000, "k": 6144, "n": 2048, "weights": 1},
        # The text projection of a paragraph's tokens (build_trailing_text).
        {"name": "text_96", "kind": "text", "tokens": 96},
        # The prompt that every request starts with: 10 rows, then the head.
        {"name": "prompt", "kind": "prompt", "tokens": 12, "voice": False},
        # A long prompt (1064 rows, no multiple of a tile) and the first
        # single steps after it, each reading the whole cache.
        {"name": "context_1064", "kind": "context", "rows": 1064, "steps": 4, "capacity": 2064},
        # The crate's own frame loop with each call replaced one by one:
        # sampler, semantic row, acoustic codes, embedding sum, talker step.
        {"name": "frames_4", "kind": "frames", "frames": 4, "capacity": 592},
        # A short request from token ids to audio: prompt, trailing text,
        # frame loop, decoder.
        {"name": "speech_24", "kind": "speech", "tokens": 12, "frames": 24, "capacity": 592},
        # Sixteen requests at once: their prefills, then the lockstep loop.
        {"name": "batch_16", "kind": "batch", "streams": 16, "rows": 64, "frames": 16, "capacity": 592},
        # One second of audio from host codes to host samples (streaming).
        {"name": "decode_13", "kind": "decode", "frames": 13, "device": False},
        # 40 seconds of audio on device buffers.
        {"name": "decode_500", "kind": "decode", "frames": 500, "device": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv_host", "gemv", "gemm", "gemm", "text", "prompt", "context", "frames", "speech", "batch",
                       "decode", "decode"])
    if kind == "gemv_host":
        return {"kind": kind, "k": _log(rng, 100, 6144), "n": 32 * _log(rng, 8, 384)}
    if kind == "gemv":
        return {"kind": kind, "k": 8 * _log(rng, 32, 768), "n": 32 * _log(rng, 8, 384), "weights": _log(rng, 1, 20)}
    if kind == "gemm":
        k, n, rows = 16 * _log(rng, 16, 384), 32 * _log(rng, 8, 384), _log(rng, 2, 1000)
        most = max(1, int(20 * 64 * 2048 * 12288 / (float(rows) * k * n)))
        return {"kind": kind, "rows": rows, "k": k, "n": n, "weights": min(most, rng.randint(1, 8))}
    if kind == "text":
        return {"kind": kind, "tokens": _log(rng, 1, 96)}
    if kind == "prompt":
        return {"kind": kind, "tokens": rng.randint(0, 60), "voice": rng.random() < 0.5}
    if kind == "context":
        rows, steps = _log(rng, 8, 1064), rng.randint(1, 4)
        return {"kind": kind, "rows": rows, "steps": steps, "capacity": rows + steps + _log(rng, 1, 4000)}
    if kind == "frames":
        return {"kind": kind, "frames": rng.randint(1, 4), "capacity": _log(rng, 64, 8192)}
    if kind == "speech":
        return {"kind": kind, "tokens": rng.randint(1, 40), "frames": rng.randint(4, 24),
                "capacity": _log(rng, 64, 8192)}
    if kind == "batch":
        return {"kind": kind, "streams": rng.randint(2, 16), "rows": rng.randint(8, 64), "frames": rng.randint(2, 16),
                "capacity": _log(rng, 96, 2064)}
    return {"kind": kind, "frames": _log(rng, 1, 500), "device": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# Models, made once
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _ctx():
    return qtts.Context(0)


@functools.lru_cache(maxsize=None)
def _host_talker():
    return qtts.TalkerWeights(WEIGHT_SEED, TALKER)


@functools.lru_cache(maxsize=None)
def _host_text():
    return qtts.TextWeights(WEIGHT_SEED)


@functools.lru_cache(maxsize=None)
def _host_decoder():
    return qtts.DecoderWeights(WEIGHT_SEED)


def _host_q4(k, n, i):
    return qtts.Q4Weight.synthetic(WEIGHT_SEED, f"cases.{k}.{n}.{i}", k, n)


@functools.lru_cache(maxsize=4)
def _weights(k, n, count):
    return [qtts.DeviceQ4(_ctx(), _host_q4(k, n, i)) for i in range(count)]


@functools.lru_cache(maxsize=None)
def _talker():
    t = qtts.Talker(_ctx(), _host_talker())
    t.attach_text(_host_text())
    return t


@functools.lru_cache(maxsize=None)
def _predictor():
    return qtts.CodePredictor(_ctx(), qtts.CodePredictorWeights(WEIGHT_SEED, PREDICTOR, talker_hidden=TALKER.hidden))


@functools.lru_cache(maxsize=None)
def _decoder():
    return qtts.SpeechDecoder(_ctx(), _host_decoder())


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------
def _activations(seed, rows, k):
    """N(0, 1) rows with channels of unequal size, as normed hidden states have them."""
    r = np.random.default_rng([seed, rows, k])
    x = r.standard_normal((rows, k), dtype=np.float32)
    return x * np.exp(0.5 * r.standard_normal(k, dtype=np.float32))


def _rows(seed, tag, rows, std=1.0):
    r = np.random.default_rng([seed, tag, rows])
    return std * r.standard_normal((rows, TALKER.hidden), dtype=np.float32)


def _tokens(seed, n):
    return np.random.default_rng([seed, 77]).integers(0, 151643, n).astype(np.uint32)


def _prompt_inputs(case, seed):
    r = np.random.default_rng([seed, 78])
    voice = _rows(seed, 79, 1)[0] if case.get("voice") else None
    return {"tokens": _tokens(seed, case["tokens"]), "speaker": int(r.integers(0, 2048)),
            "language": int(r.integers(2050, 2074)), "voice": voice}


def _codes(seed, frames):
    c = _host_decoder().cfg
    return np.random.default_rng([seed, 80]).integers(0, c.codebook_size, (c.num_rest + 1, frames)).astype(np.uint32)


def _speech_params(frames):
    return qtts.loop_params(frames, temperature=0.8, top_k=50, repetition_penalty=1.05, stop_on_eos=False)


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case, "seed": seed}
    if kind == "gemv_host":
        s["w"] = _weights(case["k"], case["n"], 1)[0]
        s["x"] = _activations(seed, 1, case["k"])[0]
    elif kind in ("gemv", "gemm"):
        rows = case.get("rows", 1)
        s["w"] = _weights(case["k"], case["n"], case["weights"])
        s["x"] = torch.from_numpy(_activations(seed, rows, case["k"])).cuda()
        s["y"] = torch.empty((case["weights"], rows, case["n"]), dtype=torch.float32, device="cuda")
    elif kind == "text":
        s["talker"] = _talker()
        s["tokens"] = _tokens(seed, case["tokens"])
    elif kind == "prompt":
        s["talker"] = _talker()
        s["kv"] = s["talker"].new_kv(592)
        s.update(_prompt_inputs(case, seed))
    elif kind == "context":
        s["talker"] = _talker()
        s["kv"] = s["talker"].new_kv(case["capacity"])
        s["x"] = _rows(seed, 1, case["rows"])
        s["steps"] = _rows(seed, 2, case["steps"])
    elif kind == "frames":
        s["talker"], s["predictor"] = _talker(), _predictor()
        s["kv"], s["pkv"] = s["talker"].new_kv(case["capacity"]), s["predictor"].new_kv()
        s.update(_prompt_inputs({"tokens": 12}, seed))
        s["text"] = _rows(seed, 3, case["frames"], 0.1)
    elif kind == "speech":
        s["talker"], s["predictor"], s["decoder"] = _talker(), _predictor(), _decoder()
        s["kv"], s["pkv"] = s["talker"].new_kv(case["capacity"]), s["predictor"].new_kv()
        s.update(_prompt_inputs(case, seed))
    elif kind == "batch":
        s["talker"], s["predictor"] = _talker(), _predictor()
        s["kvs"] = [s["talker"].new_kv(case["capacity"]) for _ in range(case["streams"])]
        s["x"] = [_rows(seed, 100 + b, case["rows"]) for b in range(case["streams"])]
        s["text"] = _rows(seed, 4, 8 * case["streams"], 0.1).reshape(case["streams"], 8, -1)
        s["pad"] = _rows(seed, 5, 1, 0.1)[0]
        s["seeds"] = [seed * 64 + b + 1 for b in range(case["streams"])]
    else:
        s["decoder"] = _decoder()
        s["codes"] = _codes(seed, case["frames"])
        if case["device"]:
            s["n"] = s["decoder"].num_samples(case["frames"])
            s["d_codes"] = torch.from_numpy(s["codes"].astype(np.int32)).cuda()
            s["d_audio"] = torch.empty(s["n"], dtype=torch.float32, device="cuda")
    return s


def run(s):
    return globals()["_run_" + s["kind"]](s)


def _run_gemv_host(s):
    return s["w"].gemv(s["x"])


def _run_gemv(s):
    x, y = s["x"].data_ptr(), s["y"]
    for i, w in enumerate(s["w"]):
        w.gemv_device(x, y[i].data_ptr())
    return y


def _run_gemm(s):
    x, y, rows = s["x"].data_ptr(), s["y"], s["case"]["rows"]
    for i, w in enumerate(s["w"]):
        w.gemm_device(x, rows, y[i].data_ptr())
    return y


def _run_text(s):
    return s["talker"].build_trailing_text(s["tokens"])


def _prompt(s):
    s["kv"].clear()
    return s["talker"].prefill_custom_voice(s["tokens"], s["speaker"], s["language"], s["kv"], s.get("voice"))


def _run_prompt(s):
    hidden, logits, position = _prompt(s)
    return {"hidden": hidden, "logits": logits, "position": position}


def _run_context(s):
    t, kv, n = s["talker"], s["kv"], s["case"]["rows"]
    kv.clear()
    hidden = t.prefill_talker_raw(s["x"], n, kv)
    logits = t.apply_codec_head(hidden)
    steps = [t.forward_with_embedding(e, kv, n + i) for i, e in enumerate(s["steps"])]
    return {"hidden": hidden, "logits": logits, "steps": np.stack(steps)}


def _run_frames(s):
    t, p, kv, ctx = s["talker"], s["predictor"], s["kv"], s["talker"].ctx
    hidden, logits, position = _prompt(s)
    prev, rng, outs, codes = [0] * 16, s["seed"] + 1, [], []
    for i in range(s["case"]["frames"]):
        token, rng = ctx.sample_token(logits, 0.8, 50, 1.05, prev, rng)
        prev = [token] + prev[:15]
        semantic = t.embed_codec_token(token)
        acoustic = p.generate_acoustic_codes(hidden, semantic, s["pkv"])
        codes.append(np.concatenate([[token], acoustic.astype(np.int64)]))
        out = t.forward_with_embedding(semantic + p.get_acoustic_embeddings_sum(acoustic) + s["text"][i], kv,
                                       position + i)
        hidden, logits = out[: TALKER.hidden], out[TALKER.hidden:]
        outs.append(out)
    return {"codes": np.stack(codes), "steps": np.stack(outs)}


def _run_speech(s):
    t = s["talker"]
    hidden, logits, position = _prompt(s)
    trailing = t.build_trailing_text(s["tokens"])
    pad = t.embed_text_token(qtts.TTS_PAD)
    codes = qtts.generate_codes(t, s["predictor"], s["kv"], s["pkv"], hidden, logits, position, trailing, pad,
                                _speech_params(s["case"]["frames"]), s["seed"] + 1)
    codes[0] %= 2048  # random weights also draw control tokens, which have no codebook row
    audio = s["decoder"].decode_to_audio(codes)
    return {"hidden": hidden, "logits": logits, "codes": codes, "audio": audio}


def _run_batch(s):
    t, n = s["talker"], s["case"]["rows"]
    hidden, logits = [], []
    for kv, x in zip(s["kvs"], s["x"]):
        kv.clear()
        hidden.append(t.prefill_talker_raw(x, n, kv))
        logits.append(t.apply_codec_head(hidden[-1]))
    hidden, logits = np.stack(hidden), np.stack(logits)
    codes = qtts.generate_codes_batch(t, s["predictor"], s["kvs"], hidden, logits, [n] * len(s["kvs"]), s["text"],
                                      s["pad"], _speech_params(s["case"]["frames"]), s["seeds"])
    return {"hidden": hidden, "logits": logits, "codes": np.stack(codes)}


def _run_decode(s):
    if not s["case"]["device"]:
        return s["decoder"].decode_to_audio(s["codes"])
    f = s["case"]["frames"]
    s["decoder"].decode_to_audio_device(s["d_codes"].data_ptr(), f, f, s["d_audio"].data_ptr(), s["n"])
    return s["d_audio"]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _q4_bytes(k, n):
    return k * n // 2 + k * (n // 32) * 2


def _stack_layer(c):
    """(bytes, weights) of one layer's Q4 matrices."""
    qd, kd = c.heads * c.head_dim, c.kv_heads * c.head_dim
    shapes = [(c.hidden, qd + 2 * kd), (qd, c.hidden), (c.hidden, 2 * c.inter), (c.inter, c.hidden)]
    return sum(_q4_bytes(*s) for s in shapes), sum(k * n for k, n in shapes)


def _add(*works):
    return {k: float(sum(w[k] for w in works)) for k in ("bytes", "flops")}


def _times(n, w):
    return {k: n * v for k, v in w.items()}


def _gemm_work(rows, k, n):
    return {"bytes": _q4_bytes(k, n) + 4 * rows * (k + n), "flops": 2.0 * rows * k * n}


def _prefill_work(rows):
    """All layers over `rows` new rows, the cache written, the last row's head."""
    c = TALKER
    b, w = _stack_layer(c)
    kv = 2 * rows * c.kv_heads * c.head_dim * 4
    attn = 4.0 * c.heads * c.head_dim * rows * (rows + 1) / 2
    return {"bytes": c.layers * (b + kv) + _q4_bytes(c.hidden, c.vocab) + 4 * rows * c.hidden,
            "flops": c.layers * (2.0 * rows * w + attn) + 2.0 * c.hidden * c.vocab}


def _step_work(cached, streams=1):
    """One talker step of `streams` rows over `cached` positions each."""
    c = TALKER
    b, w = _stack_layer(c)
    kv = 2 * (cached + 1) * c.kv_heads * c.head_dim * 4
    return {"bytes": c.layers * (b + streams * kv) + _q4_bytes(c.hidden, c.vocab),
            "flops": streams * (c.layers * (2.0 * w + 4.0 * c.heads * c.head_dim * (cached + 1))
                                + 2.0 * c.hidden * c.vocab)}


def _predictor_work(streams=1):
    """One frame's 15 passes: the layers and one head each, input rows projected."""
    c = PREDICTOR
    b, w = _stack_layer(c)
    passes, tokens = GROUPS, GROUPS + 1
    return {"bytes": passes * (c.layers * b + _q4_bytes(c.hidden, c.vocab)) + _q4_bytes(TALKER.hidden, c.hidden),
            "flops": streams * (2.0 * tokens * (c.layers * w + TALKER.hidden * c.hidden)
                                + 2.0 * passes * c.hidden * c.vocab)}


def _text_work(tokens):
    h = TALKER.hidden
    return _add(_gemm_work(tokens, h, h), _gemm_work(tokens, h, h))


def _decoder_work(frames):
    c, T = qtts.DECODER_1P7B, frames
    ad, flops, weights = c.heads * c.head_dim, 0.0, 0.0

    def lin(k, n, length):
        nonlocal flops, weights
        flops += 2.0 * k * n * length
        weights += k * n

    lin(c.codebook_dim, c.vq_dim, 2 * T)
    lin(3 * c.vq_dim, c.latent, T)
    lin(c.latent, c.hidden, 2 * T)
    for _ in range(c.layers):
        lin(c.hidden, 4 * ad + 3 * c.inter, T)
        flops += 4.0 * ad * sum(min(t + 1, c.window) for t in range(T))
    L = T
    for stride in c.upsample:
        lin(c.latent, c.latent * stride, L)
        L *= stride
        lin(c.latent, c.convnext_kernel + 2 * c.latent * c.convnext_mult, L)
    lin(7 * c.latent, c.vocos_channels, L)
    for cin, cout, k, stride in c.vocos:
        lin(cin * k, cout, L)
        L *= stride
        for _ in c.dilations:
            lin(cout * (c.res_kernel + 1), cout, L)
    lin(c.vocos[-1][1] * c.out_kernel, 1, L)
    return {"bytes": 4 * weights + 4.0 * L + 4 * (c.num_rest + 1) * T * (1 + c.codebook_dim), "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "gemv_host":
        return _gemm_work(1, case["k"], case["n"])
    if kind in ("gemv", "gemm"):
        return _times(case["weights"], _gemm_work(case.get("rows", 1), case["k"], case["n"]))
    if kind == "text":
        return _text_work(max(1, case["tokens"]))
    prompt = _add(_text_work(6), _prefill_work(10))
    if kind == "prompt":
        return prompt
    if kind == "context":
        return _add(_prefill_work(case["rows"]), *[_step_work(case["rows"] + i) for i in range(case["steps"])])
    if kind == "frames":
        return _add(prompt, *[_add(_step_work(10 + i), _predictor_work()) for i in range(case["frames"])])
    if kind == "speech":
        return _add(prompt, _text_work(case["tokens"]), _decoder_work(case["frames"]),
                    *[_add(_step_work(10 + i), _predictor_work()) for i in range(case["frames"])])
    if kind == "batch":
        b = case["streams"]
        return _add(_times(b, _prefill_work(case["rows"])),
                    *[_add(_step_work(case["rows"] + i, b), _predictor_work(b)) for i in range(case["frames"])])
    return _decoder_work(case["frames"])


def tolerance(case):
    """About four times the distance from the same in 64 bits: 1.3e-6 for a
    block of rows (f32 sums of split products), 0.9e-6 for the logits after 28
    layers, 9.4e-6 for the decoder's chain of stages.  Codes are whole numbers:
    two logits that are equal to rounding may swap."""
    kind = case["kind"]
    if kind in ("gemv_host", "gemv", "gemm", "text"):
        return {"rel": 5e-6}
    if kind == "decode":
        return {"rel": 4e-5}
    if kind == "speech":
        return {"rel": 4e-5, "differ": 0.01}
    if kind in ("frames", "batch"):
        return {"rel": 1e-5, "differ": 0.01}
    return {"rel": 1e-5}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(_DEV).double()


def _f16bits(a):
    return _f64(np.ascontiguousarray(a).view(np.float16))


def _dequant(w):
    """Q4 [k][n]: two nibbles a byte, low one first, less 8, times the scale of 32 columns."""
    b = torch.from_numpy(w.packed).to(_DEV)
    q = torch.stack([b & 15, b >> 4], dim=-1).reshape(w.k, w.n).double() - 8.0
    return q * _f16bits(w.scales).repeat_interleave(32, dim=1)


def _rms(x, gamma, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gamma


def _rope(x, pos, theta):
    """x [L][heads][hd], pairs (i, i + hd/2)."""
    hd = x.shape[-1]
    freq = theta ** (-torch.arange(hd // 2, dtype=torch.float64, device=_DEV) * 2.0 / hd)
    ang = (pos.double()[:, None] * freq)[:, None, :]
    a, b = x[..., : hd // 2], x[..., hd // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _attend(q, k, v, mask):
    """q [R][nq][hd], k and v [L][nkv][hd], mask [R][L] of what a row sees."""
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        sc = (q[:, h] @ k[:, h].T.contiguous()) / math.sqrt(q.shape[-1])
        out[:, h] = torch.softmax(sc.masked_fill(~mask, -math.inf), -1) @ v[:, h].contiguous()
    return out


def _talker_rows(x, streams=1):
    """The layers over `streams` equal runs of rows, each at positions 0.. (row i sees
    0..i of its own run); the final-normed rows."""
    w, c = _host_talker(), TALKER
    n = x.shape[0]
    row = torch.arange(n, device=_DEV)
    pos, run_of = row % (n // streams), row // (n // streams)
    mask = (pos[None, :] <= pos[:, None]) & (run_of[None, :] == run_of[:, None])
    for L in w.layers:
        xn = _rms(x, _f16bits(L.input_norm_gamma), 1e-6)
        q = (xn @ _dequant(L.q_proj)).reshape(n, c.heads, c.head_dim)
        k = (xn @ _dequant(L.k_proj)).reshape(n, c.kv_heads, c.head_dim)
        v = (xn @ _dequant(L.v_proj)).reshape(n, c.kv_heads, c.head_dim)
        q = _rope(_rms(q, _f16bits(L.q_norm), 1e-6), pos, c.rope_theta)
        k = _rope(_rms(k, _f16bits(L.k_norm), 1e-6), pos, c.rope_theta)
        x = x + _attend(q, k, v, mask).reshape(n, -1) @ _dequant(L.o_proj)
        xn = _rms(x, _f16bits(L.post_attn_norm_gamma), 1e-6)
        gate = xn @ _dequant(L.gate_proj)
        x = x + (gate * torch.sigmoid(gate) * (xn @ _dequant(L.up_proj))) @ _dequant(L.down_proj)
    return _rms(x, _f16bits(w.final_norm_gamma), 1e-6)


def _text_rows(tokens):
    w = _host_text()
    e = w.text_embedding
    idx = np.asarray(tokens, dtype=np.int64)
    rows = _dequant(qtts.Q4Weight(e.packed[idx], e.scales[idx], len(idx), e.n))
    h = rows @ _dequant(w.fc1) + _f64(w.fc1_bias)
    return h * torch.sigmoid(h) @ _dequant(w.fc2) + _f64(w.fc2_bias)


def _codec_rows(tokens):
    e = _host_talker().codec_embedding
    idx = np.asarray(tokens, dtype=np.int64)
    return _dequant(qtts.Q4Weight(e.packed[idx], e.scales[idx], len(idx), e.n))


def _prompt_rows(tokens, speaker, language, voice):
    """Role prefix, codec prefix under the TTS pad / BOS overlay (or the voice
    row as it is), BOS with the first text token."""
    role = _text_rows([qtts.IM_START, qtts.ASSISTANT, qtts.NEWLINE])
    pad, bos = _text_rows([qtts.TTS_PAD, qtts.TTS_BOS])
    prefix = [qtts.CODEC_THINK, qtts.CODEC_THINK_BOS, language, qtts.CODEC_THINK_EOS]
    head = _codec_rows(prefix)
    spk = _codec_rows([speaker])[0] if voice is None else None
    cpad, cbos = _codec_rows([qtts.CODEC_PAD, qtts.CODEC_BOS])
    rows = [*role, *[r + pad for r in head], _f64(voice) if voice is not None else spk + pad, cpad + bos]
    if len(tokens):
        rows.append(cbos + _text_rows(tokens[:1])[0])
    return torch.stack(rows)


def _prompt_exact(case, seed):
    i = _prompt_inputs(case, seed)
    hidden = _talker_rows(_prompt_rows(i["tokens"], i["speaker"], i["language"], i["voice"]))[-1]
    return {"hidden": hidden, "logits": hidden @ _dequant(_host_talker().codec_head)}


def _conv(x, w, b, cin, cout, k, dilation):
    w = _f64(w).reshape(cout, cin, k)
    xp = torch.nn.functional.pad(x, ((k - 1) * dilation, 0))
    out = _f64(b)[:, None].expand(cout, x.shape[1]).contiguous()
    for t in range(k):
        out += w[:, :, t].contiguous() @ xp[:, t * dilation: t * dilation + x.shape[1]]
    return out


def _causal(x, d):
    return _conv(x, d["weight"], d["bias"], d["in_channels"], d["out_channels"], d["kernel_size"], d["dilation"])


def _transposed(x, d):
    """out[i * stride + t] += x[i] w[t], cropped to len * stride."""
    cin, cout, k, s = d["in_channels"], d["out_channels"], d["kernel_size"], d["stride"]
    w, L = _f64(d["weight"]).reshape(cin, cout, k), x.shape[1]
    out = _f64(d["bias"])[:, None, None].expand(cout, L, s).contiguous()
    for t in range(k):
        y, late = w[:, :, t].T.contiguous() @ x, t // s
        out[:, late:, t % s] += y[:, : L - late]
    return out.reshape(cout, L * s)


def _snake(x, alpha, beta):
    return x + torch.exp(-_f64(beta))[:, None] * torch.sin(torch.exp(_f64(alpha))[:, None] * x) ** 2


def _decode_exact(codes):
    w = _host_decoder()
    c, T = w.cfg, codes.shape[1]
    ad = c.heads * c.head_dim
    idx = torch.from_numpy(codes.astype(np.int64)).to(_DEV)
    book = lambda a: _f64(a).reshape(c.codebook_size, c.codebook_dim)  # noqa: E731
    rest = sum(book(w.rest_codebooks[g])[idx[g + 1]] for g in range(c.num_rest))
    proj = lambda a: _f64(a).reshape(c.codebook_dim, c.vq_dim)  # noqa: E731
    x = (book(w.first_codebook)[idx[0]] @ proj(w.first_output_proj) + rest @ proj(w.rest_output_proj)).T
    x = _causal(x.contiguous(), w.pre_conv)
    x = x.T @ _f64(w.tf_input_w).reshape(c.latent, c.hidden) + _f64(w.tf_input_b)
    pos = torch.arange(T, device=_DEV)
    mask = (pos[None, :] <= pos[:, None]) & (pos[None, :] > pos[:, None] - c.window)
    for L in w.layers:
        m = lambda n, a, b: _f64(L[n]).reshape(a, b)  # noqa: E731
        xn = _rms(x, _f64(L["input_norm"]), 1e-5)
        q, k, v = ((xn @ m(n, c.hidden, ad)).reshape(T, c.heads, c.head_dim) for n in ("q_proj", "k_proj", "v_proj"))
        a = _attend(_rope(q, pos, c.rope_theta), _rope(k, pos, c.rope_theta), v, mask).reshape(T, ad)
        x = x + (a @ m("o_proj", ad, c.hidden)) * _f64(L["attn_scale"])
        xn = _rms(x, _f64(L["post_attn_norm"]), 1e-5)
        gate = xn @ m("gate_proj", c.hidden, c.inter)
        h = gate * torch.sigmoid(gate) * (xn @ m("up_proj", c.hidden, c.inter))
        x = x + (h @ m("down_proj", c.inter, c.hidden)) * _f64(L["mlp_scale"])
    x = _rms(x, _f64(w.tf_norm), 1e-5) @ _f64(w.tf_output_w).reshape(c.hidden, c.latent) + _f64(w.tf_output_b)
    x = x.T.contiguous()
    for u in w.upsample:
        x = _transposed(x, u["conv_t"])
        k = u["dw_conv"]["kernel_size"]
        dw, xp = _f64(u["dw_conv"]["weight"]).reshape(-1, k), torch.nn.functional.pad(x, (k - 1, 0))
        y = _f64(u["dw_conv"]["bias"])[:, None] + sum(dw[:, t: t + 1] * xp[:, t: t + x.shape[1]] for t in range(k))
        y = (y - y.mean(0)) / torch.sqrt(y.var(0, unbiased=False) + 1e-5)
        y = (y * _f64(u["norm_w"])[:, None] + _f64(u["norm_b"])[:, None]).T
        h = y @ _f64(u["pw1_w"]).reshape(-1, u["inner"]) + _f64(u["pw1_b"])
        h = h * 0.5 * (1.0 + torch.tanh(h / math.sqrt(2.0)))
        y = h @ _f64(u["pw2_w"]).reshape(u["inner"], -1) + _f64(u["pw2_b"])
        x = x + _f64(u["gamma"])[:, None] * y.T
    x = _causal(x, w.vocos_init)
    for b in w.blocks:
        x = _transposed(_snake(x, b["pre_snake_alpha"], b["pre_snake_beta"]), b["upsample"])
        for r in b["residuals"]:
            y = _causal(_snake(x, r["act1_alpha"], r["act1_beta"]), r["conv1"])
            x = x + _causal(_snake(y, r["act2_alpha"], r["act2_beta"]), r["conv2"])
    x = _causal(_snake(x, w.final_snake_alpha, w.final_snake_beta), w.output_conv)
    return x.reshape(-1).clamp(-1.0, 1.0)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv_host":
        return _f64(_activations(seed, 1, case["k"])[0]) @ _dequant(_host_q4(case["k"], case["n"], 0))
    if kind in ("gemv", "gemm"):
        x = _f64(_activations(seed, case.get("rows", 1), case["k"]))
        return torch.stack([x @ _dequant(_host_q4(case["k"], case["n"], i)) for i in range(case["weights"])])
    if kind == "text":
        t = _tokens(seed, case["tokens"])
        return _text_rows([*t[1:], qtts.TTS_EOS])
    if kind == "prompt":
        return {**_prompt_exact(case, seed), "position": None}
    if kind == "context":
        n = case["rows"]
        h = _talker_rows(_f64(np.concatenate([_rows(seed, 1, n), _rows(seed, 2, case["steps"])])))[n - 1:]
        out = torch.cat([h, h @ _dequant(_host_talker().codec_head)], -1)
        return {"hidden": out[0, : TALKER.hidden], "logits": out[0, TALKER.hidden:], "steps": out[1:]}
    if kind == "speech":
        return {**_prompt_exact(case, seed), "codes": None, "audio": None}
    if kind == "batch":
        n, b = case["rows"], case["streams"]
        h = _talker_rows(_f64(np.concatenate([_rows(seed, 100 + i, n) for i in range(b)])), b)[n - 1:: n]
        return {"hidden": h, "logits": h @ _dequant(_host_talker().codec_head), "codes": None}
    if kind == "decode":
        return _decode_exact(_codes(seed, case["frames"]))
    return None  # frames: every step follows a drawn token
