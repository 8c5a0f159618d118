"""Workloads of the IndexTTS 2.5 decoders as a speech service runs them, for timing and comparison.

Kinds (sizes in brackets are the ranges that `draw` covers):

  prefill   the prefix of one text segment through the 24-layer GPT: [8..600] rows, FP32 or BF16 weights
  score     a prefix and [4..32] given codes, one step each (alignment, likelihoods): [8..300] rows
  resume    a kept checkpoint of [150..1000] rows, restored and continued for [4..24] given codes:
            the steps of a long utterance
  utterance generate() with the default sampling: [16..300] rows, [8..40] codes, then the next logits
  segments  generate_segments() over a request's [2..8] text segments of ragged lengths [8..160],
            [8..32] codes each, then the first segment's next logits
  beam      generate() with [2..4] beams, [16..200] rows, [8..32] codes, beside the prefix's logits
  codec     EnhancedCodec.decode() of [1..1300] codes
  qwen      the emotion-text decoder: a prompt of [8..400] ids, [1..24] greedy ids, then the next logits

A program loads its model once and serves many requests with it, so the decoders are made once per
process; what differs between requests (speaker, emotion, text, codes, seeds) comes from `seed`.
Weights are random-init of the real shapes.
"""
import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "index-tts-25-metal_amd"))
import itts_gpt as it  # noqa: E402

LAYERS, WIDTH, HEADS, FFN, VOCAB = 24, 1280, 20, 5120, 8194
MAX_BATCH = 8


def listed():
    return [
        # one short word: latency of the whole prefix forward
        {"name": "prefill_short", "kind": "prefill", "rows": 20, "dtype": "f32"},
        # an ordinary sentence (the benchmark's prefix length)
        {"name": "prefill_usual", "kind": "prefill", "rows": 155, "dtype": "f32"},
        # a paragraph near the text position table's end
        {"name": "prefill_long", "kind": "prefill", "rows": 571, "dtype": "f32"},
        # two sentences on a decoder with BF16 weights
        {"name": "prefill_bf16", "kind": "prefill", "rows": 331, "dtype": "bf16"},
        # batch-1 sampled decode, the service's default request
        {"name": "utterance", "kind": "utterance", "rows": 91, "codes": 40, "dtype": "f32"},
        # teacher-forced scoring on BF16 weights
        {"name": "score_bf16", "kind": "score", "rows": 63, "codes": 24, "dtype": "bf16"},
        # the tail of a long utterance: steps over a large cache
        {"name": "resume_long", "kind": "resume", "rows": 923, "codes": 16, "dtype": "f32"},
        # one request's eight text segments decoded together
        {"name": "segments_8", "kind": "segments", "segments": 8, "longest": 120, "codes": 24, "dtype": "f32"},
        # beam search, the quality setting
        {"name": "beam_3", "kind": "beam", "rows": 79, "beams": 3, "codes": 24, "dtype": "f32"},
        # the codes of a short and of a long utterance to features
        {"name": "codec_short", "kind": "codec", "codes": 47},
        {"name": "codec_long", "kind": "codec", "codes": 1201},
        # the emotion description: chat prompt and a short greedy answer
        {"name": "qwen_emotion", "kind": "qwen", "prompt": 77, "codes": 20},
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["prefill", "prefill", "score", "resume", "utterance", "segments", "beam", "codec", "codec", "qwen"])
    dtype = rng.choice(["f32", "f32", "bf16"])
    if kind == "prefill":
        return {"kind": kind, "rows": log_int(8, 600), "dtype": dtype}
    if kind == "score":
        return {"kind": kind, "rows": log_int(8, 300), "codes": rng.randint(4, 32), "dtype": dtype}
    if kind == "resume":
        return {"kind": kind, "rows": rng.randint(150, 1000), "codes": rng.randint(4, 24), "dtype": dtype}
    if kind == "utterance":
        return {"kind": kind, "rows": log_int(16, 300), "codes": rng.randint(8, 40), "dtype": dtype}
    if kind == "segments":
        return {"kind": kind, "segments": rng.randint(2, 8), "longest": rng.randint(16, 160), "codes": rng.randint(8, 32), "dtype": dtype}
    if kind == "beam":
        return {"kind": kind, "rows": log_int(16, 200), "beams": rng.randint(2, 4), "codes": rng.randint(8, 32), "dtype": dtype}
    if kind == "codec":
        return {"kind": kind, "codes": log_int(1, 1300)}
    return {"kind": kind, "prompt": log_int(8, 400), "codes": rng.randint(1, 24)}


# ------------------------------------------------------------------ models, made once per process
@functools.lru_cache(maxsize=None)
def gpt_weights():
    return it.make_synthetic_weights(layers=LAYERS, seed=11, ln_random=True)


@functools.lru_cache(maxsize=None)
def gpt(dtype):
    return it.GptDecoder(gpt_weights(), max_batch=MAX_BATCH, weight_dtype=dtype)


@functools.lru_cache(maxsize=None)
def codec_weights():
    return it.make_synthetic_codec_weights(seed=12)


@functools.lru_cache(maxsize=None)
def codec():
    return it.EnhancedCodec(codec_weights())


@functools.lru_cache(maxsize=None)
def qwen_weights():
    return it.make_synthetic_qwen_weights(seed=13)


@functools.lru_cache(maxsize=None)
def qwen():
    return it.QwenDecoder(qwen_weights())


# ------------------------------------------------------------------ inputs
def inputs(case, seed):
    """What the request brings: everything here comes from the seed."""
    r = np.random.default_rng([seed, 77])
    kind, x = case["kind"], {}
    if kind == "codec":
        return {"codes": r.integers(0, 8192, case["codes"])}
    if kind == "qwen":
        return {"prompt": r.integers(0, 151643, case["prompt"]).astype(np.uint32)}
    x["speaker"] = r.standard_normal(192).astype(np.float32)
    x["emotion"] = (0.5 * r.standard_normal(WIDTH)).astype(np.float32)
    x["language"] = int(r.integers(0, 107))
    x["seed"] = int(r.integers(0, 1 << 62))
    if kind == "segments":
        x["ids"] = [r.integers(2, 12000, int(r.integers(8, case["longest"] + 1))).astype(np.uint32) for _ in range(case["segments"])]
    elif kind == "resume":  # as deep a cache as a prefix and the codes after it give
        x["prefix"] = (0.5 * r.standard_normal((case["rows"], WIDTH))).astype(np.float32)
    else:  # conditioning 3 rows, text begin and end, mel start
        x["ids"] = r.integers(2, 12000, case["rows"] - 6).astype(np.uint32)
    x["codes"] = r.integers(0, 8192, case["codes"]) if kind in ("score", "resume") else None
    return x


def options(case, x):
    return it.GenerationOptions(seed=x["seed"], num_beams=case.get("beams", 1), suppress_stop=True)


def prepare(case, seed):
    x, kind = inputs(case, seed), case["kind"]
    s = {"case": case, "x": x}
    if kind == "codec":
        s["model"] = codec()
    elif kind == "qwen":
        s["model"] = qwen()
    else:
        s["model"] = gpt(case["dtype"])
        if kind == "resume":
            s["model"].prefill(x["prefix"])
            s["kept"] = s["model"].checkpoint()
        elif kind != "segments":
            s["prefix"] = s["model"].prepare(x["speaker"], x["emotion"], x["ids"], x["language"])
            assert s["prefix"].size == case["rows"] * WIDTH
        if "codes" in case and kind not in ("score", "resume"):
            s["options"] = options(case, x)
    return s


def run(s):
    m, x, case, kind = s["model"], s["x"], s["case"], s["case"]["kind"]
    if kind == "prefill":
        return m.prefill(s["prefix"])
    if kind in ("score", "resume"):
        if kind == "score":
            out = [m.prefill(s["prefix"])]
        else:
            m.restore(s["kept"])
            out = []
        return np.stack(out + [m.step(int(c), i + 2) for i, c in enumerate(x["codes"])])
    if kind == "utterance":
        r = m.generate(s["prefix"], s["options"], case["codes"])
        return {"codes": np.array(r.codes), "logits": m.step(r.codes[-1], len(r.codes) + 1)}
    if kind == "segments":
        rs = m.generate_segments(x["speaker"], x["emotion"], x["ids"], x["language"], s["options"], case["codes"])
        return {"codes": np.array([r.codes for r in rs]), "logits": m.step(rs[0].codes[-1], len(rs[0].codes) + 1)}
    if kind == "beam":
        r = m.generate(s["prefix"], s["options"], case["codes"])
        return {"codes": np.array(r.codes), "logits": m.prefill(s["prefix"])}
    if kind == "codec":
        return m.decode(x["codes"])
    ids, _ = m.generate_tokens(x["prompt"], case["codes"])
    return {"codes": np.array(ids), "logits": m.step(ids[-1])}


# ------------------------------------------------------------------ work
GPT_LAYER = 3 * WIDTH * WIDTH + WIDTH * WIDTH + 2 * WIDTH * FFN
GPT_SMALL = 4 * (LAYERS * 16640 + 4 * WIDTH + VOCAB)
GPT_KV_ROW = LAYERS * 2 * WIDTH * 4
QWEN_LAYER, QWEN_HEAD, QWEN_KV_ROW = 15_728_640, 151_936 * 1024, 28 * 2 * 1024 * 4


def gpt_pass(case, nseq, rows, cached, logits):
    """One forward of `nseq` sequences, `rows` new rows in all after `cached` rows in all, and its `logits` rows."""
    wb = 4 if case["dtype"] == "f32" else 2
    keys = cached * rows / max(1, nseq) + rows * rows / max(1, nseq) / 2
    return {"bytes": wb * (LAYERS * GPT_LAYER + VOCAB * WIDTH) + GPT_SMALL + GPT_KV_ROW * (cached + rows) + 4 * (rows * WIDTH + logits * VOCAB),
            "flops": 2.0 * rows * LAYERS * GPT_LAYER + LAYERS * 4.0 * WIDTH * keys + 2.0 * logits * VOCAB * WIDTH}


def qwen_pass(rows, cached):
    return {"bytes": 4 * (28 * QWEN_LAYER + QWEN_HEAD + 28 * 2304 + 1024) + QWEN_KV_ROW * (cached + rows) + 4 * 151_936,
            "flops": 2.0 * rows * 28 * QWEN_LAYER + 28 * 4.0 * 2048 * rows * (cached + rows / 2) + 2.0 * QWEN_HEAD}


def work(case):
    kind = case["kind"]
    if kind == "codec":
        t = case["codes"]
        per_row = 7 * 1024 * 384 + 12 * (2 * 384 * 2048 + 7 * 384) + 384 * 1024 + 2 * 3 * 1024 * 1024 + 8 * 1024
        weights = 8 * 8192 + 8 * 1024 + 7 * 1024 * 384 + 12 * 2 * 384 * 2048 + 384 * 1024 + 3 * 1024 * 1024
        return {"bytes": 4 * (weights + 2 * t * 1024 + t), "flops": 2.0 * t * per_row}
    if kind == "qwen":
        passes = [qwen_pass(case["prompt"], 0)] + [qwen_pass(1, case["prompt"] + i) for i in range(case["codes"])]
    elif kind == "segments":
        n, rows = case["segments"], case["segments"] * ((8 + case["longest"]) / 2 + 6)
        passes = [gpt_pass(case, n, rows, 0, n)] + [gpt_pass(case, n, n, rows + i * n, n) for i in range(case["codes"] - 1)]
        passes.append(gpt_pass(case, 1, 1, rows / n + case["codes"], 1))
    else:
        rows, codes, n = case["rows"], case.get("codes", 0), case.get("beams", 1)
        passes = [] if kind == "resume" else [gpt_pass(case, 1, rows, 0, 1)]
        if kind == "beam":
            passes += [gpt_pass(case, n, n, n * (rows + i), n) for i in range(codes - 1)] + [gpt_pass(case, 1, rows, 0, 1)]
        else:
            passes += [gpt_pass(case, 1, 1, rows + i, 1) for i in range(codes)]
        if kind == "resume":
            passes.append({"bytes": 2 * GPT_KV_ROW * rows, "flops": 0})
    return {k: sum(p[k] for p in passes) for k in ("bytes", "flops")}


def tolerance(case):
    # FP32 sums throughout (BF16 is a storage type of the weights): against 64 bits the kinds with
    # `exact` measured 5e-7 .. 1.5e-6; another order of the sums shows up to about twice that apart.
    return {"rel": 1e-5, "max": 1e-4}


# ------------------------------------------------------------------ the same in 64 bits
def d64(a):
    return torch.as_tensor(np.ascontiguousarray(a)).cuda().double()


def norm64(x, w, b=None, eps=1e-5):
    if b is None:
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w + b


def causal64(q, k, v, scale):
    """q [H][T][d], k and v [H][T][d]; a head at a time."""
    t = q.shape[1]
    mask = torch.full((t, t), -math.inf, dtype=torch.float64, device=q.device).triu(1)
    return torch.stack([torch.softmax(q[h] @ k[h].T * scale + mask, -1) @ v[h] for h in range(q.shape[0])])


def gpt64(case, x, first):
    """Logits of rows first, first + 1, ... of the prefix followed by the given codes."""
    w = gpt_weights()

    def matrix(name):
        m = d64(w[name])
        return m.float().bfloat16().double() if case["dtype"] == "bf16" else m

    if "prefix" in x:
        h = d64(x["prefix"])
    else:
        ids = np.concatenate([[0], x["ids"], [1]]).astype(np.int64)
        text = d64(w["gpt.text_embedding.weight"][ids]) + d64(w["gpt.text_pos_embedding.emb.weight"][: len(ids)])
        text = text + d64(w["gpt.lang_embedding.weight"][x["language"]])
        spk = d64(w["gpt.spk_emb_proj.weight"]) @ d64(x["speaker"]) + d64(w["gpt.spk_emb_proj.bias"]) + d64(x["emotion"])
        start = d64(w["gpt.mel_embedding.weight"][8192]) + d64(w["gpt.mel_pos_embedding.emb.weight"][0])
        h = torch.cat([spk[None], torch.zeros_like(spk).expand(2, -1), text, start[None]])
    if x["codes"] is not None:
        codes = np.asarray(x["codes"])
        h = torch.cat([h, d64(w["gpt.mel_embedding.weight"][codes]) + d64(w["gpt.mel_pos_embedding.emb.weight"][2:2 + len(codes)])])
    t = h.shape[0]
    for i in range(LAYERS):
        p = f"gpt.gpt.h.{i}."
        ln = [d64(w[p + n]) for n in ("ln_1.weight", "ln_1.bias", "ln_2.weight", "ln_2.bias")]
        y = norm64(h, ln[0], ln[1]) @ matrix(p + "attn.c_attn.weight") + d64(w[p + "attn.c_attn.bias"])
        q, k, v = (z.reshape(t, HEADS, 64).transpose(0, 1) for z in y.split(WIDTH, 1))
        y = causal64(q, k, v, 0.125).transpose(0, 1).reshape(t, WIDTH)
        h = h + y @ matrix(p + "attn.c_proj.weight") + d64(w[p + "attn.c_proj.bias"])
        y = norm64(h, ln[2], ln[3]) @ matrix(p + "mlp.c_fc.weight") + d64(w[p + "mlp.c_fc.bias"])
        y = 0.5 * y * (1 + torch.tanh(0.7978845608028654 * (y + 0.044715 * y ** 3)))
        h = h + y @ matrix(p + "mlp.c_proj.weight") + d64(w[p + "mlp.c_proj.bias"])
    h = norm64(h[first:], d64(w["gpt.gpt.ln_f.weight"]), d64(w["gpt.gpt.ln_f.bias"]))
    h = norm64(h, d64(w["gpt.final_norm.weight"]), d64(w["gpt.final_norm.bias"]))
    return h @ matrix("gpt.mel_head.weight").T + d64(w["gpt.mel_head.bias"])


def qwen64(ids):
    """Logits of the last id."""
    w = qwen_weights()
    t = len(ids)
    h = d64(w["qwen.model.embed_tokens.weight"][np.asarray(ids, dtype=np.int64)])
    angle = torch.arange(t, dtype=torch.float64, device=h.device)[:, None] * (1e6 ** (-torch.arange(64, dtype=torch.float64, device=h.device) / 64))
    cos, sin = torch.cat([angle.cos()] * 2, -1), torch.cat([angle.sin()] * 2, -1)

    def heads(z, n, norm):
        z = norm64(z.reshape(t, n, 128), norm, eps=1e-6).transpose(0, 1)
        return z * cos + torch.cat([-z[..., 64:], z[..., :64]], -1) * sin

    for i in range(28):
        m = {n: d64(w[f"qwen.model.layers.{i}.{n}.weight"]) for n in (
            "self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "self_attn.q_norm", "self_attn.k_norm",
            "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj", "input_layernorm", "post_attention_layernorm")}
        y = norm64(h, m["input_layernorm"], eps=1e-6)
        q = heads(y @ m["self_attn.q_proj"].T, 16, m["self_attn.q_norm"])
        k = heads(y @ m["self_attn.k_proj"].T, 8, m["self_attn.k_norm"]).repeat_interleave(2, 0)
        v = (y @ m["self_attn.v_proj"].T).reshape(t, 8, 128).transpose(0, 1).repeat_interleave(2, 0)
        h = h + causal64(q, k, v, 128 ** -0.5).transpose(0, 1).reshape(t, 2048) @ m["self_attn.o_proj"].T
        y = norm64(h, m["post_attention_layernorm"], eps=1e-6)
        h = h + (torch.nn.functional.silu(y @ m["mlp.gate_proj"].T) * (y @ m["mlp.up_proj"].T)) @ m["mlp.down_proj"].T
    return d64(w["qwen.model.embed_tokens.weight"]) @ norm64(h[-1], d64(w["qwen.model.norm.weight"]), eps=1e-6)


def conv64(x, w, b):
    """Same-length convolution of x [T][Cin] with w [Cout][Cin][k], a tap at a time."""
    k, t = w.shape[2], x.shape[0]
    x = torch.nn.functional.pad(x, (0, 0, k // 2, k // 2))
    return sum(x[j:j + t] @ w[:, :, j].T for j in range(k)) + b


def codec64(codes):
    w = {n: d64(v) for n, v in codec_weights().items()}
    q, p = "codec.quantizer.quantizers.0", "codec.decoder.0"
    x = w[q + ".codebook.weight"][torch.as_tensor(codes).cuda()] @ w[q + ".out_project.weight"].T + w[q + ".out_project.bias"]
    x = norm64(conv64(x, w[p + ".embed.weight"], w[p + ".embed.bias"]), w[p + ".norm.weight"], w[p + ".norm.bias"], 1e-6)
    for i in range(12):
        b = f"{p}.convnext.{i}."
        t = x.shape[0]
        y = torch.nn.functional.pad(x, (0, 0, 3, 3))
        y = sum(y[j:j + t] * w[b + "dwconv.weight"][:, 0, j] for j in range(7)) + w[b + "dwconv.bias"]
        y = norm64(y, w[b + "norm.weight"], w[b + "norm.bias"], 1e-6) @ w[b + "pwconv1.weight"].T + w[b + "pwconv1.bias"]
        y = 0.5 * y * (1 + torch.erf(y / math.sqrt(2)))
        x = x + (y @ w[b + "pwconv2.weight"].T + w[b + "pwconv2.bias"]) * w[b + "gamma"]
    x = norm64(x, w[p + ".final_layer_norm.weight"], w[p + ".final_layer_norm.bias"], 1e-6)
    x = (x @ w["codec.decoder.1.weight"].T + w["codec.decoder.1.bias"]).repeat_interleave(2, 0)
    return conv64(x, w["codec.up.weight"], w["codec.up.bias"])


def exact(case, seed):
    x, kind = inputs(case, seed), case["kind"]
    with torch.no_grad():
        if kind == "prefill":
            return gpt64(case, x, case["rows"] - 1)[0]
        if kind == "score":
            return gpt64(case, x, case["rows"] - 1)
        if kind == "resume":
            return gpt64(case, x, case["rows"])
        if kind == "beam":
            return {"codes": None, "logits": gpt64(case, x, case["rows"] - 1)[0]}
        if kind == "codec":
            return codec64(x["codes"])
        if kind == "qwen":  # greedy, over the whole sequence each time
            ids = [int(i) for i in x["prompt"]]
            for _ in range(case["codes"]):
                ids.append(int(qwen64(ids).argmax()))
            return {"codes": None, "logits": qwen64(ids)}
    return None  # the logits after sampled codes belong to those codes alone
