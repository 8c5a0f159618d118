"""Infinities, NaN and values near FLT_MAX through the prefill and codec kernels (MI355X).

Those kernels split FP32 operands into BF16 numbers, which no infinity and no value past the
largest BF16 (3.3895e38) survives; what they return must be what FP32 products give.  Every
model here has a finite answer that passes through such a value, so it is compared with the
oracle, and each fails if one product of the path turns into NaN.
"""
import ctypes as C

import numpy as np
import pytest

import codec_oracle as co
from conftest import rel_err, same_bits

pytestmark = pytest.mark.gpu

BIG = np.float32(3.4e38)           # past the largest BF16, below FLT_MAX
TINY = np.float32(2.0 ** -124)     # BIG * TINY = 15.99
ROWS = (1, 17, 33, 64, 65, 155, 331)  # one operand tile, the few-row kernel and the tiled ones, K split and not


def prefix_of(rows, seed=0):
    return (0.5 * np.random.default_rng([rows, seed]).standard_normal((rows, 1280))).astype(np.float32)


# ---------------------------------------------------------------------------- sequences stay apart
@pytest.mark.parametrize("rows", [(20, 20), (3, 5), (33, 7)])
def test_stacked_prefill_keeps_a_nan_sequence_apart(itts, small_weights, rows):
    """Two sequences share a 16-row attention tile; the second is NaN throughout.  The call fails
    for it (greedy, no processors: no code is a maximum), with the first one's codes already
    written: they are those it gets alone."""
    dec = itts.GptDecoder(small_weights, kv_capacity=256, max_batch=4)
    o = itts.GenerationOptions(do_sample=False, repetition_penalty=1.0, suppress_stop=True)
    good, bad = prefix_of(rows[0]), np.full((rows[1], 1280), np.nan, np.float32)
    alone = dec.generate(good, o, 6).codes
    fp = lambda a: a.ctypes.data_as(C.POINTER(C.c_float))
    up = lambda a: a.ctypes.data_as(C.POINTER(C.c_uint32))
    codes, n, stopped = np.zeros((2, 6), np.uint32), np.zeros(2, np.uint32), np.zeros(2, np.int32)
    st = itts._lib.itts_gpt_generate_batch(dec._h, 2, (C.POINTER(C.c_float) * 2)(fp(good), fp(bad)), up(np.array(rows, np.uint32)),
                                           (type(o._c()) * 2)(o._c(), o._c()), 6, up(codes), up(n), stopped.ctypes.data_as(C.POINTER(C.c_int32)))
    assert st != 0
    assert n[0] == 6 and [int(c) for c in codes[0]] == alone
    dec.close()


@pytest.mark.parametrize("rows", [(5, 6, 4), (1, 2, 3, 4), (14, 15, 17, 18), (16, 16, 16), (30, 1, 1, 40)])
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_short_sequences_sharing_attention_tiles(itts, small_weights, rows, dtype):
    """Three or four sequences in one 16-row attention tile, or tiles split at every kind of place:
    each gets the codes it gets alone."""
    dec = itts.GptDecoder(small_weights, kv_capacity=256, max_batch=4, weight_dtype=dtype)
    opts = [itts.GenerationOptions(seed=50 + b, suppress_stop=True) for b in range(len(rows))]
    prefixes = [prefix_of(r, b) for b, r in enumerate(rows)]
    together = dec.generate_batch(prefixes, opts, 8)
    for p, o, r in zip(prefixes, opts, together):
        assert dec.generate(p, o, 8).codes == r.codes
    dec.close()


# ---------------------------------------------------------------------------- GPT
def bf16_round(a):
    a = np.ascontiguousarray(a, np.float32)
    u = a.view(np.uint32)
    r = ((u.astype(np.uint64) + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
    return np.where(np.isinf(a), a, r)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows", ROWS)
def test_prefill_with_infinite_and_huge_ffn_values_matches_oracle(itts, oracle, rows, dtype):
    """mlp.c_fc reads a constant 1 at input 0 (gain 0, bias 1): a weight of -inf there gives -inf and
    the GELU 0, -3.4e38 likewise, and a bias of 3.4e38 an activation of 3.4e38 that mlp.c_proj
    brings back with weights of 2^-124."""
    w = dict(itts.make_synthetic_weights(layers=2, seed=41, ln_random=True))
    h = "gpt.gpt.h.0."
    for n in ("ln_2.weight", "ln_2.bias", "mlp.c_fc.weight", "mlp.c_fc.bias", "mlp.c_proj.weight"):
        w[h + n] = w[h + n].copy()
    w[h + "ln_2.weight"][0], w[h + "ln_2.bias"][0] = 0.0, 1.0
    w[h + "mlp.c_fc.weight"][0, [7, 70, 4999]] = -np.inf
    w[h + "mlp.c_fc.weight"][0, [100, 3001]] = -BIG
    w[h + "mlp.c_fc.weight"][:, 5000] = 0.0
    w[h + "mlp.c_fc.bias"][5000] = BIG
    w[h + "mlp.c_proj.weight"][5000] = np.where(np.arange(1280) % 3 == 0, TINY, -TINY)
    dec = itts.GptDecoder(w, kv_capacity=512, weight_dtype=dtype)
    if dtype == "bf16":
        matrices = ("attn.c_attn.weight", "attn.c_proj.weight", "mlp.c_fc.weight", "mlp.c_proj.weight", "mel_head.weight")
        w = {k: bf16_round(v) if k.endswith(matrices) else v for k, v in w.items()}
    orc = oracle.OracleGpt(w, kv_capacity=512)
    got, ref = dec.prefill(prefix_of(rows)), orc.prefill(prefix_of(rows))
    assert np.isfinite(ref).all()
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), np.max(np.abs(got - ref))
    dec.close()


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("rows", ROWS)
def test_prefill_after_a_nan_prefill_gives_the_same_bits(itts, small_weights, rows, dtype):
    """A longer prefix of NaN leaves NaN in the operands' padding rows: the next prefill's tiles then
    take the repairing epilogue, and its results are still those of a fresh decoder."""
    fresh = itts.GptDecoder(small_weights, kv_capacity=512, weight_dtype=dtype)
    used = itts.GptDecoder(small_weights, kv_capacity=512, weight_dtype=dtype)
    used.prefill(np.full((rows + 20, 1280), np.nan, np.float32))
    assert same_bits(used.prefill(prefix_of(rows)), fresh.prefill(prefix_of(rows)))
    fresh.close()
    used.close()


@pytest.mark.parametrize("rows", ROWS)
def test_prefill_with_huge_keys_matches_oracle(itts, oracle, rows):
    """One dimension of a head has key 3.4e38 and query 2^-124 in every row: every score of it gains
    the same 2, which the softmax takes out again."""
    w = dict(itts.make_synthetic_weights(layers=2, seed=42, ln_random=True))
    n = "gpt.gpt.h.0.attn.c_attn."
    w[n + "weight"], w[n + "bias"] = w[n + "weight"].copy(), w[n + "bias"].copy()
    for col, value in ((3 * 64 + 5, TINY), (1280 + 3 * 64 + 5, BIG)):
        w[n + "weight"][:, col] = 0.0
        w[n + "bias"][col] = value
    dec, orc = itts.GptDecoder(w, kv_capacity=512), oracle.OracleGpt(w, kv_capacity=512)
    got, ref = dec.prefill(prefix_of(rows)), orc.prefill(prefix_of(rows))
    assert np.isfinite(ref).all()
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), np.max(np.abs(got - ref))
    dec.close()


@pytest.mark.parametrize("rows", [2, 16, 17, 40, 155])
def test_prefill_past_a_row_with_an_infinite_key_matches_oracle(itts, oracle, rows):
    """Row 0's key overflows to +inf in a dimension where every query is negative: later rows score
    it -inf and give it no weight.  (Row 0 itself has no finite score; one layer, so its NaN
    reaches no other row.)"""
    w = dict(itts.make_synthetic_weights(layers=1, seed=43))
    n = "gpt.gpt.h.0.attn.c_attn."
    w[n + "weight"], w[n + "bias"] = w[n + "weight"].copy(), w[n + "bias"].copy()
    q, k, j = 5 * 64 + 9, 1280 + 5 * 64 + 9, 200
    w[n + "weight"][:, [q, k]] = 0.0
    w[n + "bias"][q], w[n + "bias"][k] = -TINY, 0.0
    w[n + "weight"][j, k] = 1e38   # LayerNorm of row 0 is 35 there, of the others about 0
    x = prefix_of(rows)
    x[0, j] = 1000.0
    x[1:, j] = x[1:].mean(-1)
    dec, orc = itts.GptDecoder(w, kv_capacity=512), oracle.OracleGpt(w, kv_capacity=512)
    got, ref = dec.prefill(x), orc.prefill(x)
    assert np.isfinite(ref).all()
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), np.max(np.abs(got - ref))
    dec.close()


# ---------------------------------------------------------------------------- codec
@pytest.mark.parametrize("n", [1, 17, 47, 64, 65, 200])
def test_codec_with_huge_weights_and_activations_matches_oracle(itts, n):
    """Constant 2^-124 inputs against weights of 3.4e38 (the embed convolution, pwconv1) and
    constant 3.4e38 inputs against weights of 2^-124 (pwconv2, the up convolution): 16 each."""
    w = {k: v.copy() for k, v in itts.make_synthetic_codec_weights(seed=6).items()}
    q, d = "codec.quantizer.quantizers.0", "codec.decoder.0"
    sign = lambda m: np.where(np.arange(m) % 3 == 0, np.float32(1), np.float32(-1))
    w[q + ".out_project.weight"][11], w[q + ".out_project.bias"][11] = 0.0, TINY
    w[d + ".embed.weight"][:, 11] = BIG * sign(384)[:, None]
    b = d + ".convnext.0."
    w[b + "norm.weight"][3], w[b + "norm.bias"][3] = 0.0, TINY
    w[b + "pwconv1.weight"][:, 3] = BIG * sign(2048)
    w[b + "pwconv1.weight"][900], w[b + "pwconv1.bias"][900] = 0.0, BIG
    w[b + "pwconv2.weight"][:, 900] = TINY * sign(384)
    w["codec.decoder.1.weight"][77], w["codec.decoder.1.bias"][77] = 0.0, BIG
    w["codec.up.weight"][:, 77] = TINY * sign(1024)[:, None]
    c = itts.EnhancedCodec(w)
    codes = [int(x) for x in np.random.default_rng(n).integers(0, 8192, n)]
    got, ref = c.decode(codes), co.decode(w, codes)
    assert np.isfinite(ref).all() and np.isfinite(got).all()
    assert rel_err(got, ref) < 1e-5 and np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), rel_err(got, ref)
    c.close()


# ---------------------------------------------------------------------------- Qwen
@pytest.mark.parametrize("n", [1, 20, 64, 65, 200])
def test_qwen_prefill_zero_times_huge_weights_matches_oracle(itts, oracle, n):
    """Residual column 0 is zero in every row (embedding column 0 and o_proj row 0 of layer 0 are
    zero), and q/k/v and gate/up weights of 3.4e38 multiply it: they add exactly nothing."""
    w = {k: v.copy() if "layers.0." in k or "embed" in k else v for k, v in itts.make_synthetic_qwen_weights(layers=1, seed=8).items()}
    p = "qwen.model.layers.0."
    w["qwen.model.embed_tokens.weight"][:, 0] = 0.0
    w[p + "self_attn.o_proj.weight"][0] = 0.0
    for m, r in (("self_attn.q_proj", 5), ("self_attn.k_proj", 1000), ("self_attn.v_proj", 63), ("mlp.gate_proj", 3000), ("mlp.up_proj", 12)):
        w[p + m + ".weight"][r, 0] = BIG
    dec, orc = itts.QwenDecoder(w, layers=1), oracle.OracleQwen(w, layers=1)
    ids = [int(x) for x in np.random.default_rng(n).integers(0, 151936, n)]
    got, ref = dec.prefill(ids), orc.prefill(ids)
    assert np.isfinite(ref).all()
    assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), np.max(np.abs(got - ref))
    dec.close()
