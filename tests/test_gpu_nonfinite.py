"""Infinities, NaN and values near FLT_MAX through the prefill kernels (MI355X).

Those kernels split FP32 operands into BF16 numbers, which no infinity and no value past the
largest BF16 (3.3895e38) survives; what they return must be what FP32 products give.  The models
here have a finite answer that passes through such a value, so they are compared with the
oracle, and each fails if one product of the path turns into NaN.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = np.float32(3.4e38)           # past the largest BF16, below FLT_MAX
TINY = np.float32(2.0 ** -124)     # BIG * TINY = 15.99
ROWS = (1, 17, 33, 64, 65, 155, 331)


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
