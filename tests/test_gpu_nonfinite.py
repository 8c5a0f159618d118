"""Infinities, NaN and values near FLT_MAX through the prefill kernels (MI355X)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
