"""HIP codec decode (EnhancedCodec::decode, src/codec.cpp:64-72) against the float64 oracle.

Tolerance: the reference's own codec bar (src/main.cpp:19-30, 67-76): max-abs error < 1e-4 and
RMSE < 1e-5 per case.  Lengths 1, 2, 7 and 31 are those of the reference's decode fixtures
(docs/codec-validation.jsonl), plus 300.
"""
import numpy as np
import pytest

import codec_oracle as co

pytestmark = pytest.mark.gpu

MAX_ABS, RMSE = 1e-4, 1e-5


@pytest.fixture(scope="module")
def codec_weights(itts):
    return itts.make_synthetic_codec_weights(seed=5)


@pytest.fixture(scope="module")
def codec(itts, codec_weights):
    c = itts.EnhancedCodec(codec_weights)
    yield c
    c.close()


def _close(got, ref, what):
    d = np.abs(got.astype(np.float64) - ref)
    peak, rmse = float(d.max()), float(np.sqrt(np.mean(d * d)))
    assert peak < MAX_ABS and rmse < RMSE, f"{what}: max-abs {peak:.3e} rmse {rmse:.3e}"


@pytest.mark.parametrize("n", [1, 2, 7, 31, 300])
def test_codec_decode_matches_oracle(codec, codec_weights, n):
    rng = np.random.default_rng(n)
    codes = [int(x) for x in rng.integers(0, 8192, n)]
    codes[0] = 8191
    if n > 1:
        codes[-1] = 0
    print(f"codec decode: {n} codes", flush=True)
    got = codec.decode(codes)
    assert got.shape == (2 * n, 1024)
    _close(got, co.decode(codec_weights, codes), f"decode.{n}")


@pytest.mark.parametrize("n", [15, 16, 17, 33, 48, 63, 64, 65, 127, 193])
def test_codec_decode_tile_edges_match_oracle(codec, codec_weights, n):
    """Lengths either side of the 16-row operand tiles, of the 64 rows up to which the plain GEMMs
    take 16-column workgroups, and of the row blocks of the 64-column tiles (the embed and up
    convolutions read past a tile's rows).  FP32 sums: a tenth of the codec bar, which is what the
    reference's lengths measure (max-abs 8e-6)."""
    codes = [int(x) for x in np.random.default_rng(1000 + n).integers(0, 8192, n)]
    d = np.abs(codec.decode(codes).astype(np.float64) - co.decode(codec_weights, codes))
    assert float(d.max()) < MAX_ABS / 10 and float(np.sqrt(np.mean(d * d))) < RMSE / 10, (n, float(d.max()))


def test_codec_decode_5000_codes_matches_oracle_windows(codec, codec_weights):
    """The longest decode the reference accepts (codec.cpp:58: 1..5000 codes).  An output row
    depends only on the codes within 40 of its own (embed conv7: 3, twelve depthwise conv7:
    36, the up conv3 after the x2 upsampling: 1; every other op is per row), so the float64
    oracle decodes three windows of the 5000 codes (the start, the middle, the end) with 48
    codes of context at each cut, and their rows away from the cuts must equal the device's
    full decode at the codec bar."""
    rng = np.random.default_rng(5000)
    codes = [int(x) for x in rng.integers(0, 8192, 5000)]
    print("codec decode: 5000 codes", flush=True)
    got = codec.decode(codes)
    assert got.shape == (10000, 1024) and np.isfinite(got).all()
    ctx = 48
    for a, b in ((0, 200), (2400, 2600), (4800, 5000)):
        lo, hi = max(0, a - ctx), min(5000, b + ctx)
        ref = co.decode(codec_weights, codes[lo:hi])
        _close(got[2 * a: 2 * b], ref[2 * (a - lo): 2 * (b - lo)], f"decode.5000 codes {a}..{b}")


def test_codec_decode_is_deterministic(codec):
    codes = list(range(0, 8192, 97))
    a, b = codec.decode(codes), codec.decode(codes)
    assert np.array_equal(a, b)


def test_codec_errors(itts, codec, codec_weights):
    for bad in ([], [8192], [0] * 5001):
        with pytest.raises(itts.InvalidArgument, match=r"Codec expects 1\.\.5000 code IDs in \[0,8192\)"):
            codec.decode(bad)
    w = dict(codec_weights)
    w["codec.up.weight"] = w["codec.up.weight"][:, :, :2]
    with pytest.raises(itts.GptRuntimeError, match="Unsupported 2.5 codec shape: codec.up.weight"):
        itts.EnhancedCodec(w)
    w = dict(codec_weights)
    del w["codec.decoder.0.convnext.11.gamma"]
    with pytest.raises(itts.GptRuntimeError, match="Missing tensor: codec.decoder.0.convnext.11.gamma"):
        itts.EnhancedCodec(w)


def test_codec_from_bundle_equals_arrays(itts, codec, codec_weights, tmp_path):
    path = itts.write_mit2_bundle(tmp_path / "codec.mit2", codec_weights, single_file=True)
    b = itts.Bundle(path, require_model=False)
    c = itts.EnhancedCodec.from_bundle(b)
    b.close()
    codes = [5, 17, 4000, 8191, 0, 123]
    assert np.array_equal(c.decode(codes), codec.decode(codes))
    c.close()


def test_gpt_codes_into_codec(itts, small_weights, codec, codec_weights):
    """The path's consumer end to end: codes generated by the GPT decode into features."""
    dec = itts.GptDecoder(small_weights, kv_capacity=1024)
    cond, text = itts.synthetic_prefix_inputs(20, seed=6)
    r = dec.generate(dec.prepare_cond(cond, text, 0), itts.GenerationOptions(seed=2, suppress_stop=True), 24)
    dec.close()
    assert len(r.codes) == 24
    _close(codec.decode(r.codes), co.decode(codec_weights, r.codes), "gpt codes")


def test_codec_graph_replays_equal_eager(itts, codec_weights):
    """Decodes replayed from a captured graph equal eager launches (ITTS_CODEC_GRAPHS=0), bit for
    bit, over several replays with other work between them: decodes of other lengths (their own
    graphs) and host synchronisations."""
    import os

    old = os.environ.get("ITTS_CODEC_GRAPHS")
    os.environ["ITTS_CODEC_GRAPHS"] = "0"
    try:
        eager = itts.EnhancedCodec(codec_weights)
    finally:
        if old is None:
            del os.environ["ITTS_CODEC_GRAPHS"]
        else:
            os.environ["ITTS_CODEC_GRAPHS"] = old
    graph = itts.EnhancedCodec(codec_weights)
    rng = np.random.default_rng(9)
    for rep in range(4):
        codes = [int(x) for x in rng.integers(0, 8192, 23)]
        other = [int(x) for x in rng.integers(0, 8192, 5 + rep)]
        a = graph.decode(codes)
        assert np.array_equal(graph.decode(other), eager.decode(other)), rep
        assert np.array_equal(a, eager.decode(codes)), rep
    big = [int(x) for x in rng.integers(0, 8192, 200)]  # buffers grow: earlier graphs are dropped
    assert np.array_equal(graph.decode(big), eager.decode(big))
    assert np.array_equal(graph.decode(codes), eager.decode(codes))
    eager.close()
    graph.close()
