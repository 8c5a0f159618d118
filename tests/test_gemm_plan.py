"""How the prefill GEMMs are cut: every cut covers its product exactly (on the CPU), and every kernel
that the cuts of a 1..1024-row prefill reach gives the oracle's logits (MI355X).

The four GEMMs of a layer take a plan each: sixteen columns over the whole K range for few rows
(gemm_small_plan), else one of five tile shapes with K in up to sixteen ranges (gemm_plan).
"""
import ctypes as C

import numpy as np
import pytest

SHAPES = {"c_attn": (3840, 1280), "attn.c_proj": (1280, 1280), "c_fc": (5120, 1280), "mlp.c_proj": (1280, 5120)}
QWEN_SHAPES = {"qkv": (4096, 1024), "o": (1024, 2048), "gate_up": (6144, 1024), "down": (1024, 3072)}
ROW_TILES = (1, 2, 4, 8, 12)
MAX_SPLITS, WORKSPACE = 16, 8 << 20


class Plan(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("tile", "mblocks", "splits", "kchunk")]


class SmallPlan(C.Structure):
    _fields_ = [(n, C.c_int) for n in ("splits", "kchunk")]


@pytest.fixture(scope="module")
def plans(itts):
    tiled = itts._lib._ZN4itts9gemm_planEiiiibb
    tiled.restype, tiled.argtypes = Plan, [C.c_int] * 4 + [C.c_bool] * 2
    small = itts._lib._ZN4itts15gemm_small_planEiiiib
    small.restype, small.argtypes = SmallPlan, [C.c_int] * 4 + [C.c_bool]

    def of(m, n, k, bf16):
        splits = max(1, min(MAX_SPLITS, WORKSPACE // (m * n)))
        return small(m, n, k, splits, bf16), tiled(m, n, k, splits, bf16, True), splits

    return of


@pytest.mark.parametrize("bf16", [False, True])
def test_every_cut_covers_its_product(plans, bf16):
    for name, (n, k) in {**SHAPES, **({} if bf16 else QWEN_SHAPES)}.items():
        for m in list(range(1, 1025)) + [1200, 2047, 4095, 8192, 10240]:
            small, p, limit = plans(m, n, k, bf16)
            assert 0 <= p.tile < len(ROW_TILES) and 1 <= p.splits <= limit, (name, m)
            assert (p.mblocks - 1) * ROW_TILES[p.tile] * 16 < m <= p.mblocks * ROW_TILES[p.tile] * 16, (name, m)
            assert p.kchunk % 128 == 0 and (p.splits - 1) * p.kchunk < k <= p.splits * p.kchunk, (name, m)
            if small.splits:
                assert m <= (32 if bf16 else 64) and small.splits <= limit, (name, m)
                assert small.kchunk % 256 == 0 and (small.splits - 1) * small.kchunk < k <= small.splits * small.kchunk, (name, m)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_every_cut_of_a_prefill_matches_oracle(itts, oracle, plans, dtype):
    """Row counts that between them reach every (GEMM, kernel, split count) of 1..1024 rows: last-row
    logits within 2e-5 of the oracle's largest, as FP32 sums of up to 5120 products give.  Two
    layers: the second one's keys and values carry every row of the first to the last row."""
    reach = {}
    for m in range(1, 1025):
        for name, (n, k) in SHAPES.items():
            small, p, _ = plans(m, n, k, dtype == "bf16")
            one_tile = name == "c_fc" and small.splits == 1 and m > 16  # its GELU kernel has one row tile
            reach.setdefault((name, "small", -(-m // 16), small.splits) if small.splits and not one_tile else (name, p.tile, p.splits), set()).add(m)
    left, rows = set(reach), []
    while left:
        best = max(range(1, 1025), key=lambda m: sum(m in reach[c] for c in left))
        rows.append(best)
        left = {c for c in left if best not in reach[c]}
    w = itts.make_synthetic_weights(layers=2, seed=61, ln_random=True)
    dec = itts.GptDecoder(w, kv_capacity=1100, weight_dtype=dtype)
    if dtype == "bf16":
        def bf16_round(a):
            u = np.ascontiguousarray(a, np.float32).view(np.uint32)
            return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)

        matrices = ("attn.c_attn.weight", "attn.c_proj.weight", "mlp.c_fc.weight", "mlp.c_proj.weight", "mel_head.weight")
        w = {k: bf16_round(v) if k.endswith(matrices) else v for k, v in w.items()}
    orc = oracle.OracleGpt(w, kv_capacity=1100)
    assert len(rows) >= 10
    for m in sorted(rows):
        prefix = (0.5 * np.random.default_rng(m).standard_normal((m, 1280))).astype(np.float32)
        got, ref = dec.prefill(prefix), orc.prefill(prefix)
        assert np.max(np.abs(got - ref)) <= 2e-5 * np.max(np.abs(ref)), (m, np.max(np.abs(got - ref)), np.max(np.abs(ref)))
        print(f"{dtype} {m} rows", flush=True)
    dec.close()
