"""Decode calls beside other work of the process (MI355X): they wait for nothing but their own
stream, and fail for nothing that other threads do."""
import ctypes as C
import os
import threading
import time

import numpy as np
import pytest

from conftest import same_bits

pytestmark = pytest.mark.gpu

CODES = (17, 4000, 8191, 0, 300, 5)


@pytest.fixture
def env():
    """Sets environment variables for decoders made in the test."""
    old = {}

    def put(name, value):
        old.setdefault(name, os.environ.get(name))
        os.environ[name] = value

    yield put
    for n, v in old.items():
        if v is None:
            os.environ.pop(n, None)
        else:
            os.environ[n] = v


def prefix_of(rows):
    return (0.5 * np.random.default_rng(rows).standard_normal((rows, 1280))).astype(np.float32)


def steps(dec, prefix, codes=CODES):
    return [dec.prefill(prefix)] + [dec.step(c, i + 2) for i, c in enumerate(codes)]


@pytest.fixture
def held_stream():
    """hold(null) makes a stream (or the null stream) of this process busy for 0.4 s with a host
    function that does nothing but wait, and returns an event object set when it ends."""
    hip = C.CDLL("libamdhip64.so.7", mode=C.RTLD_GLOBAL)
    fn_t = C.CFUNCTYPE(None, C.c_void_p)
    keep, streams = [], []

    def hold(null):
        s = C.c_void_p()
        if not null:
            assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
            streams.append(s)
        done = threading.Event()

        def wait(_):
            time.sleep(0.4)
            done.set()

        keep.append(fn_t(wait))
        assert hip.hipLaunchHostFunc(s, keep[-1], None) == 0
        return done

    yield hold
    assert hip.hipDeviceSynchronize() == 0
    for s in streams:
        assert hip.hipStreamDestroy(s) == 0


@pytest.fixture
def capture():
    """While entered, another thread captures a graph on a stream of its own."""
    hip = C.CDLL("libamdhip64.so.7", mode=C.RTLD_GLOBAL)

    class Capture:
        def __enter__(self):
            self.go, self.stop, self.rc = threading.Event(), threading.Event(), []
            self.thread = threading.Thread(target=self.run)
            self.thread.start()
            assert self.go.wait(20)

        def run(self):
            s, g = C.c_void_p(), C.c_void_p()
            self.rc.append(hip.hipStreamCreate(C.byref(s)))
            self.rc.append(hip.hipStreamBeginCapture(s, 1))  # thread-local mode
            self.go.set()
            self.stop.wait(60)
            self.rc.append(hip.hipStreamEndCapture(s, C.byref(g)))
            self.rc.append(hip.hipGraphDestroy(g))
            self.rc.append(hip.hipStreamDestroy(s))

        def __exit__(self, *exc):
            self.stop.set()
            self.thread.join(20)
            assert exc[0] or self.rc == [0] * 5, self.rc

    return Capture()


def steps_beside_a_busy_stream(itts, weights, hold, null):
    """A BF16 decoder's prefill and steps while a stream (or the null stream) is held: what they give
    alone, and before the stream is free again.  Streams share a few hardware queues: a decoder
    whose prefill, which has always waited for its own stream only, comes out behind the held
    stream shares that one's queue and is put aside."""
    decs = []
    try:
        for _ in range(8):
            dec = itts.GptDecoder(weights, kv_capacity=256, weight_dtype="bf16")
            decs.append(dec)
            ref = steps(dec, prefix_of(20))
            done = hold(null)
            got = [dec.prefill(prefix_of(20))]
            if done.is_set():
                continue
            got += [dec.step(c, i + 2) for i, c in enumerate(CODES)]
            assert not done.is_set(), "step() waited for a stream that is not its own"
            assert done.wait(10)
            assert dec.last_timing()["decode_path"] == "step"
            assert all(same_bits(a, b) for a, b in zip(got, ref))
            return
        pytest.skip("every decoder shares the held stream's hardware queue")
    finally:
        for d in decs:
            d.close()


def test_bf16_step_does_not_wait_for_the_null_stream(itts, small_weights, held_stream):
    steps_beside_a_busy_stream(itts, small_weights, held_stream, True)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_decode_calls_while_another_thread_captures(itts, small_weights, capture, dtype):
    """step(), generate() and generate_batch() give what they give alone."""
    dec = itts.GptDecoder(small_weights, kv_capacity=256, max_batch=2, weight_dtype=dtype)
    o = itts.GenerationOptions(seed=3, suppress_stop=True)
    calls = (lambda: steps(dec, prefix_of(20)), lambda: dec.generate(prefix_of(21), o, 20).codes,
             lambda: [r.codes for r in dec.generate_batch([prefix_of(22), prefix_of(9)], [o, o], 20)])
    ref = [f() for f in calls]
    with capture:
        got = [f() for f in calls]
    assert all(same_bits(a, b) for a, b in zip(got[0], ref[0])) and got[1:] == ref[1:]
    dec.close()


@pytest.mark.parametrize("null", [False, True])
def test_bf16_step_does_not_wait_for_other_streams(itts, small_weights, held_stream, null):
    """With an FP32 decoder of the process idle on the device."""
    f32 = itts.GptDecoder(small_weights, kv_capacity=256)
    f32.generate(prefix_of(20), itts.GenerationOptions(seed=1, suppress_stop=True), 4)
    steps_beside_a_busy_stream(itts, small_weights, held_stream, null)
    f32.close()


def test_bf16_steps_beside_other_decoders(itts, small_weights):
    """Threads of one process, all at once: two BF16 decoders' step(), an FP32 generate() and FP32
    step() (persistent grids), and a codec decoding new lengths (graph captures).  Every result is
    what the call gives alone, and a BF16 step alone again takes the persistent kernel."""
    bf = [itts.GptDecoder(small_weights, kv_capacity=512, weight_dtype="bf16") for _ in range(2)]
    f32 = [itts.GptDecoder(small_weights, kv_capacity=512) for _ in range(2)]
    codec = itts.EnhancedCodec(itts.make_synthetic_codec_weights(seed=5))
    o = itts.GenerationOptions(seed=3, suppress_stop=True)
    codes = [int(c) for c in np.random.default_rng(1).integers(0, 8192, 60)]

    def bf_steps(i):
        out = steps(bf[i], prefix_of(30 + i), codes[:24])
        assert bf[i].last_timing()["decode_path"] in ("step", "multi")
        return out

    calls = {
        "bf16 a": lambda: bf_steps(0),
        "bf16 b": lambda: bf_steps(1),
        "f32 generate": lambda: f32[0].generate(prefix_of(40), o, 64).codes,
        "f32 step": lambda: steps(f32[1], prefix_of(41), codes[:24]),
        "codec": lambda: [codec.decode(codes[:n]) for n in range(10, 26)],
    }
    ref = {k: f() for k, f in calls.items()}
    assert bf[1].last_timing()["decode_path"] == "step"
    out, errors = {}, []

    def run(k, f):
        try:
            out[k] = [f() for _ in range(3)]
        except Exception as e:  # reported below: a thread's exception is not raised by join()
            errors.append((k, e))

    threads = [threading.Thread(target=run, args=kf) for kf in calls.items()]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not errors, errors
    for k, r in ref.items():
        for got in out[k]:
            if k == "f32 generate":
                assert got == r, k
            else:
                assert all(same_bits(a, b) for a, b in zip(got, r)), k
    for d in bf:
        steps(d, prefix_of(30), codes[:2])
        assert d.last_timing()["decode_path"] == "step"
    for d in bf + f32 + [codec]:
        d.close()


def test_bf16_step_repeated_on_the_multikernel_path_after_a_timeout(itts, small_weights, env):
    """ITTS_GPT_STEP_TIMEOUT_ONCE=1: the decoder's first persistent step is reported as a hand-off
    that timed out.  A BF16 step() is then repeated on the multi-kernel path: the same logits, one
    row cached, and the later steps stay on that path.  An FP32 step() raises, caches nothing, and
    the next one works."""
    env("ITTS_GPT_STEP_TIMEOUT_ONCE", "0")
    plain = itts.GptDecoder(small_weights, kv_capacity=256, weight_dtype="bf16")
    plain32 = itts.GptDecoder(small_weights, kv_capacity=256)
    env("ITTS_GPT_STEP_TIMEOUT_ONCE", "1")
    dec = itts.GptDecoder(small_weights, kv_capacity=256, weight_dtype="bf16")
    dec32 = itts.GptDecoder(small_weights, kv_capacity=256)
    prefix = prefix_of(21)
    ref, got = steps(plain, prefix), [dec.prefill(prefix)]
    for i, c in enumerate(CODES):
        got.append(dec.step(c, i + 2))
        assert dec.last_timing()["decode_path"] == "multi"
        assert dec.cached_tokens() == 22 + i
    assert plain.last_timing()["decode_path"] == "step"
    assert all(same_bits(a, b) for a, b in zip(got, ref))
    dec32.prefill(prefix)
    with pytest.raises(itts.GptRuntimeError, match="hand-off timed out"):
        dec32.step(CODES[0], 2)
    assert dec32.cached_tokens() == 21
    plain32.prefill(prefix)
    for i, c in enumerate(CODES):
        assert same_bits(dec32.step(c, i + 2), plain32.step(c, i + 2))
        assert dec32.last_timing()["decode_path"] == "step"
    for d in (dec, dec32, plain, plain32):
        d.close()
