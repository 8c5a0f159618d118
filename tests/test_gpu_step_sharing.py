"""Decode calls beside other work of the process (MI355X): they wait for nothing but their own
stream, and fail for nothing that other threads do."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from conftest import same_bits

pytestmark = pytest.mark.gpu

CODES = (17, 4000, 8191, 0, 300, 5)


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


def test_bf16_step_does_not_wait_for_the_null_stream(itts, small_weights, held_stream):
    dec = itts.GptDecoder(small_weights, kv_capacity=256, weight_dtype="bf16")
    ref = steps(dec, prefix_of(20))
    done = held_stream(True)
    got = steps(dec, prefix_of(20))
    assert not done.is_set(), "step() waited for the null stream"
    assert done.wait(10)
    assert all(same_bits(a, b) for a, b in zip(got, ref))
    dec.close()


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
