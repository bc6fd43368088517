"""When a decoder's step is recorded and replayed (csrc/step_record.h), on the CPU with launches that are only counted: a
step is enqueued once, plainly or as a replay, whatever the recording did."""
import ctypes
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

DRIVER = """
#include "step_record.h"
using namespace mi;
struct Api {
    int launch_ok = 1, replay_ok = 1, outcome = 0;             // outcome: a Recorded
    int plain = 0, recorded = 0, replayed = 0, next_exec = 1, last_exec = 0;
    int enqueue() { ++plain; return launch_ok; }
    Recorded record(int* exec) {
        ++recorded;
        if (outcome == 0) *exec = next_exec++;
        return static_cast<Recorded>(outcome);
    }
    int replay(int exec) { ++replayed; last_exec = exec; return replay_ok; }
    long gone_stream = 0;
    int drained = 0, dropped = 0;                              // dropped: a bit per exec
    bool gone(const StepKey& k) { return reinterpret_cast<long>(k.stream) == gone_stream; }
    void drain() { ++drained; }
    void drop(int exec) { dropped |= 1 << exec; }
};
static Api api;
static StepRecordings<int>* held;
extern "C" void start() { delete held; held = new StepRecordings<int>; api = Api{}; }
extern "C" void set(int launch_ok, int outcome) { api.launch_ok = launch_ok; api.outcome = outcome; }
extern "C" int step(long stream, long workspace, int mode, int splits, int weights) {
    StepKey k;
    k.stream = reinterpret_cast<const void*>(stream); k.workspace = reinterpret_cast<const void*>(workspace);
    k.gemv_mode = mode; k.splits = splits; k.weights = weights;
    return held->step(api, k);
}
extern "C" void stream_goes(long stream) { api.gone_stream = stream; }
extern "C" void drops(int* out) { out[0] = api.drained; out[1] = api.dropped; }
extern "C" void counts(int* out) { out[0] = api.plain; out[1] = api.recorded; out[2] = api.replayed; out[3] = api.last_exec; }
"""


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    at = tmp_path_factory.mktemp("step")
    (at / "step.cpp").write_text(DRIVER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "adreno-llms_amd", "csrc"),
                           "-o", str(at / "step.so"), str(at / "step.cpp")])
    return ctypes.CDLL(str(at / "step.so"))


def _counts(rule):
    out = (ctypes.c_int * 4)()
    rule.counts(out)
    return list(out)


KEY = (1, 2, 0, 0, 1)


def test_plain_then_recorded_then_replayed(rule):
    rule.start()
    assert rule.step(*KEY) and _counts(rule) == [1, 0, 0, 0]
    assert rule.step(*KEY) and _counts(rule) == [1, 1, 1, 1]
    assert rule.step(*KEY) and _counts(rule) == [1, 1, 2, 1]
    for place, other in enumerate(((9, 2, 0, 0, 1), (1, 9, 0, 0, 1), (1, 2, 9, 0, 1), (1, 2, 0, 9, 1), (1, 2, 0, 0, 9))):
        assert rule.step(*other) and rule.step(*KEY) and _counts(rule) == [1 + 2 * (place + 1), 1, 2, 1]
    assert rule.step(*KEY) and _counts(rule) == [11, 1, 3, 1]


@pytest.mark.parametrize("outcome", [1, 2], ids=["a launch failed", "the runtime refused"])
@pytest.mark.parametrize("launch_ok", [0, 1])
def test_what_fails_while_it_is_recorded_is_enqueued_plainly(rule, outcome, launch_ok):
    """The step's result is that of the plain launches: a step that is at fault itself fails there again."""
    rule.start()
    rule.step(*KEY)
    rule.set(launch_ok, outcome)
    assert rule.step(*KEY) == launch_ok and _counts(rule) == [2, 1, 0, 0]
    rule.set(1, 0)
    assert rule.step(*KEY) == 1
    # refused: never tried again; otherwise the next step is recorded
    assert _counts(rule) == ([3, 1, 0, 0] if outcome == 2 else [2, 2, 1, 1])


def _drops(rule):
    out = (ctypes.c_int * 2)()
    rule.drops(out)
    return list(out)


def _steps(rule, key, n=3):
    """(plain steps, recordings, replays) of n steps in a row."""
    before = _counts(rule)
    for _ in range(n):
        assert rule.step(*key)
    return [b - a for a, b in zip(before, _counts(rule))][:3]


def test_weights_registered_again_any_number_of_times(rule):
    """Each version of the weights is recorded; of a full table the outdated ones go, behind one wait for the stream."""
    rule.start()
    for version in range(1, 30):
        assert _steps(rule, (1, 2, 0, 0, version)) == [1, 1, 2], version
        assert _drops(rule) == [(version - 1) // 8, (1 << (version - 1) // 8 * 8 + 1) - 2], version


def test_streams_that_come_and_go(rule):
    rule.start()
    for stream in range(1, 9):
        assert _steps(rule, (stream, 2, 0, 0, 1)) == [1, 1, 2]
    assert _steps(rule, (9, 2, 0, 0, 1)) == [3, 0, 0]          # eight that live: plainly
    rule.stream_goes(3)
    assert _steps(rule, (9, 2, 0, 0, 1)) == [0, 1, 3]          # (again the circumstances of the step before)
    assert _drops(rule) == [0, 1 << 3]
    for stream in (1, 2, 4, 5, 6, 7, 8, 9):
        assert _steps(rule, (stream, 2, 0, 0, 1)) == [1, 0, 2], stream


def test_outdated_recordings_of_another_stream_stay(rule):
    """Their last replay may still be running."""
    rule.start()
    for splits in range(8):
        assert _steps(rule, (1, 2, 0, splits, 1)) == [1, 1, 2]
    assert _steps(rule, (9, 2, 0, 0, 2)) == [3, 0, 0] and _drops(rule) == [0, 0]
    assert _steps(rule, (1, 2, 0, 0, 2)) == [1, 1, 2] and _drops(rule) == [1, 0b111111110]
    assert _steps(rule, (9, 2, 0, 0, 2)) == [1, 1, 2]


@pytest.mark.gpu
def test_more_circumstances_than_recordings():
    """A weight registered again and again, and streams that come and go, replay against plain launches (two streams in turn)."""
    import numpy as np

    from helpers import mil
    from test_step_replay_gpu import SHAPE, _pair, _same

    a, b = _pair("int8")
    for s in (a, b):
        assert s.dec.reset(s.queues[0], 0, 5)
    for version in range(20):
        if version % 3 == 2:
            a.queues = [mil.Queue()]
        for s in (a, b):
            scale = mil.Buffer.from_host(np.full(SHAPE[1], 0x1c00 + 16 * version, np.uint16))
            s.keep.append(scale)
            assert mil.nnopt_register_int8_weight(s.bufs["wgate"][1], scale, SHAPE[1], SHAPE[0])
        print("version", version, flush=True)
        for _ in range(3):
            a.step(), b.step()
        _same(a, b, version)


@pytest.mark.gpu
def test_another_thread_waits_on_the_stream():
    """Steps that are recorded, one decoder and set of splits after the other, while another thread does nothing but wait
    for their stream: neither a step nor a wait fails, and the outputs are those of steps that nobody waits for."""
    import threading

    import numpy as np

    from helpers import mil
    from test_step_replay_gpu import Stepper

    assert mil.lib().mi_init(0) == 1
    queue, outputs = mil.Queue(), []
    for watched in (False, True):
        stop, failed, waits = threading.Event(), [], [0]

        def wait():
            while not stop.is_set():
                waits[0] += 1
                if not mil.lib().mi_stream_sync(queue.handle):
                    failed.append(waits[0])

        thread = threading.Thread(target=wait)
        if watched:
            thread.start()
        try:
            for turn in range(3):
                s = Stepper("int8", [queue])
                assert s.dec.reset(queue, 0, 5 + turn)
                for splits in (0, 2, 4, 8):
                    print("decoder", turn, "splits", splits, "watched", watched, flush=True)
                    assert s.dec.set_attention_splits(splits)
                    assert all([s.dec.step(queue) for _ in range(4)])
                queue.finish()
                outputs.append(s.outputs())
        finally:
            stop.set()
            if watched:
                thread.join()
        assert not failed and (waits[0] > 12 or not watched), (failed, waits)
    for a, b in zip(outputs[:3], outputs[3:]):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
