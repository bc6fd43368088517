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
