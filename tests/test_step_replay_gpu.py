"""mi_decoder_step records a step that comes twice in a row under the same circumstances and replays it: every step
leaves the residual stream, the logits and the token of a step whose launches were enqueued one by one (which a decoder that is
stepped on two streams in turn always does), also when the circumstances change in between: position and token, prompts,
attention splits, the GEMV arithmetic, a weight registered with other scales, the stream, a caller's own recording."""
import numpy as np
import pytest

from helpers import mil
from test_prefill_slices_gpu import VOCAB, _decoder

pytestmark = pytest.mark.gpu

SHAPE = (576, 1536, 9, 3, 64)


class Stepper:
    """A decoder and where it is stepped: always on one queue, or on two in turn."""

    def __init__(self, kind, queues):
        self.queues, self.turn = queues, 0
        self.dec, self.bufs, self.keep = _decoder(queues[0], kind, *SHAPE, False)

    def queue(self):
        return self.queues[self.turn % len(self.queues)]

    def step(self):
        q = self.queue()
        assert self.dec.step(q)
        q.finish()
        self.turn += 1

    def outputs(self):
        out = [np.array(self.dec.read(self.queues[0]), np.int64)]
        for ptr, n in ((mil.lib().mi_decoder_buffer(self.dec.handle, 0), SHAPE[0]), (self.dec.logits_ptr, VOCAB)):
            host = np.empty(n, np.uint16)
            assert mil.lib().mi_memcpy_d2h(host.ctypes.data, ptr, 2 * n, self.queues[0].handle)
            out.append(host)
        return out


def _pair(kind):
    assert mil.lib().mi_init(0) == 1
    q = mil.Queue()
    return Stepper(kind, [q]), Stepper(kind, [q, mil.Queue()])


def _same(a, b, what):
    for x, y in zip(a.outputs(), b.outputs()):
        assert np.array_equal(x, y), what


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
def test_replayed_steps_equal_plain_ones(kind):
    a, b = _pair(kind)
    def both(f):
        f(a), f(b)
    def steps(n, what):
        for t in range(n):
            both(lambda s: s.step())
            _same(a, b, (what, t))
    both(lambda s: s.dec.reset(s.queues[0], 0, 5))
    steps(5, "from the start")
    both(lambda s: s.dec.set_token(s.queues[0], 77))
    steps(2, "token set")
    both(lambda s: s.dec.reset(s.queues[0], 3, 9))
    steps(3, "position set")
    both(lambda s: s.dec.prefill(s.queues[0], [(13 * t) % VOCAB for t in range(200)], 0))
    steps(4, "behind a prompt")
    both(lambda s: s.dec.set_attention_splits(4))
    steps(4, "splits")
    both(lambda s: s.dec.set_attention_splits(0))
    steps(4, "no splits")
    if kind == "q4":
        for q in b.queues:
            assert mil.lib().mi_stream_set_modes(q.handle, 0, -1)
        steps(3, "exact Q4")
        for q in b.queues:
            assert mil.lib().mi_stream_set_modes(q.handle, -1, -1)
        steps(3, "throughput Q4")


def test_a_weight_registered_again_takes_effect():
    a, b = _pair("int8")
    for s in (a, b):
        assert s.dec.reset(s.queues[0], 0, 5)
    for turn in range(10):
        if turn in (4, 8):                      # one matrix with scales of its own, then both decoders alike again
            for s in (a, b) if turn == 4 else (a,):
                scale = mil.Buffer.from_host(np.full(SHAPE[1], 0x2000 + turn, np.uint16))
                s.keep.append(scale)
                assert mil.nnopt_register_int8_weight(s.bufs["wgate"][1], scale, SHAPE[1], SHAPE[0])
        a.step(), b.step()
        if turn < 8:
            _same(a, b, turn)
    assert any(not np.array_equal(x, y) for x, y in zip(a.outputs(), b.outputs()))     # the last change was a's alone


def test_other_streams_and_a_callers_recording():
    a, b = _pair("int8")
    for s in (a, b):
        assert s.dec.reset(s.queues[0], 0, 5)
    own, other = a.queues[0], mil.Queue()
    for turn in range(18):
        if turn == 6:
            a.queues = [other]                  # recorded again for the other stream
        if turn == 10:
            a.queues = [mil.Queue(default=True)]          # the null stream: never recorded
        if turn == 12:
            a.queues = [own]                    # the first recording again
        if turn == 14:
            with mil.Graph(own) as graph:
                assert a.dec.step(own)
        if turn >= 14:
            graph.launch()
            own.finish()
        else:
            a.step()
        b.step()
        _same(a, b, turn)


def test_two_decoders_in_turn_and_decoders_that_come_and_go():
    a, b = _pair("int8")
    c = Stepper("int8", a.queues)
    for s in (a, b, c):
        assert s.dec.reset(s.queues[0], 0, 5)
    for turn in range(6):
        for s in (a, b, c):
            s.step()
        _same(a, b, turn)
        _same(c, b, turn)
    for _ in range(5):
        d = Stepper("int8", a.queues)
        assert d.dec.reset(d.queues[0], 0, 5)
        for _ in range(4):
            assert d.dec.step(a.queues[0])      # the last replay still runs when the decoder goes
        del d
