"""mi_linear_batch enqueues its calls "in order, exactly as n calls of mi_linear would" also where one of them is refused:
the calls in front of it are enqueued and counted, those behind it are not touched, whatever launch they could share."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

FILL = 0x7bff


class _Calls:
    """Calls (rows, N, K, x, W, out), each with buffers of its own; `bad` says what is wrong with one."""

    def __init__(self, rows, kind):
        self.rows, self.kind, self.keep, self.seed = rows, kind, [], 1

    def up(self, a):
        self.keep.append(mil.Buffer.from_host(a))
        return self.keep[-1]

    def make(self, n=64, k=576, x=None, bad=None):
        self.seed += 1
        k = {"K": 6, "long K": 32772, "K of several rows": 36}.get(bad, k)
        if x is None or k != 576:
            x = self.up(mil.synth_normal_f16(self.seed, 1.0, (self.rows, k + 8))).ptr
        w = mil.synth_normal_f16(self.seed, 0.02, (n, k))
        if self.kind == "int8" and bad is None:
            q, s = mil.quantize_int8(w)
            w = self.up(q).ptr
            assert mil.lib().mi_register_int8_weight(w, self.up(s).ptr, n, k)
        else:
            w = self.up(np.concatenate([w.ravel(), np.zeros(8, np.float16)])).ptr
        out = self.up(np.full(self.rows * n + 8, FILL, np.uint16))
        at = {"x": (2, 0, 0), "W": (0, 2, 0), "out": (0, 0, 1)}.get(bad, (0, 0, 0))
        return (self.rows, n, k, x + at[0], w + at[1], out.ptr + at[2]), out


@pytest.mark.parametrize("kind", ["f16", "int8"])
@pytest.mark.parametrize("bad,rows", [("K", 1), ("K", 4), ("long K", 1), ("K of several rows", 4), ("x", 1), ("x", 4), ("W", 1), ("W", 4),
                                      ("out", 1)])
@pytest.mark.parametrize("shared_x", [False, True])
@pytest.mark.parametrize("front", [0, 1, 2])
def test_refused_by_the_gemv(kind, bad, rows, shared_x, front):
    """A shape or an operand that the GEMV's host check refuses, between calls that it takes."""
    assert mil.lib().mi_init(0) == 1
    queue, c = mil.Queue(), _Calls(rows, kind)
    x = c.up(mil.synth_normal_f16(99, 1.0, (rows, 584))).ptr if shared_x else None
    print(kind, bad, rows, shared_x, front, flush=True)
    calls = [c.make(x=x) for _ in range(front)] + [c.make(x=x, bad=bad)] + [c.make(x=x) for _ in range(2)]
    assert not mil.lib().mi_linear(queue.handle, *calls[front][0])
    assert mil.linear_batch(queue, mil.make_calls([a for a, _ in calls])) == front
    queue.finish()
    for j, (args, out) in enumerate(calls):
        got = out.read(np.uint16, (rows * args[1] + 8,))
        if j >= front:
            assert (got == FILL).all(), j
        else:
            want = c.up(np.full(rows * args[1] + 8, FILL, np.uint16))
            assert mil.lib().mi_linear(queue.handle, *args[:5], want.ptr)
            queue.finish()
            assert np.array_equal(got, want.read(np.uint16, (rows * args[1] + 8,))), j


@pytest.mark.parametrize("mode,bad", [(5, (65, 64, 576)), (211, (16, 64, 192))], ids=["rows beyond the kernel", "slices that do not fit"])
@pytest.mark.parametrize("rows", [1, 16])
def test_refused_by_the_gemm(mode, bad, rows):
    """A call that a pinned kernel has no launch for, between calls that it, or the GEMV, takes and that could share one."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode)
    good, other = _Calls(rows, "int8"), _Calls(bad[0], "int8")
    print(mode, bad, rows, flush=True)
    calls = [good.make(), other.make(n=bad[1], k=bad[2]), good.make(), good.make()]
    assert not mil.lib().mi_linear(queue.handle, *calls[1][0])
    assert mil.linear_batch(queue, mil.make_calls([a for a, _ in calls])) == 1
    queue.finish()
    for j, (args, out) in enumerate(calls):
        assert (out.read(np.uint16, (args[0] * args[1] + 8,)) == FILL).all() == (j > 0), j
