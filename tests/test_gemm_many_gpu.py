"""GEMMs of a few rows that share no x, given together: independent calls of the streaming kernel go out as one launch
(launch_gemm_many), slices of K over blocks meet inside it, and every output is bit for bit that of the call by itself.
Rows around the 16-row tiles, strips and slices of every shape the plan has (x in LDS or not, 1 to 8 slices inside a
block, slices over blocks), launches that take more than half of a CU's LDS, more calls than a launch holds, calls of other
kernels between them; three times over, since the counters of the slices have to be back at 0."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

# (K, N): strips 1 .. 320, K over blocks (4864, 2560, 4096), x in LDS (896 and 576 with many strips), short K, a ragged N
SHAPES = [(896, 1152), (896, 896), (896, 4864), (896, 4864), (4864, 896), (576, 1), (2560, 960), (576, 1536), (64, 37), (128, 16),
          (4096, 130), (960, 5120), (4864, 15)]


def _weight(kind, n, k, seed, keep):
    w = mil.synth_normal_f16(seed, 0.02, (n, k))
    if kind == "f16":
        keep.append(mil.Buffer.from_host(w))
        return keep[-1]
    q, s = mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)
    qb, sb = mil.Buffer.from_host(q), mil.Buffer.from_host(s)
    keep += [qb, sb]
    assert (mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight)(qb, sb, n, k)
    return qb


def _blank(count):
    return mil.Buffer.from_host(np.full(count + 8, 0x7bff, np.uint16))


def _check(queue, calls, times):
    want = [_blank(c[0] * c[1]) for c in calls]
    for c, o in zip(calls, want):
        assert mil.pytorch_linear(queue, *c, o)
    queue.finish()
    want = [o.read(np.uint16, (c[0] * c[1] + 8,)) for c, o in zip(calls, want)]
    for turn in range(times):
        got = [_blank(c[0] * c[1]) for c in calls]
        assert mil.linear_batch(queue, mil.make_calls([(*c, o) for c, o in zip(calls, got)])) == len(calls)
        queue.finish()
        for c, w, o in zip(calls, want, got):
            assert np.array_equal(w, o.read(np.uint16, (c[0] * c[1] + 8,))), (c[:3], turn)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows,mode", [(2, 5), (5, 0), (15, 0), (16, 0), (17, 0), (33, 0), (48, 0), (49, 5), (64, 5), (64, 0)])
def test_calls_of_different_x(kind, rows, mode):
    """Mode 0: the library's own choice of kernel, which differs from call to call; 5 names the streaming kernel."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    # (Q4 rows of GEMV in their exact mode: the throughput order is chosen by the rows of a launch)
    assert mil.lib().mi_stream_set_modes(queue.handle, 0, mode if mode else -1)
    calls = []
    for j, (k, n) in enumerate(SHAPES):
        x = mil.Buffer.from_host(mil.synth_normal_f16(3 + j, 1.0, (rows, k)))
        keep.append(x)
        calls.append((rows, n, k, x, _weight(kind, n, k, 60 + j, keep)))
    print(f"{kind} rows {rows} mode {mode}", flush=True)
    _check(queue, calls, 3)


def test_more_calls_than_a_launch_holds():
    assert mil.lib().mi_init(0) == 1
    queue, keep, rows = mil.Queue(), [], 16
    calls = []
    for j in range(70):
        k, n = [(2560, 64), (576, 48)][j % 2]
        x = mil.Buffer.from_host(mil.synth_normal_f16(3 + j, 1.0, (rows, k)))
        keep.append(x)
        calls.append((rows, n, k, x, _weight("int8", n, k, 60 + j, keep)))
    _check(queue, calls, 2)


@pytest.mark.parametrize("kind,rows,n,k", [("int8", 16, 896, 4864), ("q4", 33, 896, 4864), ("f16", 64, 960, 2560), ("int8", 2, 17, 2048)])
def test_slices_over_blocks_meet_in_one_launch(kind, rows, n, k):
    """One call: repeated launches agree bit for bit whichever block arrives last, eagerly and as a replayed graph."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 5)
    x = mil.Buffer.from_host(mil.synth_normal_f16(1, 1.0, (rows, k)))
    w, out = _weight(kind, n, k, 2, keep), _blank(rows * n)
    assert mil.pytorch_linear(queue, rows, n, k, x, w, out)
    queue.finish()
    want = out.read(np.uint16, (rows * n + 8,))
    assert (want[-8:] == 0x7bff).all()
    with mil.Graph(queue) as graph:
        assert mil.pytorch_linear(queue, rows, n, k, x, w, out)
    for turn in range(20):
        if turn % 2:
            graph.launch()
        else:
            assert mil.pytorch_linear(queue, rows, n, k, x, w, out)
        queue.finish()
        assert np.array_equal(want, out.read(np.uint16, (rows * n + 8,))), turn
