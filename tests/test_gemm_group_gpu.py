"""GEMM projections of one x given together (mi_linear_batch) against the same projections given one by one
(mi_linear): one launch serves several matrices, and every output keeps its order of operations, so the two agree
bit for bit.  Widths around the tiles along N (16, 64, 256), rows around the tiles along M and around the lines
between the kernels, matrices whose own plans differ, and outputs that must not share a launch."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

SHAPES = [(128, [64, 16, 16]), (896, [896, 128, 128]), (576, [577, 191, 15, 3]), (896, [4864, 4864]), (1152, [300, 300, 300, 300, 300])]


def _weights(kind, n, k, seed, keep):
    w = mil.synth_normal_f16(seed, 0.02, (n, k))
    if kind == "f16":
        keep.append(mil.Buffer.from_host(w))
        return keep[-1]
    q, s = mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)
    qb, sb = mil.Buffer.from_host(q), mil.Buffer.from_host(s)
    keep += [qb, sb]
    assert (mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight)(qb, sb, n, k)
    return qb


def _together_as_one_by_one(queue, kind, rows, k, widths):
    keep = []
    x = mil.Buffer.from_host(mil.synth_normal_f16(5 + rows, 1.0, (rows, k)))
    ws = [_weights(kind, n, k, 100 + j, keep) for j, n in enumerate(widths)]
    fill = np.full(1, 0x7bff, np.uint16)
    one = [mil.Buffer.from_host(np.repeat(fill, rows * n)) for n in widths]
    many = [mil.Buffer.from_host(np.repeat(fill, rows * n)) for n in widths]
    print(f"{kind} rows {rows} K {k} N {widths}", flush=True)
    for n, w, o in zip(widths, ws, one):
        assert mil.pytorch_linear(queue, rows, n, k, x, w, o)
    calls = mil.make_calls([(rows, n, k, x, w, o) for n, w, o in zip(widths, ws, many)])
    assert mil.linear_batch(queue, calls) == len(widths)
    queue.finish()
    for n, a, b in zip(widths, one, many):
        assert np.array_equal(a.read(np.uint16, (rows, n)), b.read(np.uint16, (rows, n))), (rows, k, n)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows,mode", [(2, 5), (15, 5), (15, 3), (16, 0), (17, 0), (48, 0), (65, 0), (129, 0), (300, 0), (1025, 0)])
def test_together_as_one_by_one(kind, rows, mode):
    """Mode 0: the library's own choice of kernel; 5 and 3 name the streaming and the wide kernel."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode if mode else -1)
    for k, widths in SHAPES:
        _together_as_one_by_one(queue, kind, rows, k, widths)
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows", [2, 4, 7, 12, 15])
def test_together_where_gemv_and_gemm_meet(kind, rows):
    """Below 16 rows a matrix goes to the GEMV or to the GEMM by its size: a neighbour of the other kind does not
    change which, whichever of the two comes first.  (Q4 rows of GEMV in their exact mode: the throughput order is
    chosen by the rows of a launch, and so not alike for one matrix and for several.)"""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    assert mil.lib().mi_stream_set_modes(queue.handle, 0, -1)
    for k, widths in [(896, [128, 896, 4864]), (896, [4864, 896, 128]), (576, [64, 576, 64, 1536]), (4864, [64, 896]), (104, [64, 896])]:
        if kind != "q4" or k % 32 == 0:
            _together_as_one_by_one(queue, kind, rows, k, widths)
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)


def test_dependent_calls_keep_their_order():
    """The second call writes the first one's output again, the third reads it: as one by one."""
    assert mil.lib().mi_init(0) == 1
    queue, keep, rows, n = mil.Queue(), [], 40, 256
    x = mil.Buffer.from_host(mil.synth_normal_f16(1, 1.0, (rows, n)))
    ws = [_weights("int8", n, n, 7 + j, keep) for j in range(3)]
    got = []
    for together in (False, True):
        y, z = mil.Buffer(2 * rows * n), mil.Buffer(2 * rows * n)
        plan = [(rows, n, n, x, ws[0], y), (rows, n, n, x, ws[1], y), (rows, n, n, y, ws[2], z)]
        if together:
            assert mil.linear_batch(queue, mil.make_calls(plan)) == 3
        else:
            for c in plan:
                assert mil.pytorch_linear(queue, *c)
        queue.finish()
        got.append((y.read(np.uint16, (rows, n)), z.read(np.uint16, (rows, n))))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
