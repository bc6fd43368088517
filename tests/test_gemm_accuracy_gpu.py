"""The matrix-core GEMM's error against 64 bits (2-norm of the difference over 2-norm of the result) is that of rounding the
exact result to fp16 once: sums in fp32 over K = 64 .. 4864, in any kernel, tile and number of slices, move a few outputs in
a thousand to the neighbouring fp16 number, which adds less than a thousandth to it.  Shapes that each kernel has by the library's own
choice, and the tiles of rows by name; Q4 weights as q * scale exactly."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu


def _weights(kind, n, k, keep):
    """-> device weights, their values in 64 bits"""
    w = mil.synth_normal_f16(n, 0.02, (n, k))
    if kind == "f16":
        keep.append(mil.Buffer.from_host(w))
        return keep[-1], w.astype(np.float64)
    if kind == "int8":
        q, s = mil.quantize_int8(w)
        value = q.astype(np.float64) * s.reshape(n, 1).view(np.float16).astype(np.float64)
        register = mil.nnopt_register_int8_weight
    else:
        q, s = mil.quantize_q4(w)
        value = np.empty((n, k))
        value[:, 0::2], value[:, 1::2] = (q & 15).astype(np.float64) - 8, (q >> 4).astype(np.float64) - 8
        value *= np.repeat(s.reshape(n, k // 32).view(np.float16).astype(np.float64), 32, axis=1)
        register = mil.nnopt_register_q4_weight
    wb, sb = mil.Buffer.from_host(q), mil.Buffer.from_host(s)
    keep += [wb, sb]
    assert register(wb, sb, n, k)
    return wb, value


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows,n,k", [(16, 896, 4864), (37, 960, 2560), (64, 1152, 896), (100, 896, 4864), (300, 1152, 896), (300, 9728, 896),
                                      (700, 960, 960), (1200, 896, 896), (2048, 1536, 576), (130, 1024, 64)])
def test_no_more_than_one_rounding(kind, rows, n, k):
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    w, value = _weights(kind, n, k, keep)
    x = mil.synth_normal_f16(rows, 1.0, (rows, k))
    want = x.astype(np.float64) @ value.T
    once = np.linalg.norm(want.astype(np.float16).astype(np.float64) - want) / np.linalg.norm(want)
    xb, out = mil.Buffer.from_host(x), mil.Buffer(2 * rows * n)
    for mode in (-1, 6):
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode)
        plan = mil.linear_plan(queue, rows, n, k, xb, w)
        assert mil.pytorch_linear(queue, rows, n, k, xb, w, out)
        queue.finish()
        got = out.read(np.float16, (rows, n)).astype(np.float64)
        error = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"{kind} {rows} x {n} x {k} plan {plan}: {error:.4e}, one rounding {once:.4e}", flush=True)
        assert error <= 1.001 * once
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)
