"""The SwiGLU in the launch of a stacked gate | up projection (what mi_decoder_prefill runs) against the projection
alone (mi_linear) with the SwiGLU computed here: rows and widths around the tiles, K in slices and not, every kind of
weights.  Gate and up are the same fp16 values on both sides, and the result is fp32 arithmetic (relative error below
1e-6) rounded to fp16 once: half a step of fp16, 2^-11 of the value and a hundredth more, or 2^-25 below the normal range."""
import ctypes

import numpy as np
import pytest

from helpers import mil
from test_gemm_group_gpu import _weights

pytestmark = pytest.mark.gpu


def _fused():
    f = mil.lib()["_ZN2mi10linear_gluEP12ihipStream_tiiiPKvS3_Pv"]       # mi::linear_glu
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p]
    f.restype = ctypes.c_int
    return f


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("inter,k", [(16, 64), (48, 1152), (1520, 576), (2560, 960), (4864, 896), (304, 4864)])
def test_swiglu_of_the_projection(kind, inter, k):
    assert mil.lib().mi_init(0) == 1
    queue, keep, taken = mil.Queue(), [], {}
    w = _weights(kind, 2 * inter, k, 31, keep)
    for rows in (2, 16, 17, 37, 48, 64, 65, 130, 300, 1025):
        for mode in (0, 3, 5) if rows <= 64 else (0, 3):
            assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode if mode else -1)
            x = mil.Buffer.from_host(mil.synth_normal_f16(rows, 3.0, (rows, k)))
            both, out = mil.Buffer(4 * rows * inter), mil.Buffer.from_host(np.full(rows * inter + 8, 0x7bff, np.uint16))
            print(f"{kind} rows {rows} mode {mode} inter {inter} K {k}", flush=True)
            assert mil.pytorch_linear(queue, rows, 2 * inter, k, x, w, both)
            took = _fused()(queue.handle, rows, 2 * inter, k, x.ptr, w.ptr, out.ptr)
            queue.finish()
            assert took >= 0
            taken[rows, mode] = took
            got = out.read(np.float16, (rows * inter + 8,))
            assert np.all(got[-8:].view(np.uint16) == 0x7bff)
            if not took:
                assert np.all(got.view(np.uint16) == 0x7bff)
                continue
            gu = both.read(np.float16, (rows, 2 * inter)).astype(np.float64).reshape(rows, inter // 16, 2, 16)
            g, u = gu[:, :, 0].reshape(rows, inter), gu[:, :, 1].reshape(rows, inter)
            want = g / (1.0 + np.exp(-g)) * u
            diff = np.abs(got[:-8].astype(np.float64).reshape(rows, inter) - want)
            assert np.all(diff <= 1.01 * 2.0 ** -11 * np.abs(want) + 1.01 * 2.0 ** -25)
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)
    assert all(taken[rows, 3] == 1 for rows in (2, 37, 130, 1025))
    if inter == 2560:
        assert taken[37, 0] == 1                                     # the streaming kernel, by its own choice
