"""mi_stream_create leaves nothing to run on the new stream, and the counters behind its workspace (slices of K that meet inside
a launch) are 0: a stream's first GEMM in slices is right."""
import ctypes

import numpy as np
import pytest

from helpers import mil
from test_gemm_group_gpu import _weights

pytestmark = pytest.mark.gpu


def test_a_new_stream_is_idle_and_its_counters_clear():
    assert mil.lib().mi_init(0) == 1
    hip, rows, n, k, keep = ctypes.CDLL("libamdhip64.so"), 16, 896, 4864, []
    hip.hipStreamQuery.argtypes = [ctypes.c_void_p]
    w, x = _weights("int8", n, k, 3, keep), mil.Buffer.from_host(mil.synth_normal_f16(1, 1.0, (rows, k)))
    want, busy, queues = None, 0, []
    for _ in range(12):
        queues.append(mil.Queue())
        busy += hip.hipStreamQuery(queues[-1].handle) != 0
        out = mil.Buffer.from_host(np.full(rows * n, 0x7bff, np.uint16))
        for _ in range(2):
            assert mil.pytorch_linear(queues[-1], rows, n, k, x, w, out)
        queues[-1].finish()
        got = out.read(np.uint16, (rows * n,))
        want = got if want is None else want
        assert np.array_equal(got, want)
    assert busy == 0
