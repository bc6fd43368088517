"""Where a prompt's projection is cut into slices that the next launch adds, mode 4 (Q4 weights as one fp16 term) weighs the
cut against its own launch in one piece, not against the two-term launch of the other modes, which is the dearer one."""
import ctypes

import pytest

from helpers import mil
from test_gemm_group_gpu import _weights

pytestmark = pytest.mark.gpu


def _slices():
    f = mil.lib()["_ZN2mi13linear_slicesEP12ihipStream_tiiiPKvS3_PPKfPS3_"]       # mi::linear_slices
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                  ctypes.c_void_p]
    f.restype = ctypes.c_int
    return f


# (rows, N, K, cut in modes 4 and 0); the estimates lie 0.25 us and more apart
@pytest.mark.parametrize("rows,n,k,cut", [(1000, 576, 576, False), (1600, 896, 896, False), (2000, 960, 2560, False),
                                          (300, 960, 960, True), (700, 960, 960, True)])
def test_cut_against_the_launch_that_runs(rows, n, k, cut):
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    w, x = _weights("q4", n, k, 7, keep), mil.Buffer.from_host(mil.synth_normal_f16(rows, 1.0, (rows, k)))
    sums, scale = ctypes.c_void_p(), ctypes.c_void_p()
    for mode in (4, -1):
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode)
        print(f"{rows} x {n} x {k} mode {mode}", flush=True)
        assert mil.linear_plan(queue, rows, n, k, x, w)[2] == 1 or cut
        got = _slices()(queue.handle, rows, n, k, x.ptr, w.ptr, ctypes.byref(sums), ctypes.byref(scale))
        queue.finish()
        assert got > 1 if cut else got == 0
