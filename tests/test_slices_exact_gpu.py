"""The sums that linear_slices leaves for another launch, [slices][M][N] in fp32 at the start of the stream's workspace, on
integers: their total is integer arithmetic's in any order.  Where a call has to be cut it is asserted to be: by the
streaming kernel up to 64 rows, in tiles of rows beyond, by the wide kernel; where it must not be, that nothing is
launched.  Columns in whole fours that end inside a strip of 16, row tiles that are not full, and what lies behind
the sums, which stays as it was."""
import ctypes

import numpy as np
import pytest

from helpers import mil
from test_gemm_streaming_gpu import _weights
from test_prefill_slices_mode4_gpu import _slices

pytestmark = pytest.mark.gpu

FEW = [(16, 132, 896), (16, 896, 896), (17, 132, 896), (37, 900, 960), (49, 1152, 896), (64, 132, 4864), (64, 960, 2560)]
MORE = [(65, 132, 896), (65, 1152, 896), (97, 900, 960), (97, 896, 4864), (130, 896, 896), (300, 896, 4864), (300, 900, 960),
        (301, 576, 1536), (600, 896, 4864), (600, 132, 2560), (705, 576, 1536)]
GUARD = 4096


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows,n,k", FEW + MORE)
def test_sums_for_another_launch(kind, rows, n, k):
    assert mil.lib().mi_init(0) == 1
    queue, keep, rng = mil.Queue(), [], np.random.default_rng(rows + n)
    w, q, scale = _weights(kind, n, k, rng, keep)
    x = rng.integers(-3, 4, (rows, k))
    xb, sums, scales = mil.Buffer.from_host(x.astype(np.float16)), ctypes.c_void_p(), ctypes.c_void_p()
    total = x.astype(np.float64) @ q.T.astype(np.float64)
    assert np.abs(total).max() < 2 ** 24
    args = (queue.handle, rows, n, k, xb.ptr, w.ptr, ctypes.byref(sums), ctypes.byref(scales))
    slices = _slices()(*args)
    print(f"{kind} {rows} x {n} x {k}: {slices} slices", flush=True)
    assert slices >= 2
    size = slices * rows * n
    pattern = np.full(size + GUARD, 0x7fa00001, np.uint32)       # no sum: a NaN
    queue.finish()
    assert 4 * pattern.size <= 16 << 20
    assert mil.lib().mi_memcpy_h2d(sums.value, pattern.ctypes.data, pattern.nbytes, queue.handle)
    assert _slices()(*args) == slices
    host = np.empty_like(pattern)
    queue.finish()
    assert mil.lib().mi_memcpy_d2h(host.ctypes.data, sums.value, host.nbytes, queue.handle)
    assert np.all(host[size:] == 0x7fa00001)
    got = host[:size].view(np.float32).reshape(slices, rows, n).astype(np.float64).sum(0)
    assert np.array_equal(got, total if kind != "q4" else total * scale)


@pytest.mark.parametrize("kind,rows,n,k", [("int8", 400, 1152, 896), ("f16", 400, 1600, 960), ("int8", 64, 9728, 896), ("f16", 300, 898, 960)])
def test_no_slices_where_the_launch_in_one_piece_is_the_faster_one(kind, rows, n, k):
    """... (the first two: by more than the sums cost), where the chip is full of strips, and for columns not in whole fours."""
    assert mil.lib().mi_init(0) == 1
    queue, keep, rng = mil.Queue(), [], np.random.default_rng(1)
    w, _, _ = _weights(kind, n, k, rng, keep)
    x, sums, scales = mil.Buffer(2 * rows * k), ctypes.c_void_p(), ctypes.c_void_p()
    assert _slices()(queue.handle, rows, n, k, x.ptr, w.ptr, ctypes.byref(sums), ctypes.byref(scales)) == 0
