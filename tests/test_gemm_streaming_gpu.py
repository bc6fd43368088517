"""The streaming kernel (named by mode 5) and its sums for another launch (linear_slices), on integers: every product and
sum is exact in fp32 whatever the order, so the result is integer arithmetic's, bit for bit.  Rows around the 16-row
tiles; strips that end inside a tile of one and of two; K of one unit of 64, of fewer and of more units than wavefronts
share it, and of more than a ring holds (32 768: 64 units a wavefront with 8 wavefronts)."""
import ctypes

import numpy as np
import pytest

from helpers import mil
from test_gemm_many_gpu import _check, _weight
from test_prefill_slices_mode4_gpu import _slices

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64), (15, 128), (17, 576), (33, 896), (130, 1536), (4132, 320), (48, 32768)]


def _weights(kind, n, k, rng, keep):
    """-> device weights, their integer values, the scale they are to be multiplied with (a power of two per row)"""
    if kind == "f16":
        q = rng.integers(-8, 9, (n, k))
        keep.append(mil.Buffer.from_host(q.astype(np.float16)))
        return keep[-1], q, np.ones(n)
    scale = 2.0 ** rng.integers(-9, -5, n)
    if kind == "int8":
        q, stored, scales = rng.integers(-127, 128, (n, k)), None, scale
        stored = q.astype(np.int8)
    else:
        nib = rng.integers(0, 16, (n, k))
        q, stored = nib - 8, (nib[:, 0::2] | (nib[:, 1::2] << 4)).astype(np.uint8)
        scales = np.repeat(scale[:, None], k // 32, axis=1)
    w, s = mil.Buffer.from_host(stored), mil.Buffer.from_host(scales.astype(np.float16))
    keep += [w, s]
    assert (mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight)(w, s, n, k)
    return w, q, scale


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows", [2, 16, 17, 33, 49, 64])
def test_exact_on_integers(kind, rows):
    assert mil.lib().mi_init(0) == 1
    queue, keep, rng = mil.Queue(), [], np.random.default_rng(rows)
    for n, k in SHAPES:
        w, q, scale = _weights(kind, n, k, rng, keep)
        x = rng.integers(-3, 4, (rows, k))
        xb, out = mil.Buffer.from_host(x.astype(np.float16)), mil.Buffer.from_host(np.full(rows * n + 8, 0x7bff, np.uint16))
        print(f"{kind} rows {rows} N {n} K {k}", flush=True)
        total = (x @ q.T).astype(np.float64)
        assert np.abs(total).max() < 2 ** 24
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, 5)
        assert mil.linear_plan(queue, rows, n, k, xb, w)[0] == 4
        assert mil.pytorch_linear(queue, rows, n, k, xb, w, out)
        queue.finish()
        got = out.read(np.uint16, (rows * n + 8,))
        assert np.all(got[-8:] == 0x7bff)
        with np.errstate(over="ignore"):
            want = (total * scale).astype(np.float32).astype(np.float16)
        assert np.array_equal(got[:-8].view(np.float16).reshape(rows, n), want), (n, k)
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)
        sums, scales = ctypes.c_void_p(), ctypes.c_void_p()
        slices = _slices()(queue.handle, rows, n, k, xb.ptr, w.ptr, ctypes.byref(sums), ctypes.byref(scales))
        assert slices >= 0
        if slices:
            assert n % 4 == 0 and k >= 64 * 4 * slices
            host = np.empty((slices, rows, n), np.float32)
            queue.finish()
            assert mil.lib().mi_memcpy_d2h(host.ctypes.data, sums.value, host.nbytes, queue.handle)
            want = total if kind != "q4" else total * scale
            assert np.array_equal(host.astype(np.float64).sum(0), want), (n, k, slices)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows", [2, 65, 96, 97, 300, 1200])
def test_tiles_of_rows_exact_on_integers(kind, rows):
    """Mode 6: tiles of 32, 48 and 64 rows with a last one that is not full, of 16, 32 and 64 columns likewise, K in 2, 4 and 8
    slices; and the library's own choice at the same calls."""
    assert mil.lib().mi_init(0) == 1
    queue, keep, rng = mil.Queue(), [], np.random.default_rng(rows)
    for n, k in [(1, 64), (130, 576), (904, 960), (896, 4864), (1700, 128), (3080, 192), (9728, 128)]:
        w, q, scale = _weights(kind, n, k, rng, keep)
        x = rng.integers(-3, 4, (rows, k))
        xb = mil.Buffer.from_host(x.astype(np.float16))
        total = x.astype(np.float64) @ q.T.astype(np.float64)
        assert np.abs(total).max() < 2 ** 24
        with np.errstate(over="ignore"):
            want = (total * scale).astype(np.float32).astype(np.float16)
        for mode in (6, -1):
            out = mil.Buffer.from_host(np.full(rows * n + 8, 0x7bff, np.uint16))
            assert mil.lib().mi_stream_set_modes(queue.handle, -1, mode)
            plan = mil.linear_plan(queue, rows, n, k, xb, w)
            print(f"{kind} rows {rows} N {n} K {k} mode {mode} plan {plan}", flush=True)
            assert mode != 6 or plan[0] == 6
            assert mil.pytorch_linear(queue, rows, n, k, xb, w, out)
            queue.finish()
            got = out.read(np.uint16, (rows * n + 8,))
            assert np.all(got[-8:] == 0x7bff)
            assert np.array_equal(got[:-8].view(np.float16).reshape(rows, n), want), (n, k, mode)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows", [65, 97, 128, 300, 513])
def test_calls_in_tiles_of_rows_together_as_one_by_one(kind, rows):
    """Independent calls of different x and K beyond 64 rows: one launch for those in tiles of rows, 2, 4 and 8 slices of K
    side by side, ragged widths, a call of another kernel between them; each output bit for bit that of the call alone."""
    assert mil.lib().mi_init(0) == 1
    queue, keep, calls = mil.Queue(), [], []
    for j, (k, n) in enumerate([(896, 1152), (896, 130), (576, 9728), (4864, 896), (64, 1), (960, 2560), (128, 4864), (2560, 17)]):
        x = mil.Buffer.from_host(mil.synth_normal_f16(3 + j, 1.0, (rows, k)))
        keep.append(x)
        calls.append((rows, n, k, x, _weight(kind, n, k, 60 + j, keep)))
    plans = {mil.linear_plan(queue, *c)[0] for c in calls}
    print(f"{kind} rows {rows} plans {plans}", flush=True)
    assert 6 in plans
    _check(queue, calls, 3)
