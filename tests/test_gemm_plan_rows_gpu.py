"""The choice between the streaming kernel in tiles of rows (mode 6) and the other GEMM kernels, by the clock, as
tests/test_gemm_plan_gpu.py holds the choice among those: no more than 20 % behind the fastest pinned one.  Calls on
both sides of every line that rows_preferred draws: many columns, a short K, many outputs, a long K with the wide
kernel in slices (mode 100 s + 10 + t), and calls of some hundred rows, which the tiles of rows win."""
import numpy as np
import pytest

from helpers import mil
from test_gemm_plan_gpu import _time_us, queue  # noqa: F401
from test_gemm_group_gpu import _weights
from test_gemm_many_gpu import _check

pytestmark = pytest.mark.gpu

BEHIND = 1.2
CALLS = [("f16", 56, 14592, 896), ("int8", 80, 19456, 896), ("f16", 200, 4096, 256), ("int8", 300, 4096, 256), ("f16", 512, 1024, 512),
         ("int8", 600, 896, 896), ("f16", 300, 1152, 896), ("q4", 300, 1152, 896), ("q4", 3072, 1536, 576), ("q4", 600, 2048, 8192),
         ("f16", 130, 2048, 8192), ("int8", 200, 960, 2560)]


@pytest.mark.parametrize("kind,M,N,K", CALLS)
def test_the_choice_is_near_the_fastest_pinned_kernel(queue, kind, M, N, K):  # noqa: F811
    keep = []
    x, w, out = mil.Buffer.from_host(mil.synth_normal_f16(71, 1.0, (M, K))), _weights(kind, N, K, 72, keep), mil.Buffer(2 * M * N)
    modes = [6] + [10 + t for t in range(1, 6) if 32 * (t - 1) < M] + ([2, 3] if kind != "q4" else [])
    modes += [100 * s + 10 + t for s in (2, 3, 8) for t in (1, 2, 3) if K >= 2560 and 4 * s * M * N <= 16 << 20]      # (a stream's workspace)
    worst = None
    for _ in range(3):                                   # further looks before a failure: boxes jitter
        own, plan = _time_us(queue, 0, M, N, K, x, w, out)
        pinned = {m: us for m in modes for us in [_time_us(queue, m, M, N, K, x, w, out)[0]] if us is not None}
        best = min(pinned, key=pinned.get)
        print(f"{kind} M={M} N={N} K={K} plan {plan} own {own:.2f} us, best pinned: mode {best} {pinned[best]:.2f} us", flush=True)
        worst = (own / pinned[best], plan, best)
        if worst[0] <= BEHIND:
            return
    assert False, f"{kind} M={M} N={N} K={K}: plan {worst[1]} takes {worst[0]:.2f} times what mode {worst[2]} does"


@pytest.mark.parametrize("kind,M,N,K,plan", [
    ("f16", 16, 1536, 576, (4, 16, 4)), ("int8", 24, 960, 704, (4, 32, 4)), ("q4", 16, 576, 576, (4, 16, 4)),       # a short K: 4 slices,
    ("int8", 24, 960, 768, (4, 32, 8)), ("q4", 24, 1600, 960, (4, 32, 8)),                                          # 8 from 768 on
    ("q4", 8, 2048, 2048, (4, 16, 8)), ("int8", 16, 2048, 2048, (4, 16, 8)),                                        # one block per strip,
    ("int8", 16, 2048, 2112, (4, 16, 16)), ("int8", 16, 896, 4864, (4, 16, 32)),                                    # over blocks beyond 4 units each
    ("int8", 32, 32000, 320, (4, 32, 4)), ("int8", 33, 32000, 320, (2, 64, 1)),                                     # many rows of W
    ("int8", 48, 14592, 896, (4, 48, 4)), ("int8", 49, 14592, 896, (2, 64, 1)), ("int8", 64, 9728, 896, (4, 64, 8))])
def test_slices_of_the_streaming_kernel_where_they_measured_faster(kind, M, N, K, plan):
    """Both sides of the lines of pick_shape and preferred for up to 64 rows."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    x, w = mil.Buffer(2 * M * K), _weights(kind, N, K, 73, keep)
    assert mil.linear_plan(queue, M, N, K, x, w) == plan


def _layer(kind, rows, shapes, keep):
    calls = []
    for j, (n, k) in enumerate(shapes):
        x = mil.Buffer.from_host(mil.synth_normal_f16(80 + j, 1.0, (rows, k)))
        keep.append(x)
        calls.append((rows, n, k, x, _weights(kind, n, k, 90 + j, keep)))
    return calls


@pytest.mark.parametrize("kind,rows,shapes", [
    ("int8", 2049, [(576, 576), (192, 576), (576, 576), (576, 1536)]), ("q4", 2305, [(576, 576), (192, 576), (576, 1536)]),
    ("f16", 900, [(896, 896), (128, 896), (896, 4864)]), ("int8", 2304, [(896, 896), (128, 896), (896, 4864)])])
def test_batches_beyond_2048_rows_and_long_calls_that_go_alone(kind, rows, shapes):
    """Tiles of rows at any number of rows share a launch but for the call that fills the chip and has a better tile of its
    own (the last one of the last two cases): each output bit for bit that of the call by itself."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    calls = _layer(kind, rows, shapes, keep)
    print(f"{kind} rows {rows} plans {[mil.linear_plan(queue, *c) for c in calls]}", flush=True)
    assert all(mil.linear_plan(queue, *c)[0] == 6 for c in calls)
    _check(queue, calls, 2)


def test_a_row_more_than_2048_costs_no_launch(queue):  # noqa: F811
    """Five small calls, which go out together: 2049 rows within 8 % of 2048 (1.5 times as long while they went one by one)."""
    keep, us = [], {}
    shapes = [(576, 576), (192, 576), (192, 576), (576, 576), (576, 1536)]
    for attempt in range(3):
        for rows in (2048, 2049):
            calls = _layer("int8", rows, shapes, keep)
            outs = [mil.Buffer(2 * rows * c[1]) for c in calls]
            keep += outs                                 # (the calls hold addresses only)
            arr = mil.make_calls([(*c, o) for c, o in zip(calls, outs)])
            assert mil.linear_batch(queue, arr) == len(calls)
            queue.finish()
            with mil.Graph(queue) as g:
                for _ in range(8):
                    assert mil.linear_batch(queue, arr) == len(calls)
            e0, e1, got = mil.Event(), mil.Event(), []
            for _ in range(9):
                e0.record(queue)
                g.launch()
                e1.record(queue)
                e1.synchronize()
                got.append(e0.elapsed_ms(e1) * 125)
            us[rows] = sorted(got)[4]
        print(us, flush=True)
        if us[2049] <= 1.08 * us[2048]:
            return
    assert False, us


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
def test_more_tiles_of_rows_than_a_grid_counts(kind):
    """65 535 in its third dimension: beyond 65 535 x 32 rows in taller tiles, beyond 65 535 x 64 not at all."""
    assert mil.lib().mi_init(0) == 1
    queue, keep, n, k = mil.Queue(), [], 16, 64
    rows = 65535 * 32 + 1
    w = _weights(kind, n, k, 74, keep)
    x, out, row = mil.Buffer(2 * rows * k), mil.Buffer(2 * rows * n), mil.synth_normal_f16(75, 1.0, (1, k))
    assert mil.lib().mi_memset(x.ptr, 0, 2 * rows * k, queue.handle)
    last = mil.Buffer.from_host(row)
    assert mil.lib().mi_memcpy_d2d(x.ptr + 2 * (rows - 1) * k, last.ptr, 2 * k, queue.handle)
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 6)
    for m, tile in ((rows, 48), (65535 * 64, 64), (65535 * 64 + 1, 0)):
        plan = mil.linear_plan(queue, m, n, k, x, w)
        print(f"{kind} {m} rows plan {plan}", flush=True)
        assert plan[0] == (6 if tile else -1) and plan[1] >= tile
    assert mil.pytorch_linear(queue, rows, n, k, x, w, out)
    two, want = mil.Buffer.from_host(np.concatenate([row, row])), mil.Buffer(4 * n)      # (the same slices of K: the same bits)
    assert mil.linear_plan(queue, 2, n, k, two, w)[0] == 6 and mil.pytorch_linear(queue, 2, n, k, two, w, want)
    queue.finish()
    got = out.read(np.uint16, (rows, n))
    assert np.array_equal(got[-1], want.read(np.uint16, (2, n))[0]) and got[-1].any()
    assert not got[:-1].any()
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)


@pytest.mark.parametrize("kind,M,N,K,kernel", [("int8", 1200, 960, 960, 6), ("f16", 1200, 960, 960, 6), ("int8", 1600, 320, 960, 6),
                                               ("int8", 2048, 320, 960, 2), ("int8", 2048, 576, 576, 6), ("f16", 1200, 1600, 960, 2)])
def test_tiles_of_rows_beside_64_x_64_tiles_in_bands(kind, M, N, K, kernel):
    """Odd numbers of columns of 64 x 64 tiles: the tiles of rows up to 7000 outputs per CU, by a K of 768 and more up to 7 rows."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    x, w = mil.Buffer(2 * M * K), _weights(kind, N, K, 76, keep)
    assert mil.linear_plan(queue, M, N, K, x, w)[0] == kernel
