"""The choice between the streaming kernel in tiles of rows (mode 6) and the other GEMM kernels, by the clock, as
tests/test_gemm_plan_gpu.py holds the choice among those: no more than 20 % behind the fastest pinned one.  Calls on
both sides of every line that rows_preferred draws: many columns, a short K, many outputs, a long K with the wide
kernel in slices (mode 100 s + 10 + t), and calls of some hundred rows, which the tiles of rows win."""
import pytest

from helpers import mil
from test_gemm_plan_gpu import _time_us, queue  # noqa: F401
from test_gemm_group_gpu import _weights

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
