"""The 64 x 64 tile kernel (named by mode 2) sums K in one order whatever else the launch holds: a row of x has the same
bits among 65, 300 or 1100 rows, a matrix the same bits by itself and beside others of one x.  K above and below 12
tiles and with an odd number of them, odd numbers of tile columns (which are walked in bands per XCD), and three
matrices that have at most a tile per CU each and more together."""
import numpy as np
import pytest

from helpers import mil
from test_gemm_group_gpu import _together_as_one_by_one, _weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["f16", "int8"])
@pytest.mark.parametrize("k", [576, 896, 960, 1536])
@pytest.mark.parametrize("n", [960, 1152])
def test_a_row_among_few_and_many(kind, k, n):
    assert mil.lib().mi_init(0) == 1
    queue, keep, most = mil.Queue(), [], 1100
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 2)
    x, w = mil.Buffer.from_host(mil.synth_normal_f16(11, 1.0, (most, k))), _weights(kind, n, k, 12, keep)
    got = {}
    for rows in (65, 300, most):
        print(f"{kind} rows {rows} K {k} N {n}", flush=True)
        assert mil.linear_plan(queue, rows, n, k, x, w)[0] == 2
        out = mil.Buffer(2 * rows * n)
        assert mil.pytorch_linear(queue, rows, n, k, x, w, out)
        queue.finish()
        got[rows] = out.read(np.uint16, (rows, n))
    for rows in (65, 300):
        assert np.array_equal(got[rows], got[most][:rows]), rows


@pytest.mark.parametrize("kind", ["f16", "int8"])
@pytest.mark.parametrize("rows,k,widths", [(300, 960, [1920, 1920, 1920]), (300, 896, [960, 896, 64]), (1000, 896, [896, 128, 128]),
                                           (65, 1536, [577, 191, 15, 3])])
def test_together_as_one_by_one(kind, rows, k, widths):
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 2)
    _together_as_one_by_one(queue, kind, rows, k, widths)


@pytest.mark.parametrize("kind,rows,n,k,kernel", [("int8", 2048, 960, 960, 2), ("f16", 1184, 1600, 960, 2), ("f16", 1408, 960, 576, 2),
                                                  ("int8", 320, 5120, 960, 1), ("f16", 416, 5120, 960, 1), ("f16", 704, 3072, 576, 1)])
def test_tiles_in_bands_are_chosen_where_they_are_faster(kind, rows, n, k, kernel):
    """Odd numbers of tile columns, 75 tiles and more, K to 1024: the 64 x 64 tiles (2); even numbers: the wide kernel (1)."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    x, w = mil.Buffer(2 * rows * k), _weights(kind, n, k, 12, keep)
    assert mil.linear_plan(queue, rows, n, k, x, w)[0] == kernel
