"""Split decode attention where a block's run of keys is longer than a tile (256 keys at head width 64, 128 at 128): runs
one key short of a tile, a tile, and one and two keys over it, for the first and the second boundary; the current
position's key is then the last of a tile, alone in one, or in its middle.  Bar: that of test_attention_splits.py, on the
attention output against the CPU restatement of the reference's kernel (one key left out or taken twice among 500
turns the output by about 1 / sqrt(500), a cosine of 0.999)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from decode_harness import SMOL, GpuDecoder, Model, _lib as L
from helpers import assert_tolerance, mil
from test_attention_splits import _oracle_buffers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,cfg,splits,checked", [
    ("head_dim_64", dict(SMOL, n_layers=1, max_pos=1040), 2, [*range(508, 517), 700, *range(1020, 1030)]),
    ("head_dim_64", dict(SMOL, n_layers=1, max_pos=800), 3, [*range(764, 773)]),
    ("head_dim_128", dict(hidden=1024, inter=1536, n_heads=8, n_kv_heads=2, head_dim=128, n_layers=1, vocab=2048,
                          max_pos=520, rms_eps=1e-6, rope_theta=500000.0), 2, [*range(252, 261), 385, *range(508, 517)]),
])
def test_runs_of_several_tiles(name, cfg, splits, checked):
    L.orc_decoder_buffer.restype = C.c_void_p
    L.orc_decoder_buffer.argtypes = [C.c_void_p, C.c_int]
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    m = Model(cfg, seed=34)
    cs = m.c_struct()
    dec = L.orc_decoder_new(C.byref(cs), O.THREADS)
    gd = GpuDecoder(m, queue)
    nq = cfg["n_heads"] * cfg["head_dim"]
    got, margin, token = np.empty(nq, np.uint16), C.c_float(), 7
    try:
        assert gd.dec.set_attention_splits(splits) and gd.dec.reset(queue, 0, token)
        for pos in range(checked[-1] + 1):
            nxt = L.orc_decoder_step(dec, token, pos, None, None, C.byref(margin))
            assert gd.dec.set_token(queue, token) and gd.dec.step(queue)
            if pos in checked:
                queue.finish()
                want, _ = _oracle_buffers(dec, cfg)
                assert mil.lib().mi_memcpy_d2h(got.ctypes.data, mil.lib().mi_decoder_buffer(gd.dec.handle, 4), nq * 2, queue.handle)
                print(name, splits, "splits, pos", pos, flush=True)
                assert_tolerance(got.view(np.float16), want.view(np.float16))
            token = nxt                                   # both follow the reference's tokens
    finally:
        L.orc_decoder_free(dec)
        gd.close()
