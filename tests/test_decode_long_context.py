"""A decode step's attention at contexts that take several tiles of keys and of values: the step must equal the
prompt's reference-order attention bit for bit (mi_set_gemm_mode(1): other kernels, held to the CPU harness in
test_prefill.py).  Positions around the kernel's edges: the short form's 128 keys, batches of 32, key tiles of
512 (head width 128: 256) rows, value tiles of 256 (128)."""
import numpy as np
import pytest

from decode_harness import GpuDecoder, Model
from helpers import mil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,heads,positions", [
    ("head_dim_64", (6, 2, 64), [0, 1, 31, 32, 63, 95, 126, 127, 128, 129, 159, 160, 255, 256, 257, 287, 511, 512, 513,
                                 767, 768, 769, 1023, 1024, 1025, 1279]),
    ("head_dim_128", (4, 1, 128), [0, 30, 33, 64, 127, 128, 129, 130, 255, 256, 257, 383, 384, 385, 511, 512, 513, 639]),
])
def test_steps_equal_the_prompt_in_reference_order(name, heads, positions):
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    n_heads, n_kv, d = heads
    cfg = dict(hidden=256, inter=256, n_heads=n_heads, n_kv_heads=n_kv, head_dim=d, n_layers=2, vocab=512,
               max_pos=positions[-1] + 1, rms_eps=1e-6, rope_theta=100000.0)
    gd = GpuDecoder(Model(cfg, seed=91), queue)
    ids = [int(t) for t in np.random.default_rng(17).integers(0, cfg["vocab"], positions[-1] + 1)]
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 1)
    try:
        for pos in positions:
            assert gd.dec.prefill(queue, ids[:pos + 1])                       # rows 0 .. pos and what follows them
            want = (gd.dec.read(queue), gd.logits())
            assert gd.dec.reset(queue, pos, ids[pos]) and gd.dec.step(queue)   # the last of them again, as a step
            got = (gd.dec.read(queue), gd.logits())
            assert got[0] == want[0], (name, pos)
            assert np.array_equal(got[1], want[1]), (name, pos)
    finally:
        mil.lib().mi_stream_set_modes(queue.handle, -1, -1)
        gd.close()
