"""The prompt attention on the matrix cores (the default mode of mi_decoder_prefill) against the launches that
keep the reference's order (mi_set_gemm_mode(1)), which equal the CPU harness bit for bit (test_prefill.py).

Three layers, so that every row's attention reaches the compared residual stream through the keys and values of
the next layers, not the last row's alone.  What these models bring: scores below 1 nat, nearly even weights, and one
comparison per prompt, of the last row; single rows, large scores and values that are not finite are
test_prompt_attention_rows.py's.  Bound: the reference's order rounds scores (half a step of 2^-11 below 1),
exponentials and probabilities to fp16, the matrix cores' the exponentials, so the two sides' probabilities differ by up
to 2e-3 of themselves, with random signs; an attention output, an average over keys, differs by less, and the
projections by a fp16 rounding each: 2e-3 of the residual stream's 2-norm covers three layers of it (measured 3e-4 to
7e-4)."""
import numpy as np
import pytest

from decode_harness import GpuDecoder, Model
from helpers import mil

pytestmark = pytest.mark.gpu


def _cfg(n_heads, n_kv, head_dim, max_pos, hidden=256):
    return dict(hidden=hidden, inter=256, n_heads=n_heads, n_kv_heads=n_kv, head_dim=head_dim, n_layers=3, vocab=512,
                max_pos=max_pos, rms_eps=1e-6, rope_theta=100000.0)


CASES = [
    # (config, [(prompt rows, first position), ...]): rows around the 16 of a wavefront, keys around the 64 of a
    # tile, several tiles per wavefront, a first position inside a tile; one head per group to nine
    ("one_head_per_group", _cfg(4, 4, 64, 512), [(2, 0), (15, 0), (16, 0), (17, 1), (33, 63), (64, 0), (65, 64), (128, 0), (129, 3)]),
    ("three_per_group", _cfg(9, 3, 64, 512), [(31, 0), (48, 16), (65, 62), (200, 0), (255, 257)]),
    ("nine_per_group", _cfg(9, 1, 64, 300), [(5, 0), (71, 0), (130, 130)]),
    # few blocks and more than 512 keys: eight wavefronts, four to a set; positions past the last whole step
    ("long_keys", _cfg(7, 1, 64, 1100), [(40, 560), (3, 1000), (129, 700), (17, 1083)]),
    # enough blocks for the chip: eight wavefronts, two to a set
    ("many_rows", _cfg(16, 2, 64, 900), [(801, 0), (769, 131)]),
    ("head_dim_128", _cfg(4, 2, 128, 400), [(2, 0), (17, 0), (64, 1), (65, 127), (200, 200)]),
    # 16 blocks per 16 rows: the one-wavefront-per-set form of head width 128
    ("head_dim_128_many_rows", _cfg(16, 4, 128, 300), [(257, 0), (272, 28)]),
]


def _hidden(gd, n):
    out = np.empty(n, np.float16)
    gd.queue.finish()
    assert mil.lib().mi_memcpy_d2h(out.ctypes.data, mil.lib().mi_decoder_buffer(gd.dec.handle, 0), 2 * n, gd.queue.handle)
    return out.astype(np.float64)


@pytest.mark.parametrize("name,cfg,prompts", CASES, ids=[c[0] for c in CASES])
def test_prompt_attention_within_tolerance(name, cfg, prompts):
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    gd = GpuDecoder(Model(cfg, seed=77), queue)
    L = mil.lib()
    try:
        for rows, pos0 in prompts:
            ids = [int(t) for t in np.random.default_rng(rows + 1000 * pos0).integers(0, cfg["vocab"], pos0 + rows)]
            got = {}
            for mode in (1, 0):
                assert L.mi_stream_set_modes(queue.handle, -1, 1)
                if pos0:
                    assert gd.dec.prefill(queue, ids[:pos0])                # the older rows, the same on both sides
                assert L.mi_stream_set_modes(queue.handle, -1, mode)
                assert gd.dec.prefill(queue, ids[pos0:], pos0)
                got[mode] = _hidden(gd, cfg["hidden"])
                assert gd.dec.read(queue)[0] == pos0 + rows
            assert np.all(np.isfinite(got[0]))
            rel = np.linalg.norm(got[0] - got[1]) / np.linalg.norm(got[1])
            print(f"{name}: {rows} rows at {pos0}: rel {rel:.2e}", flush=True)
            assert rel <= 2e-3
    finally:
        L.mi_stream_set_modes(queue.handle, -1, -1)
        gd.close()


def test_prompt_attention_ignores_what_lies_behind_the_prompt():
    """Cache rows past the prompt's last position hold whatever an earlier, longer prompt left there: the result is
    the one a fresh cache gives, bit for bit."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    cfg = _cfg(6, 2, 64, 256)
    ids = [int(t) for t in np.random.default_rng(5).integers(0, cfg["vocab"], 256)]
    first = None
    for before in (0, 256):
        gd = GpuDecoder(Model(cfg, seed=78), queue)
        try:
            if before:
                assert gd.dec.prefill(queue, ids[::-1])
            assert gd.dec.prefill(queue, ids[:37])
            h = _hidden(gd, cfg["hidden"])
        finally:
            gd.close()
        if first is None:
            first = h
    assert np.array_equal(first, h)
