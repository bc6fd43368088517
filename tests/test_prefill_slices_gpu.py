"""Prompts whose projections are cut into slices of K: the launch that adds the slices also adds the residual and norms
the row (o and down projection), or adds the biases, rotates q and k and fills the cache rows (q | k | v).  The first is
held bit for bit to the separate launches, which run where a matrix's scales are not 8-byte aligned; both are held to
the rows of GEMV within the GEMM's tolerance.  Rows around the tiles, hidden widths with and without a part
of 256 columns left over, head widths 64 and 128, every weight kind."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

VOCAB, LAYERS = 512, 2


def _decoder(queue, kind, hidden, inter, heads, kv, width, off_scales):
    """off_scales: the scales of the o and down projections start 2 bytes behind a multiple of 8."""
    keep, seed = [], iter(range(1, 10_000))
    up = lambda a: keep.append(mil.Buffer.from_host(np.ascontiguousarray(a))) or keep[-1]  # noqa: E731

    def weight(n, k, off=False):
        w = mil.synth_normal_f16(next(seed), 0.03, (n, k))
        if kind == "f16":
            return up(w)
        q, s = mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)
        wb = up(q)
        flat = s.reshape(-1).view(np.uint16)
        sb = up(np.concatenate([np.zeros(1, np.uint16), flat]) if off else flat)
        reg = mil.lib().mi_register_int8_weight if kind == "int8" else mil.lib().mi_register_q4_weight
        assert reg(wb.ptr, sb.ptr + (2 if off else 0), n, k)
        return wb

    vec = lambda n, mean=0.0: up((mil.synth_normal_f16(next(seed), 0.05, (n,)).astype(np.float32) + mean).astype(np.float16))  # noqa: E731
    qd, kvd, lay = heads * width, kv * width, range(LAYERS)
    off = off_scales and kind == "int8"
    bufs = dict(embed=up(mil.synth_normal_f16(next(seed), 1.0, (VOCAB, hidden))), final_norm=vec(hidden, 1.0), lm_head=weight(VOCAB, hidden),
                in_norm=[vec(hidden, 1.0) for _ in lay], post_norm=[vec(hidden, 1.0) for _ in lay], bq=[vec(qd) for _ in lay],
                bk=[vec(kvd) for _ in lay], bv=[vec(kvd) for _ in lay], wq=[weight(qd, hidden) for _ in lay],
                wk=[weight(kvd, hidden) for _ in lay], wv=[weight(kvd, hidden) for _ in lay],
                wo=[weight(hidden, qd, off) for _ in lay], wgate=[weight(inter, hidden) for _ in lay],
                wup=[weight(inter, hidden) for _ in lay], wdown=[weight(hidden, inter, off) for _ in lay])
    cfg = dict(hidden=hidden, inter=inter, n_heads=heads, n_kv_heads=kv, head_dim=width, n_layers=LAYERS, vocab=VOCAB, max_pos=1024,
               rms_eps=1e-6, rope_theta=1000000.0)
    return mil.Decoder(cfg, bufs), bufs, keep


def _outputs(queue, dec, hidden, ids, pos0, steps):
    """The residual stream and logits behind the prompt and behind each of `steps` single-token steps on its cache rows."""
    assert dec.prefill(queue, ids, pos0)
    out = []
    for turn in range(steps + 1):
        if turn:
            assert dec.set_token(queue, 7 * turn) and dec.step(queue)
        queue.finish()
        for ptr, n in ((mil.lib().mi_decoder_buffer(dec.handle, 0), hidden), (dec.logits_ptr, VOCAB)):
            host = np.empty(n, np.uint16)
            assert mil.lib().mi_memcpy_d2h(host.ctypes.data, ptr, 2 * n, queue.handle)
            out.append(host)
    return out


SHAPES = [(896, 4864, 14, 2, 64), (576, 1536, 9, 3, 64), (1024, 2816, 8, 2, 128), (1920, 2048, 16, 4, 128)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("rows", [65, 66, 97])
@pytest.mark.parametrize("tile,slices", [(1, 2), (2, 3), (1, 4)])
def test_sums_residual_and_norm_bit_for_bit(shape, rows, tile, slices):
    """The number of slices pinned: left to itself the library may cut a projection for the one way and not for the other."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    hidden, inter = shape[:2]
    ids, got = [(37 * t) % VOCAB for t in range(rows)], []
    print(f"{shape} rows {rows} slices {slices}", flush=True)
    for off in (False, True):
        dec, bufs, keep = _decoder(queue, "int8", *shape, off)
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, 100 * slices + 10 + tile)
        assert mil.linear_plan(queue, rows, hidden, inter, bufs["wdown"][0], bufs["wdown"][0])[2] == slices
        got.append(_outputs(queue, dec, hidden, ids, 0, 2))
        assert mil.lib().mi_stream_set_modes(queue.handle, -1, -1)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: f"{s[0]}x{s[1]}")
@pytest.mark.parametrize("rows,pos0", [(65, 0), (200, 31)])
def test_within_tolerance_of_rows_of_gemv(kind, shape, rows, pos0):
    """Two layers: max-abs 1e-2 of the largest value and cosine 0.9999, as the other prompts on the matrix cores."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    ids, got = [(11 * t) % VOCAB for t in range(pos0 + rows)], []
    dec, bufs, keep = _decoder(queue, kind, *shape, False)
    for mode in (1, -1):
        assert mil.lib().mi_stream_set_modes(queue.handle, 0, 1)
        if pos0:
            assert dec.prefill(queue, ids[:pos0])
        assert mil.lib().mi_stream_set_modes(queue.handle, 0, mode)
        got.append(_outputs(queue, dec, shape[0], ids[pos0:], pos0, 1))
    print(f"{kind} {shape} rows {rows} at {pos0}", flush=True)
    for a, b in zip(*got):
        a, b = (v.view(np.float16).astype(np.float64) for v in (a, b))
        assert np.abs(a - b).max() <= 1e-2 * np.abs(a).max()
        assert a @ b >= 0.9999 * np.linalg.norm(a) * np.linalg.norm(b)
