"""The sum of the exponentials at a long context, which a wavefront's lanes share: a step must equal the prompt's
reference-order attention bit for bit (mode 1: other kernels, one chain of additions).  Score spreads from nearly equal
exponentials (halves of the last place come up at every binade) over a few that carry the sum to one that is all of it,
positions around the line from which the sum is shared, around whole and ragged runs per lane, and the longest context."""
import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

HIDDEN, INTER, HEADS, KV, WIDTH, VOCAB, MOST = 128, 128, 4, 2, 64, 256, 8192


def _decoder(sigma, keep):
    seed = iter(range(1, 1000))
    up = lambda a: keep.append(mil.Buffer.from_host(np.ascontiguousarray(a))) or keep[-1]  # noqa: E731
    mat = lambda n, k, s: up(mil.synth_normal_f16(next(seed), s, (n, k)))  # noqa: E731
    vec = lambda n, mean=0.0: up((mil.synth_normal_f16(next(seed), 0.05, (n,)).astype(np.float32) + mean).astype(np.float16))  # noqa: E731
    q, kv = HEADS * WIDTH, KV * WIDTH
    bufs = dict(embed=mat(VOCAB, HIDDEN, 1.0), final_norm=vec(HIDDEN, 1.0), lm_head=mat(VOCAB, HIDDEN, 0.1), in_norm=[vec(HIDDEN, 1.0)],
                post_norm=[vec(HIDDEN, 1.0)], bq=[vec(q)], bk=[vec(kv)], bv=[vec(kv)], wq=[mat(q, HIDDEN, sigma)], wk=[mat(kv, HIDDEN, sigma)],
                wv=[mat(kv, HIDDEN, 0.1)], wo=[mat(HIDDEN, q, 0.1)], wgate=[mat(INTER, HIDDEN, 0.1)], wup=[mat(INTER, HIDDEN, 0.1)],
                wdown=[mat(HIDDEN, INTER, 0.1)])
    cfg = dict(hidden=HIDDEN, inter=INTER, n_heads=HEADS, n_kv_heads=KV, head_dim=WIDTH, n_layers=1, vocab=VOCAB, max_pos=MOST,
               rms_eps=1e-6, rope_theta=10000.0)
    return mil.Decoder(cfg, bufs)


@pytest.mark.parametrize("sigma", [0.0, 1e-3, 0.02, 0.1, 0.3, 2.0])
def test_steps_equal_the_prompt(sigma):
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    dec = _decoder(sigma, keep)
    ids = [int(t) for t in np.random.default_rng(5).integers(0, VOCAB, MOST)]
    logits = lambda: np.empty(VOCAB, np.uint16)  # noqa: E731
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 1)
    for pos in (800, 895, 896, 927, 928, 1000, 1023, 1024, 1500, 1901, 2047, 2048, 2100, 3333, 4095, 8191):
        print(f"sigma {sigma} position {pos}", flush=True)
        got, want = logits(), logits()
        assert dec.prefill(queue, ids[:pos + 1])
        first = dec.read(queue)
        assert mil.lib().mi_memcpy_d2h(want.ctypes.data, dec.logits_ptr, 2 * VOCAB, queue.handle)
        queue.finish()
        assert dec.reset(queue, pos, ids[pos]) and dec.step(queue)
        assert dec.read(queue) == first
        assert mil.lib().mi_memcpy_d2h(got.ctypes.data, dec.logits_ptr, 2 * VOCAB, queue.handle)
        queue.finish()
        assert np.array_equal(got, want), pos


@pytest.mark.parametrize("sigma", [0.0, 0.02, 0.3])
def test_steps_equal_the_prompt_where_a_lane_holds_more_quadruples(sigma):
    """9 of them to 2304 positions, 17 beyond."""
    assert mil.lib().mi_init(0) == 1
    queue, keep = mil.Queue(), []
    dec = _decoder(sigma, keep)
    ids = [int(t) for t in np.random.default_rng(6).integers(0, VOCAB, MOST)]
    assert mil.lib().mi_stream_set_modes(queue.handle, -1, 1)
    for pos in (2051, 2176, 2271, 2287, 2303, 2304, 2320, 2560):
        print(f"sigma {sigma} position {pos}", flush=True)
        got, want = np.empty(VOCAB, np.uint16), np.empty(VOCAB, np.uint16)
        assert dec.prefill(queue, ids[:pos + 1])
        first = dec.read(queue)
        assert mil.lib().mi_memcpy_d2h(want.ctypes.data, dec.logits_ptr, 2 * VOCAB, queue.handle)
        queue.finish()
        assert dec.reset(queue, pos, ids[pos]) and dec.step(queue)
        assert dec.read(queue) == first
        assert mil.lib().mi_memcpy_d2h(got.ctypes.data, dec.logits_ptr, 2 * VOCAB, queue.handle)
        queue.finish()
        assert np.array_equal(got, want), pos
