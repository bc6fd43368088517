"""The launch that adds a prompt's q | k | v slices, adds the biases, rotates q and k and fills the cache rows, bit for
bit against the projection and the rotary launch by themselves.  Every row of every matrix has one weight that is not
zero, so that a sum is the same in any order and any number of slices: a prompt in slices of K and the same prompt in
one piece (mode 3) then leave the same residual stream, logits and cache rows (the steps behind the prompt read them).
Heads of 24, 64 and 128 values, biases, a prompt behind another one."""
import numpy as np
import pytest

from helpers import mil
from test_prefill_slices_gpu import _outputs

pytestmark = pytest.mark.gpu

VOCAB, LAYERS = 512, 2                           # (as in _outputs)


def _selecting_decoder(kind, hidden, inter, heads, kv, width):
    rng, keep = np.random.default_rng(3), []
    up = lambda a: keep.append(mil.Buffer.from_host(np.ascontiguousarray(a))) or keep[-1]  # noqa: E731

    def weight(n, k):
        at = rng.integers(0, k, n)
        if kind == "f16":
            w = np.zeros((n, k), np.float16)
            w[np.arange(n), at] = rng.uniform(0.5, 1.5, n) * rng.choice([-1, 1], n)
            return up(w)
        if kind == "int8":
            q, s = np.zeros((n, k), np.int8), rng.uniform(0.008, 0.015, n).astype(np.float16)
            q[np.arange(n), at] = rng.integers(40, 128, n) * rng.choice([-1, 1], n)
            register = mil.nnopt_register_int8_weight
        else:
            v, s = np.full((n, k), 8, np.uint8), rng.uniform(0.1, 0.25, (n, k // 32)).astype(np.float16)
            v[np.arange(n), at] = rng.choice([0, 1, 2, 3, 13, 14, 15], n)
            q = v[:, 0::2] | v[:, 1::2] << 4
            register = mil.nnopt_register_q4_weight
        wb, sb = up(q), up(s)
        assert register(wb, sb, n, k)
        return wb

    vec = lambda n, mean=0.0: up((rng.normal(0, 0.3, n) + mean).astype(np.float16))  # noqa: E731
    qd, kvd, lay = heads * width, kv * width, range(LAYERS)
    bufs = dict(embed=up(rng.normal(0, 1, (VOCAB, hidden)).astype(np.float16)), final_norm=vec(hidden, 1.0), lm_head=weight(VOCAB, hidden),
                in_norm=[vec(hidden, 1.0) for _ in lay], post_norm=[vec(hidden, 1.0) for _ in lay], bq=[vec(qd) for _ in lay],
                bk=[vec(kvd) for _ in lay], bv=[vec(kvd) for _ in lay], wq=[weight(qd, hidden) for _ in lay],
                wk=[weight(kvd, hidden) for _ in lay], wv=[weight(kvd, hidden) for _ in lay], wo=[weight(hidden, qd) for _ in lay],
                wgate=[weight(inter, hidden) for _ in lay], wup=[weight(inter, hidden) for _ in lay],
                wdown=[weight(hidden, inter) for _ in lay])
    cfg = dict(hidden=hidden, inter=inter, n_heads=heads, n_kv_heads=kv, head_dim=width, n_layers=LAYERS, vocab=VOCAB, max_pos=256,
               rms_eps=1e-6, rope_theta=10000.0)
    return mil.Decoder(cfg, bufs), bufs, keep


@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("shape", [(896, 1024, 14, 2, 64), (384, 512, 16, 4, 24), (1024, 512, 8, 2, 128), (960, 512, 15, 5, 64)],
                         ids=lambda s: f"{s[0]}x{s[4]}")
@pytest.mark.parametrize("rows,pos0,slices", [(2, 0, 2), (33, 0, 3), (70, 31, 2)])
def test_rotary_and_cache_rows_bit_for_bit(kind, shape, rows, pos0, slices):
    assert mil.lib().mi_init(0) == 1
    queue, ids, got = mil.Queue(), [(29 * t + 3) % VOCAB for t in range(pos0 + rows)], []
    hidden, qkv = shape[0], (shape[2] + 2 * shape[3]) * shape[4]
    dec, bufs, keep = _selecting_decoder(kind, *shape)
    for mode in (3, 100 * slices + 11):
        assert mil.lib().mi_stream_set_modes(queue.handle, 0, 1)
        if pos0:
            assert dec.prefill(queue, ids[:pos0])
        assert mil.lib().mi_stream_set_modes(queue.handle, 0, mode)
        print(f"{kind} {shape} rows {rows} at {pos0} mode {mode}", flush=True)
        assert mil.linear_plan(queue, rows, hidden, hidden, bufs["embed"], bufs["embed"])[2] == (1 if mode == 3 else slices)
        got.append(_outputs(queue, dec, hidden, ids[pos0:], pos0, 3))
    for j, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), j
