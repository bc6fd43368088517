"""The prompt attention kernel (mi::launch_attention_prompt) by itself: every row, head and element of its output
against a softmax in fp64, at scores that span tens of nats and with rows that are not finite.

Bound per element, with P the exact probabilities, o the exact output and T = sum_k P_k |v_k - o|: a probability is
rounded to fp16 once (2^-11 of itself, 2^-24 of the largest below fp16's normal range; numerator and denominator
take the same rounded ones, so an error of P_k moves the output by P_k (v_k - o)), a score in nats is off by the fp32
sum over the head and the fp32 product behind it (2^-20 of the sum of its terms' magnitudes), sums and the division
are fp32 (2^-20), and the output is rounded to fp16 (2^-11 of it, 2^-25 below the normal range)."""
import ctypes

import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

# (head width, heads, key/value heads, rows, first position): every form of the launch, the number of heads per group
# the supported models have, rows and positions around the 16 queries of a set and the 64 keys of a tile
SHAPES = [
    (64, 4, 2, 2, 0), (64, 9, 3, 17, 0), (64, 15, 5, 130, 63), (64, 14, 2, 300, 212),       # up to 512 keys
    (64, 7, 1, 40, 560), (64, 9, 3, 65, 1000), (64, 14, 2, 301, 900),                        # more
    (64, 14, 2, 870, 0), (64, 16, 2, 800, 131), (64, 14, 2, 1200, 0),                        # blocks for the chip, more than a CU each
    (128, 4, 2, 17, 1), (128, 8, 2, 200, 330), (128, 16, 4, 1030, 0), (128, 16, 4, 1040, 28),
]


def _launch(queue, q, k, v, pos0, n_heads, n_kv):
    f = mil.lib()["_ZN2mi23launch_attention_promptEP12ihipStream_tPKtS3_S3_Ptiiiiif"]
    f.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int] * 5 + [ctypes.c_float]
    f.restype = ctypes.c_bool
    rows, qd = q.shape
    d = qd // n_heads
    assert d in (64, 128) and k.shape == v.shape == (pos0 + rows, n_kv * d) and n_heads % n_kv == 0
    # behind the last key, and around the output, what must not be used
    behind = np.full((70, n_kv * d), np.nan, np.float16)
    dev = [mil.Buffer.from_host(a) for a in (q, np.concatenate([k, behind]), np.concatenate([v, behind]))]
    out = mil.Buffer.from_host(np.full(rows * qd + 64, 0x7bff, np.uint16))
    print(f"head width {d}, {n_heads} heads over {n_kv}, {rows} rows at {pos0}", flush=True)
    assert f(queue.handle, dev[0].ptr, dev[1].ptr, dev[2].ptr, out.ptr, rows, pos0, n_heads, n_kv, d, 1.0 / np.sqrt(d))
    queue.finish()
    got = out.read(np.float16, (rows * qd + 64,))
    assert np.all(got[-64:].view(np.uint16) == 0x7bff)
    return got[:-64].reshape(rows, n_heads, d)


def _exact(q, k, v, pos0, n_heads, n_kv, head):
    """One head in fp64: outputs and the bound above.  Values that are not finite reach the rows that see them only."""
    rows, d = q.shape[0], q.shape[1] // n_heads
    g = head // (n_heads // n_kv)
    qh = q[:, head * d:(head + 1) * d].astype(np.float64)
    kh, vh = k[:, g * d:(g + 1) * d].astype(np.float64), v[:, g * d:(g + 1) * d].astype(np.float64)
    unseen = np.arange(len(k))[None, :] > pos0 + np.arange(rows)[:, None]
    with np.errstate(invalid="ignore"):
        s = qh @ kh.T / np.sqrt(d)
    s[unseen] = -np.inf
    size = np.where(unseen, 0.0, np.abs(np.nan_to_num(qh, posinf=0, neginf=0)) @ np.abs(np.nan_to_num(kh, posinf=0, neginf=0)).T) / np.sqrt(d)
    with np.errstate(invalid="ignore"):
        p = np.exp(s - np.max(s, axis=1, keepdims=True))         # NaN where a row has no weight at all
        p /= np.sum(p, axis=1, keepdims=True)
    p[np.all(s == -np.inf, axis=1)] = 0.0                    # no key at all: the reference's sum + 1e-20 makes that 0
    fin = np.where(np.isfinite(vh), vh, 0.0)
    o = p @ fin
    t = p @ np.abs(fin) + np.abs(o)                          # >= sum P |v - o|
    bound = (2.0 ** -11 + 2.0 ** -20 * np.max(size, axis=1, keepdims=True) + 2.0 ** -20) * t
    bound += 2.0 ** -24 * len(k) * (np.max(np.abs(fin)) + np.abs(o)) * np.max(p, axis=1, keepdims=True)
    bound += 2.0 ** -11 * np.abs(o) + 2.0 ** -25
    for key, e in zip(*np.nonzero(~np.isfinite(vh))):
        seen = ~unseen[:, key]
        with np.errstate(invalid="ignore"):
            o[seen, e] += p[seen, key] * vh[key, e]
    return o, bound


def _compare(got, q, k, v, pos0, n_heads, n_kv):
    worst = 0.0
    for head in range(n_heads):
        want, bound = _exact(q, k, v, pos0, n_heads, n_kv, head)
        g = got[:, head].astype(np.float64)
        bad = ~np.isfinite(want)
        assert np.array_equal(np.isnan(g), np.isnan(want)) and np.array_equal(g[np.isinf(g)], want[np.isinf(want)])
        with np.errstate(invalid="ignore"):
            share = np.where(bad, 0.0, np.abs(g - want) / bound)
        worst = max(worst, float(np.max(share)))
        assert np.all(share <= 1.0), (head, np.unravel_index(np.argmax(share), share.shape), float(np.max(share)))
    print(f"  largest error {worst:.2f} of the bound", flush=True)


def _operands(rng, d, n_heads, n_kv, rows, pos0, nats):
    """q, k, v with scores of about nats[key] for every query (and N(0, 1) about that)."""
    keys = pos0 + rows
    sign = np.where(rng.random(d) < 0.5, -1.0, 1.0)
    q = rng.standard_normal((rows, n_heads, d)) + 2.0 * sign
    k = rng.standard_normal((keys, n_kv, d)) * 0.4 + (nats / (2.0 * np.sqrt(d)))[:, None, None] * sign
    v = rng.standard_normal((keys, n_kv, d)) + 0.5
    return [a.reshape(len(a), -1).astype(np.float16) for a in (q, k, v)]


NATS = {
    "even": lambda j: np.zeros(len(j)),
    "first_tile": lambda j: np.where(j < 64, 25.0, 0.0) * (j % 5 == 0),
    "last_keys": lambda j: np.where(j >= len(j) - 20, 30.0, -10.0),
    "rising": lambda j: 7.0 * (j // 64),                     # by more than the kernel's slack from tile to tile
    "rising_fast": lambda j: 11.0 * np.sqrt(j),
    "falling": lambda j: -7.0 * (j // 64),
    "every_other_tile": lambda j: np.where(j // 64 % 2 == 0, -20.0, 20.0),
    "fourth_tile": lambda j: np.where(j // 64 % 4 == 3, 15.0, -15.0) + 0.05 * j,
}


@pytest.mark.parametrize("nats", list(NATS))
@pytest.mark.parametrize("d,n_heads,n_kv,rows,pos0", SHAPES)
def test_every_row(d, n_heads, n_kv, rows, pos0, nats):
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    rng = np.random.default_rng(rows + 7 * pos0 + d)
    q, k, v = _operands(rng, d, n_heads, n_kv, rows, pos0, NATS[nats](np.arange(pos0 + rows)))
    got = _launch(queue, q, k, v, pos0, n_heads, n_kv)
    assert np.array_equal(got.view(np.uint16), _launch(queue, q, k, v, pos0, n_heads, n_kv).view(np.uint16))
    _compare(got, q, k, v, pos0, n_heads, n_kv)


@pytest.mark.parametrize("d,n_heads,n_kv,rows,pos0", SHAPES)
def test_values_that_are_not_finite_stay_behind_the_mask(d, n_heads, n_kv, rows, pos0):
    """Infinities and NaN in the values (and NaN in a key) reach the rows that see the position and no earlier one."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    rng = np.random.default_rng(rows + pos0)
    q, k, v = _operands(rng, d, n_heads, n_kv, rows, pos0, np.zeros(pos0 + rows))
    last = pos0 + rows - 1
    for i, (back, what) in enumerate([(0, np.inf), (1, -np.inf), (5, np.nan), (17, np.inf), (40, np.inf), (40, -np.inf), (90, np.nan)]):
        if back < rows:                                      # (some of the rows do not see it)
            v[last - back, (11 * i) % (n_kv * d)] = what
    k[last - min(3, rows - 1), d * (n_kv - 1)] = np.nan
    _compare(_launch(queue, q, k, v, pos0, n_heads, n_kv), q, k, v, pos0, n_heads, n_kv)


@pytest.mark.parametrize("d,n_heads,n_kv,rows,pos0", SHAPES)
def test_scores_of_minus_infinity(d, n_heads, n_kv, rows, pos0):
    """Every other key has a score of -inf, or every key of the first tiles, or every key: no weight, and where no key
    has any the output is 0 (QW/kernels/attention.cl gqa_softmax divides by the sum + 1e-20)."""
    assert mil.lib().mi_init(0) == 1
    queue = mil.Queue()
    rng = np.random.default_rng(rows + pos0)
    keys = np.arange(pos0 + rows)
    for what in (keys % 2 == 0, keys < 150, keys >= 0):
        q, k, v = _operands(rng, d, n_heads, n_kv, rows, pos0, np.zeros(pos0 + rows))
        for head in range(n_heads):
            q[:, head * d] = np.abs(q[:, head * d]) + np.float16(0.5)
        for head in range(n_kv):
            k[what, head * d] = -np.inf
        _compare(_launch(queue, q, k, v, pos0, n_heads, n_kv), q, k, v, pos0, n_heads, n_kv)
