"""Calls of a batch that share no x: independent GEMVs of any K and N go out as one launch (launch_gemv_many), and
every output is bit for bit what the same call gives by itself.  Widths around the row batches and blocks, every K the
launch has an instance for with one that it has none for between them, more calls than a launch holds, several rows of x;
then batches whose calls read, overwrite and re-read one another's buffers, which have to come out as in order."""
import random

import numpy as np
import pytest

from helpers import mil

pytestmark = pytest.mark.gpu

KS = (576, 896, 960, 1024, 1536, 2048, 2560, 4608, 4864)
GUARD = 8


def _weight(kind, n, k, seed, keep):
    w = mil.synth_normal_f16(seed, 0.02, (n, k))
    if kind == "f16":
        keep.append(mil.Buffer.from_host(w))
        return keep[-1]
    q, s = mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)
    qb, sb = mil.Buffer.from_host(q), mil.Buffer.from_host(s)
    keep += [qb, sb]
    assert (mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight)(qb, sb, n, k)
    return qb


def _blank(count):
    return mil.Buffer.from_host(np.full(count + GUARD, 0x7bff, np.uint16))


@pytest.mark.parametrize("kind,gemv_mode", [("f16", 1), ("int8", 1), ("q4", 0), ("q4", 1)])
@pytest.mark.parametrize("rows", [1, 3, 15])
def test_runs_of_different_x_and_k(kind, gemv_mode, rows):
    assert mil.lib().mi_init(0) == 1
    queue, keep, rng = mil.Queue(), [], random.Random(rows)
    runs = []                                                   # [(calls without out)], one x and K each
    for j, k in enumerate(KS + (1152,) + KS + KS[::-1]):
        x = mil.Buffer.from_host(mil.synth_normal_f16(50 + j, 1.0, (rows, k)))
        keep.append(x)
        widths = [(4097,), (1, 3), (255, 64, 257), (896,), (15, 17, 16, 128)][j % 5] if k == KS[j % len(KS)] else (rng.choice((1, 5, 128, 577)),)
        runs.append([(rows, n, k, x, _weight(kind, n, k, 1000 + 8 * j + t, keep)) for t, n in enumerate(widths)])
    assert sum(map(len, runs)) > 2 and max(map(len, runs)) <= 4
    assert mil.lib().mi_stream_set_modes(queue.handle, gemv_mode, 1)      # rows of GEMV whatever their number
    want = [[_blank(c[0] * c[1]) for c in run] for run in runs]
    got = [[_blank(c[0] * c[1]) for c in run] for run in runs]
    for run, outs in zip(runs, want):                            # a run is one launch by itself
        assert mil.linear_batch(queue, mil.make_calls([(*c, o) for c, o in zip(run, outs)])) == len(run)
        queue.finish()
    flat = [(*c, o) for run, outs in zip(runs, got) for c, o in zip(run, outs)]
    print(f"{kind} mode {gemv_mode} rows {rows}: {len(flat)} calls", flush=True)
    assert mil.linear_batch(queue, mil.make_calls(flat)) == len(flat)
    queue.finish()
    for run, a, b in zip(runs, want, got):
        for c, p, q in zip(run, a, b):
            shape = (c[0] * c[1] + GUARD,)
            p, q = p.read(np.uint16, shape), q.read(np.uint16, shape)
            assert np.array_equal(p, q) and (q[-GUARD:] == 0x7bff).all(), (kind, c[:3])


@pytest.mark.parametrize("count", [64, 65, 130])
def test_more_calls_than_a_launch_holds(count):
    assert mil.lib().mi_init(0) == 1
    queue, keep, k = mil.Queue(), [], 576
    calls = [(1, 1 + j % 7, k, mil.Buffer.from_host(mil.synth_normal_f16(j, 1.0, (1, k))), _weight("int8", 1 + j % 7, k, 300 + j, keep))
             for j in range(count)]
    want, got = [[_blank(c[1]) for c in calls] for _ in range(2)]
    for c, o in zip(calls, want):
        assert mil.pytorch_linear(queue, *c, o)
    assert mil.linear_batch(queue, mil.make_calls([(*c, o) for c, o in zip(calls, got)])) == count
    queue.finish()
    for c, p, q in zip(calls, want, got):
        assert np.array_equal(p.read(np.uint16, (c[1] + GUARD,)), q.read(np.uint16, (c[1] + GUARD,))), c[:3]


@pytest.mark.parametrize("seed", range(12))
def test_calls_that_share_buffers_keep_their_order(seed):
    """Activations from a pool of four buffers: a call may read what an earlier one wrote, overwrite what an earlier one
    reads, write what an earlier one wrote, or have nothing to do with it."""
    assert mil.lib().mi_init(0) == 1
    rng, keep, k, rows = random.Random(seed), [], 576, 1 + seed % 2
    ws = [_weight("int8", k, k, 7 + j, keep) for j in range(3)]
    plan = [(rng.randrange(4), rng.randrange(3), rng.randrange(4)) for _ in range(rng.randrange(3, 20))]
    plan = [(a, w, b) for a, w, b in plan if a != b]
    start = [mil.synth_normal_f16(90 + j, 1.0, (rows, k)) for j in range(4)]
    queue, end = mil.Queue(), []
    for together in (False, True):
        pool = [mil.Buffer.from_host(s) for s in start]
        calls = [(rows, k, k, pool[a], ws[w], pool[b]) for a, w, b in plan]
        if together:
            assert mil.linear_batch(queue, mil.make_calls(calls)) == len(calls)
        else:
            for c in calls:
                assert mil.pytorch_linear(queue, *c)
        queue.finish()
        end.append([p.read(np.uint16, (rows, k)) for p in pool])
    assert all(np.array_equal(p, q) for p, q in zip(*end)), plan


def test_a_refused_call_ends_the_batch_there():
    assert mil.lib().mi_init(0) == 1
    queue, keep, k = mil.Queue(), [], 576
    xs = [mil.Buffer.from_host(mil.synth_normal_f16(j, 1.0, (1, k))) for j in range(4)]
    ws = [_weight("int8", 64, k, 7 + j, keep) for j in range(4)]
    outs, want = [_blank(64) for _ in range(4)], [_blank(64) for _ in range(2)]
    calls = [(1, 64, k, x, w, o) for x, w, o in zip(xs, ws, outs)]
    calls[2] = (1, 63, k, xs[2], ws[2], outs[2])                 # registered with 64 rows
    assert mil.linear_batch(queue, mil.make_calls(calls)) == 2
    for x, w, o in zip(xs, ws, want):
        assert mil.pytorch_linear(queue, 1, 64, k, x, w, o)
    queue.finish()
    for o, p in zip(outs, want):
        assert np.array_equal(o.read(np.uint16, (64 + GUARD,)), p.read(np.uint16, (64 + GUARD,)))
    for o in outs[2:]:
        assert (o.read(np.uint16, (64 + GUARD,)) == 0x7bff).all()
