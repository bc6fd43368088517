"""Runs the projections of a layer, and of a whole model, as batches of independent calls (mi_linear_batch), stream launches: the
program behind profiles/batch_kernel_trace.txt.  Arguments: the weight kind (f16, int8, q4), rows of x, layers, hidden and
intermediate width, width of k and v."""
import importlib, os, sys

import numpy as np
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
mil = importlib.import_module("adreno-llms_amd")
assert mil.lib().mi_init(0) == 1
queue = mil.Queue()
kind, (rows, layers, hidden, inter, kv) = sys.argv[1], map(int, sys.argv[2:7])
host, keep = {}, []


def weight(n, k):
    if (n, k) not in host:
        w = mil.synth_normal_f16(n + k, 0.02, (n, k))
        host[n, k] = (w,) if kind == "f16" else mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)
    bufs = [mil.Buffer.from_host(a) for a in host[n, k]]
    keep.extend(bufs)
    if kind != "f16":
        register = mil.nnopt_register_int8_weight if kind == "int8" else mil.nnopt_register_q4_weight
        assert register(*bufs, n, k)
    return bufs[0]


calls = []
for layer in range(layers):
    for widths, k in (((hidden, kv, kv), hidden), ((hidden,), hidden), ((inter, inter), hidden), ((hidden,), inter)):
        x = mil.Buffer.from_host(mil.synth_normal_f16(layer + k, 1.0, (rows, k)))
        keep.append(x)
        for n in widths:
            out = mil.Buffer(2 * rows * n)
            keep.append(out)
            calls.append((rows, n, k, x, weight(n, k), out))
batch = mil.make_calls(calls)
for _ in range(50):
    assert mil.linear_batch(queue, batch) == len(batch)
queue.finish()
print("done", len(batch), "calls", flush=True)
