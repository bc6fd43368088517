"""mi_linear_batch gives what n calls of mi_linear give: calls share a launch only when none of them writes what
another one reads (x, weights, scales) or writes.  The rule (csrc/batch_rule.h) is checked on the CPU against sets of
bytes, and through the library on the GPU with calls whose weights or scales are another call's output."""
import ctypes
import itertools
import os
import shutil
import subprocess

import numpy as np
import pytest

from helpers import ROOT, mil

DRIVER = """
#include "batch_rule.h"
extern "C" int independent(const long* a, const long* b) {
    auto c = [](const long* v) {
        auto p = [&](int i) { return reinterpret_cast<const void*>(v[i]); };
        return mi::call_memory(static_cast<int>(v[0]), static_cast<int>(v[1]), static_cast<int>(v[2]), static_cast<int>(v[3]),
                               p(4), p(5), p(6), p(7));
    };
    return mi::independent(c(a), c(b)) && !mi::writes_what_reads(c(a), c(a)) && !mi::writes_what_reads(c(b), c(b));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_rule_against_byte_sets(tmp_path):
    src, so = tmp_path / "rule.cpp", str(tmp_path / "rule.so")
    src.write_text(DRIVER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "adreno-llms_amd", "csrc"),
                           "-o", so, str(src)])
    rule = ctypes.CDLL(so).independent
    seen = set()
    for kind, m, n, k in itertools.product((0, 4, 8), (1, 3), (2, 5), (32, 64)):
        sizes = dict(x=2 * m * k, W={0: 2 * n * k, 4: n * k // 2, 8: n * k}[kind],
                     scale={0: 0, 4: 2 * n * (k // 32), 8: 2 * n}[kind], out=2 * m * n)
        # x shared; the other operands far apart, except that one of call b lies against one of call a: byte for
        # byte the same start, one byte of overlap at either end, or touching without a shared byte
        for ours, theirs in itertools.product(("x", "W", "scale", "out"), repeat=2):
            for shift in (0, sizes[theirs] - 1, sizes[theirs], 1 - sizes[ours], -sizes[ours]):
                a = {name: 1 << 20 | i << 16 for i, name in enumerate(sizes)}
                b = {name: 1 << 24 | i << 16 for i, name in enumerate(sizes)}
                if not sizes["scale"]:
                    a["scale"] = b["scale"] = 0
                b["x"] = a["x"]
                if not sizes[ours] or not sizes[theirs]:
                    continue
                b[ours] = a[theirs] + shift
                span = lambda c, name: set(range(c[name], c[name] + sizes[name]))  # noqa: E731
                reads = lambda c: span(c, "x") | span(c, "W") | span(c, "scale")  # noqa: E731
                want = not any(span(w, "out") & reads(r) for w in (a, b) for r in (a, b)) and not span(a, "out") & span(b, "out")
                pack = lambda c: (ctypes.c_long * 8)(kind, m, n, k, c["x"], c["W"], c["scale"], c["out"])  # noqa: E731
                assert bool(rule(pack(a), pack(b))) == want, (kind, m, n, k, ours, theirs, shift)
                assert bool(rule(pack(b), pack(a))) == want, (kind, m, n, k, ours, theirs, shift)
                seen.add((ours, theirs, want))
    assert ("W", "out", False) in seen and ("out", "W", False) in seen and ("out", "scale", False) in seen


def _weight(kind, seed, n, k):
    w = mil.synth_normal_f16(seed, 0.05, (n, k))
    if kind == "f16":
        return w, None
    return mil.quantize_int8(w) if kind == "int8" else mil.quantize_q4(w)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["f16", "int8", "q4"])
@pytest.mark.parametrize("rows", [1, 4, 16, 40, 128])
def test_an_output_as_weights_or_scales_of_a_neighbour(kind, rows):
    """Two calls of one x: the second one's weights (or scales) are the first one's output, or the second one's output
    overwrites the first one's weights (or scales).  Same bytes as one call after the other."""
    assert mil.lib().mi_init(0) == 1
    queue, k = mil.Queue(), 128
    register = {"int8": mil.nnopt_register_int8_weight, "q4": mil.nnopt_register_q4_weight}.get(kind)
    for what, later_reads in itertools.product(("W", "scale") if register else ("W",), (True, False)):
        n = 128
        got = []
        for together in (False, True):
            x = mil.Buffer.from_host(mil.synth_normal_f16(3, 1.0, (rows, k)))
            (w1, s1), (w2, s2) = _weight(kind, 4, n, k), _weight(kind, 5, n, k)
            W1, W2, y, z = mil.Buffer.from_host(w1), mil.Buffer.from_host(w2), mil.Buffer(2 * rows * n), mil.Buffer(2 * rows * n)
            S1, S2 = (mil.Buffer.from_host(s1), mil.Buffer.from_host(s2)) if register else (None, None)
            # the shared region holds the output of one call and the weights or scales of the other
            size = {"W": w1.nbytes, "scale": s1.nbytes if register else 0}[what]
            region = mil.Buffer(max(2 * rows * n, size))
            init = np.zeros(max(2 * rows * n, size), np.uint8)
            init[:size] = (w1 if what == "W" else s1).view(np.uint8).ravel()
            assert mil.lib().mi_memcpy_h2d(region.ptr, init.ctypes.data, init.nbytes, queue.handle)
            queue.finish()
            if what == "W":
                shared_w, shared_s = region, S1
            else:
                shared_w, shared_s = W1, region
            if register:
                assert register(shared_w, shared_s, n, k) and register(W2, S2, n, k)
            reader, writer = (rows, n, k, x, shared_w, y), (rows, n, k, x, W2, region)
            plan = [writer, reader] if later_reads else [reader, writer]
            if together:
                assert mil.linear_batch(queue, mil.make_calls(plan)) == 2
            else:
                for c in plan:
                    assert mil.pytorch_linear(queue, *c)
            queue.finish()
            got.append((y.read(np.uint16, (rows, n)), region.read(np.uint16, (rows, n))))
            if register:
                assert mil.nnopt_unregister_weight(shared_w) and mil.nnopt_unregister_weight(W2)
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]), (what, later_reads)
