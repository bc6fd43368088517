"""The launch that serves several GEMVs (csrc/deal_rule.h): every row batch of every call is computed by one wavefront and
no more, also where blocks are added to make their number a multiple of 8, and all blocks of all rows of x are resident at
once unless there is one per call.  The walk of the kernel, on the CPU."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

from helpers import ROOT

DRIVER = """
#include "deal_rule.h"
// taken: how often each row batch is computed, the calls' one behind the other; returns the blocks per row of x
extern "C" long deal(int n, const int* nbatch, const int* bytes, int M, long resident, int* taken) {
    constexpr int kWaves = 4;
    uint16_t first[64];
    int waves[64];
    const long blocks = mi::deal_blocks(n, nbatch, bytes, M, resident, kWaves, first, waves);
    for (int b = 0; b < blocks; ++b) {
        int i = 0, at = 0;
        while (i + 1 < n && b >= first[i + 1]) at += nbatch[i++];
        for (int w = 0; w < kWaves; ++w)
            for (int q = mi::first_batch(b, w, first[i], waves[i], kWaves); q >= 0 && q < nbatch[i]; q += waves[i]) ++taken[at + q];
    }
    return blocks;
}
"""

# rows of q | k | v, o, gate | up, down, and their K
LAYERS = {"135m": [(576, 576), (192, 576), (192, 576), (576, 576), (1536, 576), (1536, 576), (576, 1536)],
          "0.5b": [(896, 896), (128, 896), (128, 896), (896, 896), (4864, 896), (4864, 896), (896, 4864)]}


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_batch_once(tmp_path):
    src, so = tmp_path / "deal.cpp", str(tmp_path / "deal.so")
    src.write_text(DRIVER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "adreno-llms_amd", "csrc"),
                           "-o", so, str(src)])
    deal = ctypes.CDLL(so).deal
    deal.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_long, ctypes.c_void_p]
    deal.restype = ctypes.c_long
    rng, cases = random.Random(1), []
    for layer in LAYERS.values():
        for times in (1, 2, 9):
            for vl, half in ((1, 4), (2, 4), (4, 2), (4, 1)):                 # rows per batch, bytes of four values / 2
                cases.append([((n + vl - 1) // vl, vl * k * half // 2) for n, k in (layer * times)[:64]])
    for _ in range(60):
        cases.append([(rng.randint(1, 5000), rng.randint(100, 20000)) for _ in range(rng.randint(1, 64))])
    cases.append([(37984, 3584)])
    for case in cases:
        n = len(case)
        nbatch, size = ((ctypes.c_int * n)(*(c[j] for c in case)) for j in (0, 1))
        for m in (1, 2, 3, 5, 8, 15):
            taken = (ctypes.c_int * sum(nbatch))()
            blocks = deal(n, nbatch, size, m, 256 * 3 * 4, taken)
            assert set(taken) == {1}, (case, m, blocks)
            assert m == 1 or blocks % 8 == 0
            assert blocks * m <= 768 or blocks <= (n + 7) // 8 * 8, (case, m, blocks)
