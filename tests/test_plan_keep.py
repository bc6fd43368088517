"""The GEMM plans that a thread keeps (csrc/plan_keep.h): one is given again for all the numbers that it follows from and for
no others, among them the CUs of the device, which change where mi_init is called for another one; keys that share a slot
push one another out; a thread's plans are its own."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

from helpers import ROOT

DRIVER = """
#include "plan_keep.h"
#include <thread>
static long made = 0;
static long plan_of(const int* v) {                      // a plan that tells what it was made from
    long p = 1;
    for (int i = 0; i < 7; ++i) p = p * 1000003 + v[i];
    return p;
}
// returns whether the plan is that of v; *again: it was kept
extern "C" int ask(const int* v, int* again) {
    const long before = made;
    const long got = mi::kept_plan<long>(mi::PlanKey{v[0], v[1], v[2], v[3], v[4], v[5], static_cast<size_t>(v[6])},
                                         [&] { ++made; return plan_of(v); });
    *again = made == before;
    return got == plan_of(v);
}
extern "C" int ask_in_a_thread(const int* v, int* again) {
    int ok = 0;
    std::thread([&] { ok = ask(v, again); }).join();
    return ok;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_a_plan_for_all_it_follows_from(tmp_path):
    src, so = tmp_path / "keep.cpp", str(tmp_path / "keep.so")
    src.write_text(DRIVER)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "adreno-llms_amd", "csrc"),
                           "-o", so, str(src), "-lpthread"])
    lib = ctypes.CDLL(so)

    def ask(v, f=lib.ask):
        again = ctypes.c_int()
        assert f((ctypes.c_int * 7)(*v), ctypes.byref(again)), v
        return bool(again.value)

    base = [0, 256, 8, 300, 1152, 896, 16 << 20]         # mode, CUs, kind, M, N, K, bytes of workspace
    assert not ask(base) and ask(base)
    for i, other in enumerate([4, 32, 4, 301, 1153, 960, 0]):
        v = list(base)
        v[i] = other
        assert not ask(v), i                             # another plan for every number that differs
        assert ask(v) and (not ask(base) or ask(base))
    assert ask(base) or ask(base)
    assert not ask(base, lib.ask_in_a_thread) and ask(base)
    rng = random.Random(2)
    keys = [[rng.choice([0, 4, 6]), rng.choice([256, 64]), rng.choice([0, 4, 8]), rng.randint(2, 2048), 64 * rng.randint(1, 80),
             64 * rng.randint(1, 80), rng.choice([0, 16 << 20])] for _ in range(200)]
    for _ in range(3000):
        ask(rng.choice(keys))
