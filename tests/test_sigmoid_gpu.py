"""The SwiGLU's sigmoid on the device is a reciprocal and a Newton step where the oracle divides: for every value that an
fp16 gate can hold, and factors from 0 to infinity that would show a sigmoid off by its last bit or not 0 (or not 1)
where the oracle's is, fp16((gate * sigmoid(gate)) * product) has the oracle's bits."""
import numpy as np
import pytest

import oracle_lib as O
from helpers import mil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("product", [1.0, -3.5, 0.33325, 65504.0, 6e-8, 0.0, float("inf"), float("-inf")])
def test_every_gate(product):
    assert mil.lib().mi_init(0) == 1
    queue, n, k = mil.Queue(), 65536, 64
    gate = np.arange(n, dtype=np.uint32).astype(np.uint16)
    w, x = np.zeros((n, k), np.float16), np.zeros(k, np.float16)
    w[:, 0], x[0] = 1.0, product
    want = gate.copy()
    O.lib.orc_gemv_f16_silu_gate(O.u16(x), O.u16(w), want, n, k)
    xb, wb, gb = (mil.Buffer.from_host(a) for a in (x, w, gate))
    assert mil.pytorch_linear_silu_gate_fused(queue, n, k, xb, wb, gb)
    queue.finish()
    got = gb.read(np.uint16, (n,))
    nan = np.isnan(want.view(np.float16))
    assert np.array_equal(np.isnan(got.view(np.float16)), nan)
    assert np.array_equal(got[~nan], want[~nan]), gate[~nan][got[~nan] != want[~nan]].view(np.float16)
