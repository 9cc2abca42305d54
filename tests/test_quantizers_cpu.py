"""The host quantizers' wide paths against the oracle's plain loops, bit for bit, where they can go wrong: remainders of the
32 values taken at once, ties of the maximum, rows of zeros, tiny and infinite values."""
import numpy as np
import pytest

from mongoose_amd import engine as E
from oracle import binding as ob


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("cols", [1, 31, 32, 33, 64, 95, 896])
def test_q8_rows(cols, mode):
    rng = np.random.default_rng(cols)
    w = rng.standard_normal((12, cols), dtype=np.float32)
    w[1] = 0
    w[2] = -0.0
    w[3] *= np.float32(1e-38)                    # row scale subnormal
    w[4] = np.sign(w[4]) * np.float32(2e-42)      # 1 / scale overflows
    w[5, -1] = -np.abs(w[5]).max() * 2           # the maximum in the remainder
    w[6] = np.float32(0.75)
    if mode == 0:
        w[7, 0] = np.inf
        w[8, -1] = np.nan
    q, s = E.quantize_q8(w, mode)
    q0, s0 = ob.quantize_q8(w, mode)
    assert (s.view(np.uint32) == s0.view(np.uint32)).all() and (q == q0).all()


def test_q4_0_blocks():
    rng = np.random.default_rng(3)
    w = rng.standard_normal((40, 160), dtype=np.float32)
    w[0] = 0
    w[1, 5], w[1, 9] = 9.0, -9.0                 # equal sizes: the first one's sign
    w[2, 40], w[2, 33] = 9.0, -9.0
    w[3] *= np.float32(1e-40)
    w[4] = np.float32(-1.5)
    w[5] *= np.float32(1e6)                      # scale past fp16
    assert (E.quantize_q4_0(w) == ob.quantize_q4_0(w)).all()
