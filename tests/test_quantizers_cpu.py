"""The host quantizers' wide paths against the oracle's plain loops, bit for bit, where they can go wrong: remainders of the
32 values taken at once, ties of the maximum, rows of zeros, tiny and infinite values."""
import ctypes
import os
import subprocess

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


ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def variants(tmp_path_factory):
    """The quantizers' inner loops by instruction set, which the library chooses by the CPU it runs on: host_quant.cpp
    compiled into a library of its own that calls each by name (no contraction of products and sums, as in its own build)."""
    d = tmp_path_factory.mktemp("quant")
    (d / "v.cpp").write_text(r"""
#include "host_quant.cpp"
using namespace mg;
extern "C" int has(int isa) { return isa == 0 ? 1 : isa == 1 ? have_avx2() : have_avx512(); }
extern "C" void q8(int isa, const float* w, int rows, int cols, int mode, int8_t* q, float* scales) {
    for (int r = 0; r < rows; r++) {
        const float* src = w + (size_t)r * cols;
        int8_t* dst = q + (size_t)r * cols;
        const float amax = isa == 2 ? q8_absmax_avx512(src, cols) : isa == 1 ? q8_absmax_avx2(src, cols) : q8_absmax(src, 0, cols, 0.0f);
        const float s = scales[r] = amax / 127.0f;
        if (!(s > 0.0f)) std::memset(dst, 0, (size_t)cols);
        else if (isa == 2) q8_row_avx512(src, cols, s, amax, mode, dst);
        else if (isa == 1) q8_row_avx2(src, cols, s, amax, mode, dst);
        else q8_row(src, 0, cols, s, amax, mode, dst);
    }
}
extern "C" void q4(int isa, const float* w, size_t nb, uint8_t* out) {
    if (isa == 2) q4_0_blocks_avx512(w, 0, nb, out);
    else for (size_t b = 0; b < nb; b++) { if (isa == 1) q4_0_block_avx2(w + b * 32, out + b * 18); else q4_0_block(w + b * 32, out + b * 18); }
}
""")
    so = d / "v.so"
    subprocess.run(["g++", "-O3", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", "-w", "-I", os.path.join(ROOT, "mongoose_amd", "csrc"),
                    str(d / "v.cpp"), "-o", str(so), "-lpthread"], check=True)
    v = ctypes.CDLL(str(so))
    f, i8, u8 = ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int8), ctypes.POINTER(ctypes.c_uint8)
    v.q8.argtypes = [ctypes.c_int, f, ctypes.c_int, ctypes.c_int, ctypes.c_int, i8, f]
    v.q4.argtypes = [ctypes.c_int, f, ctypes.c_size_t, u8]
    return v


@pytest.mark.parametrize("isa", [0, 1, 2], ids=["plain", "avx2", "avx512"])
def test_every_instruction_set(variants, isa, monkeypatch):
    """The tests above through each of them, and more lengths of a row; scales over thirty powers of two."""
    if not variants.has(isa):
        pytest.skip("this CPU does not have it")

    def q8(w, mode=0):
        w = np.ascontiguousarray(w)
        q, s = np.empty(w.shape, np.int8), np.empty(len(w), np.float32)
        variants.q8(isa, E._fp(w), w.shape[0], w.shape[1], mode, E._i8p(q), E._fp(s))
        return q, s

    def q4(w):
        out = np.empty(w.size // 32 * 18, np.uint8)
        variants.q4(isa, E._fp(w), w.size // 32, E._u8p(out))
        return out

    monkeypatch.setattr(E, "quantize_q8", q8)
    monkeypatch.setattr(E, "quantize_q4_0", q4)
    for mode in (0, 1):
        for cols in (1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 127, 896):
            test_q8_rows(cols, mode)
    test_q4_0_blocks()
    rng = np.random.default_rng(4)
    w = rng.standard_normal((500, 64), dtype=np.float32) * np.exp(rng.uniform(-20, 8, (500, 1))).astype(np.float32)
    assert (E.quantize_q4_0(w) == ob.quantize_q4_0(w)).all()
