"""Where the few-row kernels read a weight matrix (few_rules.h), compiled for the host and walked over whole matrices."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mongoose_amd", "csrc")


def _run(tmp_path, source):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(source)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("q4", [0, 1])
def test_loads_stay_inside_the_matrix(tmp_path, q4):
    """Every lane's loads of every chunk a wave asks for -- past the end too, eight waves, both ring depths -- end inside the
    matrix (N rows clamped to the last, as the kernel does), from rows of 32 weights up."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <algorithm>
#include <cstdio>
using namespace mg;
int main() {
    const int q4 = %d;
    for (int K = 32; K <= 2176; K += 32)
        for (int N : {1, 2, 15, 16, 17, 33}) {
            const size_t bytes = (size_t)N * (q4 ? K / 2 : K);
            const long long scales = (long long)N * (K / 32);
            for (int r0 = 0; r0 < N; r0 += 16)
                for (int lane = 0; lane < 64; lane++)
                    for (int c = 0; c < (K >> 6) + 40; c++) {
                        const int fq = lane / 16, fr = lane %% 16, cc = std::min(c, few_last_chunk(K));
                        const size_t at = few_piece_at(std::min(r0 + few_load_row(fq, fr), N - 1), few_piece(fr, K), K, q4) + (size_t)cc * few_chunk_bytes(q4);
                        const long long sc = few_scales_at(std::min(r0 + fr, N - 1), K) + 2 * cc, own = sc + few_own_scale(K);
                        if (at + (q4 ? 8 : 16) > bytes || at %% (q4 ? 8 : 16) || (q4 && (sc * 2 < -(long long)bytes || sc + 2 > scales || own != (long long)std::min(r0 + fr, N - 1) * (K / 32) + 2 * cc))) {
                            std::printf("K %%d N %%d lane %%d chunk %%d\n", K, N, lane, c);
                            return 0;
                        }
                    }
        }
    std::printf("ok\n");
}
""" % q4)
    assert out == "ok\n", out
