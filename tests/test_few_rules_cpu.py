"""Where the few-row kernels read a weight matrix and which prefills take them (few_rules.h), compiled for the host."""
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


def test_integer_sums_fit_32_bits(tmp_path):
    """A wave's run of the few-row GEMM: whole chunks of 64 k, an eighth of them, of products up to (-128) (-128)."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <cstdio>
int main() {
    for (int K = 32; K > 0 && K < 2147483647 - 64; K += K < 1500000 ? 32 : 1048576) {
        const long long chunks = ((long long)K + 63) / 64, run = (chunks + 7) / 8 * 64;
        if (mg::few_gemm_sums_fit(K) != (run * 16384 <= 2147483647ll)) { std::printf("K %d\n", K); return 0; }
    }
    std::printf("%d %d\n", mg::few_gemm_sums_fit(1048064), mg::few_gemm_sums_fit(1048096));
}
""")
    assert out == "1 0\n", out


def test_digits_fit_the_callers_planes(tmp_path):
    """What the few-row GEMM keeps of the activations against the workspace that mongoose_q8_gemm asks a caller for (two bf16
    planes of T rounded up to 128 rows and K to 64), over rows and K, K = 64 and whole blocks of 128 rows the tightest."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <cstdio>
int main() {
    for (int T = 0; T <= 1100; T++)
        for (int K = 32; K < 1048096; K += K < 2048 ? 32 : 8160)
            if (mg::few_gemm_bytes(T, K) > 2 * (size_t)((T + 127) / 128 * 128) * ((K + 63) / 64 * 64) * 2) { std::printf("T %d K %d\n", T, K); return 0; }
    std::printf("%zu\n", mg::few_gemm_bytes(128, 64));
}
""")
    assert out == "%d\n" % (8 * (3072 + 640)), out


QWEN, TINY, LLAMA, TOY = (896, 128, 4864, 14), (2048, 256, 5632, 32), (4096, 1024, 14336, 32), (512, 128, 1376, 8)


# (shape, Q4_0, rows, cached rows, microseconds a layer few-row and tiled) as measured where the two differ by more than 4 %
@pytest.mark.parametrize("shape,q4,rows,pos0,few,tiled", [
    (TOY, 0, 646, 0, 73, 101), (TOY, 0, 970, 12000, 361, 438), (TOY, 0, 1293, 3000, 225, 214), (TOY, 0, 1380, 6000, 334, 304),
    (QWEN, 0, 37, 200, 38, 74), (QWEN, 0, 512, 6000, 234, 269), (QWEN, 0, 590, 3000, 233, 208), (QWEN, 1, 301, 12000, 346, 418),
    (QWEN, 1, 590, 1500, 198, 189), (TINY, 0, 301, 600, 167, 184), (TINY, 0, 301, 6000, 350, 324), (TINY, 0, 256, 12000, 391, 447),
    (TINY, 1, 340, 3000, 303, 285), (TINY, 1, 448, 0, 257, 224), (LLAMA, 0, 64, 12000, 407, 701), (LLAMA, 0, 128, 12000, 472, 757),
    (LLAMA, 0, 132, 0, 315, 275), (LLAMA, 0, 150, 6000, 564, 542), (LLAMA, 1, 128, 0, 280, 298), (LLAMA, 1, 192, 0, 441, 374),
    ((4096, 4096, 11008, 32), 0, 137, 0, 299, 322), ((3584, 512, 14336, 28), 0, 152, 0, 296, 270),
    ((3584, 512, 14336, 28), 0, 144, 3000, 333, 391), ((3584, 512, 14336, 28), 0, 152, 3000, 418, 395)])
def test_the_faster_path_is_taken(tmp_path, shape, q4, rows, pos0, few, tiled):
    out = _run(tmp_path, '#include "few_rules.h"\n#include <cstdio>\nint main() { std::puts(mg::few_rows_pay(%d, %d, %d, %d, %d, %d, %d != 0) ? "few" : "tiled"); }'
               % (rows, pos0, *shape, q4))
    assert out.strip() == ("few" if few < tiled else "tiled")


def test_reading_ahead_covers_the_tiles_and_stays_inside(tmp_path):
    """Regions as an attention launch forms them (whole and partial matrices, last tiles cut off by the matrix's end, halves of heads
    of 64 and 128, both formats' planes, rows of 32 weights up): every 16 bytes of a tile are read on the XCD that the tile's
    workgroup will run on, and nothing outside the plane is."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <cstdio>
#include <vector>
using namespace mg;
int walk(unsigned row, int N, int rows, int tiles, int tile0, int per, int half) {
    const unsigned run = rows * row, skip = half ? per * run : 0;
    FewRegion r{nullptr, run, N * row - skip, tiles, tile0, per};
    std::vector<int> by((N * row + 15) / 16, -1);
    for (int x = 0; x < 8; x++)
        for (unsigned p = 0; p < few_ahead_pieces(r, x); p++)
            for (int lane = 0; lane < 64; lane++) {
                const unsigned at = skip + few_ahead_at(r, x, p, lane);
                if (at % 16 || at + 16 > N * row) return 1;
                if (by[at / 16] < 0) by[at / 16] = x;
            }
    for (int t = 0; t < tiles; t++) {
        const unsigned first = (per ? t / per * 2 * per + t % per + (half ? per : 0) : t) * rows;
        for (unsigned b = first * row; b < (first + rows) * row && b < N * row; b += 16)
            if (by[b / 16] != ((t + tile0) & 7)) return 2;
    }
    return 0;
}
int main() {
    for (int K : {32, 96, 448, 896, 4864})
        for (int div : {1, 2, 16})                         // bytes of a row: int8, nibbles, scales
            for (int N : {64, 128, 200, 896, 1000}) {
                const unsigned row = K / div;
                for (int rows : {16, 32, 64}) {
                    const int tiles = (N + rows - 1) / rows;
                    for (int n : {tiles, tiles / 8 * 8})
                        if (int e = n ? walk(row, N, rows, n, 0, 0, 0) : 0) { std::printf("K %d / %d N %d rows %d tiles %d: %d\n", K, div, N, rows, n, e); return 0; }
                }
                for (int hd : {64, 128})
                    if (N % hd == 0)
                        for (int tile0 : {0, 28, 3})
                            for (int half : {0, 1})
                                if (int e = walk(row, N, 16, N / 32, tile0, hd / 32, half)) { std::printf("K %d / %d N %d heads of %d: %d\n", K, div, N, hd, e); return 0; }
            }
    std::puts("ok");
}
""")
    assert out == "ok\n", out


@pytest.mark.parametrize("q4", [0, 1])
@pytest.mark.parametrize("dim,kvDim,ffn,head_dim,grid", [(896, 128, 4864, 64, 56), (2048, 256, 5632, 64, 64), (1024, 256, 2816, 128, 250), (256, 256, 96, 64, 16)])
def test_what_an_attention_launch_reads_ahead(tmp_path, q4, dim, kvDim, ffn, head_dim, grid):
    """few_plan over a layer's four launches: a layer below the limits is read whole -- every 16 bytes of Wo, gate, up and down and, in Q8,
    the next layer's q, k and v, weights and scales, on the XCD of their tile -- and of a larger one the matrices in their
    order, the last one in part, up to the limits; nothing outside a plane."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>
using namespace mg;
struct Mat { int N, K, rows, tile0, per; std::vector<char> w; std::vector<int> by; };
int main() {
    const int q4 = %d, dim = %d, kvDim = %d, ffn = %d, hd = %d, grid = %d, per = hd / 32, tq = dim / 32, tk = kvDim / 32;
    Mat m[7] = {{dim, dim, 16, 0, 0}, {ffn, dim, 64, 0, 0}, {ffn, dim, 64, 0, 0}, {dim, ffn, 32, 0, 0}, {dim, dim, 16, 0, per}, {kvDim, dim, 16, tq, per}, {kvDim, dim, 32, tq + tk, 0}};
    long long total = 0;
    for (auto& x : m) {
        x.w.resize(q4 ? (size_t)x.N * x.K / 16 * 9 : (size_t)x.N * x.K);
        x.by.assign(x.w.size() / 16, -1);
        if (!q4 || &x < m + 4) total += x.w.size();
    }
    const FewNext next[4] = {{FEW_RESID, m[0].w.data(), nullptr, nullptr, dim, 0, dim, q4}, {FEW_SWIGLU, m[1].w.data(), m[2].w.data(), nullptr, ffn, 0, dim, q4},
                             {FEW_RESID, m[3].w.data(), nullptr, nullptr, dim, 0, ffn, q4}, {FEW_QKV, m[4].w.data(), m[5].w.data(), m[6].w.data(), dim, kvDim, dim, q4}};
    const FewAhead a = few_plan(grid, next, 4, hd, [&](const FewNext& n) { return n.mode == FEW_SWIGLU ? 64 : n.K == dim ? 16 : 32; });
    if (a.first %% 8 || a.first < grid || a.readers %% 8 || a.readers < 8) return std::puts("workgroups"), 0;
    for (int x = 0; x < 8; x++)
        for (int r = 0; r < a.n; r++)
            for (unsigned p = 0; p < few_ahead_pieces(a.r[r], x); p++)
                for (int lane = 0; lane < 64; lane++) {
                    const char* at = a.r[r].base + few_ahead_at(a.r[r], x, p, lane);
                    int in = -1;
                    for (int i = 0; i < 7; i++) if (at >= m[i].w.data() && at + 16 <= m[i].w.data() + m[i].w.size()) in = i;
                    if (in < 0 || (at - m[in].w.data()) %% 16) return std::puts("outside"), 0;
                    int& by = m[in].by[(at - m[in].w.data()) / 16];
                    if (by < 0) by = x;
                }
    const long long most = std::min((grid + 7) / 8 * 8 + 96 > 256 ? 96 : 256 - (grid + 7) / 8 * 8, 1 << 20) * FEW_AHEAD_EACH;
    const bool whole = total <= std::min(most, FEW_AHEAD_MOST);
    long long read = 0;
    bool cut = false;
    for (int i = 0; i < 7; i++) {
        Mat& x = m[i];
        const size_t row = q4 ? x.K / 2 : x.K;
        size_t got = 0;
        for (size_t b = 0; b < x.w.size(); b += 16) {
            if (x.by[b / 16] < 0) continue;
            got += 16;
            const size_t nr = b < x.N * row ? b / row : (b - x.N * row) / (x.K / 16);
            if (q4 && b >= x.N * row && x.K %% 256) continue;          // (16 bytes of scales of more than a row)
            const size_t tile = x.per ? nr / 16 / (2 * x.per) * x.per + nr / 16 %% x.per : nr / x.rows;
            if (x.by[b / 16] != (int)((tile + x.tile0) %% 8)) return std::printf("matrix %%d row %%zu: XCD %%d\n", i, nr, x.by[b / 16]), 0;
        }
        read += got;
        if (got && cut && i != 2) return std::puts("order"), 0;        // (up goes with gate)
        if (q4 && i >= 4) { if (got) return std::puts("q|k|v"), 0; continue; }
        if (got < x.w.size()) { cut = true; if (whole) return std::printf("matrix %%d: %%zu of %%zu bytes\n", i, got, x.w.size()), 0; }
    }
    if (read > std::min(most, FEW_AHEAD_MOST) || (!whole && 10 * read < 9 * std::min(most, FEW_AHEAD_MOST))) return std::printf("%%lld of %%lld bytes\n", read, total), 0;
    std::puts("ok");
}
""" % (q4, dim, kvDim, ffn, head_dim, grid))
    assert out == "ok\n", out


@pytest.mark.parametrize("q4", [0, 1])
@pytest.mark.parametrize("dim,kvDim,ffn,head_dim", [(2048, 256, 5632, 64), (3072, 1024, 8192, 128), (4096, 1024, 14336, 128), (1280, 320, 3584, 64)])
def test_what_is_read_ahead_beside_an_attention(tmp_path, q4, dim, kvDim, ffn, head_dim):
    """Where the reading workgroups share CUs with the attention's (more than 160 of those), a layer that does not fit whole is read up to 4 MB
    past Wo; one that fits, and any with CUs to spare, up to the limits."""
    out = _run(tmp_path, r"""
#include "few_rules.h"
#include <cstdio>
using namespace mg;
int main() {
    const int q4 = %d, dim = %d, kvDim = %d, ffn = %d, hd = %d;
    const void* w = reinterpret_cast<const void*>(16ull << 30);         // (an address for the plan, not for reading)
    const FewNext next[4] = {{FEW_RESID, w, nullptr, nullptr, dim, 0, dim, q4}, {FEW_SWIGLU, w, w, nullptr, ffn, 0, dim, q4},
                             {FEW_RESID, w, nullptr, nullptr, dim, 0, ffn, q4}, {FEW_QKV, w, w, w, dim, kvDim, dim, q4}};
    const double wb = q4 ? 9.0 / 16 : 1.0, wo = wb * dim * dim, layer = wb * (wo / wb + 3.0 * dim * ffn + (q4 ? 0 : (double)dim * (dim + 2 * kvDim)));
    for (int n = 1; n <= 4; n++)
        for (int grid = 8; grid <= 512; grid += 8) {
            const FewAhead a = few_plan(grid, next, n, hd, [&](const FewNext& m) { return m.mode == FEW_SWIGLU ? 64 : 16; });
            double read = 0, all = 0;
            for (int i = 0; i < a.n; i++) read += (double)a.r[i].run * a.r[i].tiles;
            for (int i = 0; i < n; i++) all += i == 1 ? wb * 2.0 * ffn * dim : i == 2 ? wb * dim * ffn : i == 0 ? wo : layer - wo - wb * 3.0 * dim * ffn;
            const double most = (double)(grid <= 160 ? 256 - grid : 96) * FEW_AHEAD_EACH, cap = most < FEW_AHEAD_MOST ? most : FEW_AHEAD_MOST;
            const double want = all <= cap ? all : grid > 160 && wo + (4 << 20) < cap ? wo + (4 << 20) : cap;
            // (a matrix in part goes by eight tiles an XCD: of up to 64 rows of two matrices)
            const double least = want - wb * 8 * 128 * dim;
            if (read > want * (1 + 1e-9) || (all <= cap ? read < want * (1 - 1e-9) : read < least)) return std::printf("%%d launches behind %%d: %%.0f of %%.0f bytes\n", n, grid, read, want), 0;
        }
    std::puts("ok");
}
""" % (q4, dim, kvDim, ffn, head_dim))
    assert out == "ok\n", out
