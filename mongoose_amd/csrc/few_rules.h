// few_rules.h -- where the few-row kernels (few_rows.hip, few_gemm.hip) read a weight matrix and which calls take them, in plain C++:
// the kernels and the dispatch use these functions, and so do the host tests that walk them over whole matrices and over
// what was measured.
#pragma once
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstddef>

namespace mg {

// One launch, tiles of 16 to 128 weight rows x 16 to 64 activation rows a workgroup (few_tile chooses); what follows the
// product is the epilogue of the mode.
enum FewMode {
    FEW_RESID,       // Y += v * scale + bias; optionally the next projection's split of Y * nextGain and the rows' sums of squares
    FEW_SWIGLU,    // seg0 = gate, seg1 = up: silu(g) * u as the split of the down projection's input
    FEW_QKV,         // seg0 = q, seg1 = k, seg2 = v: bias, RoPE, q rows to seg0.Y, K / V rows into the caches at pos0 + row
};

// A lane (quarter fq = lane / 16, index fr = lane % 16 in it) loads a piece of 16 bytes (Q4_0: 8 bytes of nibbles) of a
// 16-row block of weights: piece few_piece of row few_load_row, so that a quarter wave reads whole 64-k rows.  A row of
// 32 weights has only the first two of the four pieces; the lanes of the others read those again (nothing of a chunk that
// is not there is multiplied, but every load is made).
constexpr int few_load_row(int fq, int fr) { return 4 * fq + (fr >> 2); }
constexpr int few_piece(int fr, int K) { return fr & (K < 64 ? 1 : 3); }
// Byte offset of that piece in the matrix, chunk 0; the chunks of 64 k follow few_chunk_bytes apart.
constexpr size_t few_piece_at(int row, int piece, int K, int q4) { return (size_t)row * (q4 ? K >> 1 : K) + (size_t)piece * (q4 ? 8 : 16); }
constexpr int few_chunk_bytes(int q4) { return q4 ? 32 : 64; }
// Chunks past the last whole one ask for that one again; where there is none, for chunk 0.
constexpr int few_last_chunk(int K) { return K < 64 ? 0 : (K >> 6) - 1; }
// Index, from the first fp16 scale of a Q4_0 matrix, of the two scales loaded with chunk 0 of a row.  A row of 32 weights has
// one scale: the load takes the one before it along (the first row's: the last bytes of the nibbles), not the one behind,
// which the last row does not have.  few_own_scale: where the row's first scale then lies.
constexpr int few_own_scale(int K) { return K < 64 ? 1 : 0; }
constexpr long long few_scales_at(int row, int K) { return (long long)row * (K >> 5) - few_own_scale(K); }

// ---- weights read ahead of the launches that multiply them (few_rows.hip) ----
// A region is a plane of a matrix (rows of int8 weights or of nibbles, or fp16 scales; `bytes` in all): its tiles below `tiles`, `run`
// bytes each, of which tile t is wanted on XCD (t + tile0) mod 8.  per: 0, or the 16-row blocks of half a head, of which tile t is
// block t % per in head t / per (base: the first or the second halves').  run, bytes: multiples of 16.
struct FewRegion { const char* base; unsigned run, bytes; int tiles, tile0, per; };
// What an XCD's workgroups read of it, in pieces of a KB, and where a lane's 16 bytes of piece p are.  (The last piece of a tile
// reads the tile's end again, a tile past the matrix's end the matrix's.)
constexpr unsigned few_ahead_per(const FewRegion& r) { return (r.run + 1023) >> 10; }
constexpr unsigned few_ahead_pieces(const FewRegion& r, int xcd) {
    const int t0 = (xcd - r.tile0) & 7;
    return t0 < r.tiles ? ((unsigned)(r.tiles - t0 + 7) >> 3) * few_ahead_per(r) : 0;
}
constexpr unsigned few_ahead_at(const FewRegion& r, int xcd, unsigned p, int lane) {
    const unsigned i = p / few_ahead_per(r), t = (unsigned)((xcd - r.tile0) & 7) + 8 * i, in = ((p - i * few_ahead_per(r)) << 10) + (unsigned)lane * 16;
    const unsigned at = (r.per ? t / r.per * 2 * r.per + t % r.per : t) * r.run + (in < r.run - 16 ? in : r.run - 16);
    return at < r.bytes - 16 ? at : r.bytes - 16;
}

// What the launches behind an attention launch multiply T rows by, in their order (launch_few_rows: W1 and W2 where the mode has them,
// N1 their rows): its idle CUs read it into the L2s.
struct FewNext { FewMode mode; const void* W0; const void* W1; const void* W2; int N, N1, K, q4; };
// What an attention launch of `grid` workgroups reads ahead.  Up to 200 KB a reading workgroup (100: 0.5B, 200 rows 1,448 us a call
// against 1,388) and 20 MB (12: 16 rows 777 against 714; past it the 1.1B shape, 44 MB a layer, loses, 16 rows 360 at 12, 371 at 20, 370 at
// 24); a matrix that does not fit is taken in part, its first tiles.  Readers are the workgroups up to 256, but 96 at least -- they
// then share CUs with the attention's, which wait more than they load (0.5B, 301 rows, 266 workgroups of attention, with 0 / 32 / 64
// / 96 / 128 readers 1,908 / 1,896 / 1,849 / 1,814 / 1,799, 200 rows 1,388 / 1,388 / 1,386 / 1,410 / 1,402) -- and no more than
// have 64 KB each.  There a layer that does not fit whole is read up to 4 MB past its first matrix: the attention waits for its CUs, and what many
// rows are multiplied by is wanted too slowly for a cold start to matter past the first tiles.  Nothing read / 8 / 12 / 19.2 MB, us a
// call, Q8: eight 1.1B layers (44 MB), 100 rows 549 / 545 / 549 / 562, 128 573 / 566 / 571 / 583, 256 788 / 786 / 796 / 806; six of 2048 x 8192, heads of 64, 100 rows
// 465 / 460 / 463 / 475; eight of 1536 x 6144 (34) 521 / 514 / 521 / 532; four of 3072 x 8192, heads of 128 (101; Wo alone 9.4) 441 / 443 / 437 / 438; 1.1B Q4_0 (22) 975 /
// 974 / 982 / 987.  Layers that fit: 0.5B, 100 behind 300, 1,137 / 1,128 / 1,129 / 1,092, 1536 x 6144 Q4_0 (17) 256 rows 1,513 / 1,486 / 1,485 / 1,463.
constexpr long long FEW_AHEAD_EACH = 200 << 10, FEW_AHEAD_MOST = 20 << 20, FEW_AHEAD_LEAST = 64 << 10, FEW_AHEAD_SHARED = 4 << 20;
constexpr long long few_ahead_bytes(const FewNext& m) {
    const long long rows = m.mode == FEW_QKV ? m.N + 2LL * m.N1 : (m.mode == FEW_SWIGLU ? 2LL : 1LL) * m.N;
    return m.q4 ? rows * m.K / 16 * 9 : rows * m.K;
}
// Planes of Wo, gate | up and down, one a matrix or, in Q4_0, two, and of Q8 q|k|v: one of v, of q and k the halves of their heads.
constexpr int FEW_REGIONS = 13;
struct FewAhead { FewRegion r[FEW_REGIONS]; int n, first, readers; };      // first: the launch's first workgroup that reads ahead
// tileRows(next): the weight rows of a tile of that launch.
template <class TileRows>
inline FewAhead few_plan(unsigned grid, const FewNext* next, int nNext, int headDim, TileRows tileRows) {
    FewAhead a{};
    a.first = INT_MAX;
    const unsigned own = (grid + 7) / 8 * 8, room = own + 96 > 256 ? 96 : 256 - own;
    long long left = std::min(room * FEW_AHEAD_EACH, FEW_AHEAD_MOST), bytes = 0, all = 0;
    for (int i = 0; i < nNext; i++) all += next[i].mode == FEW_QKV && next[i].q4 ? 0 : few_ahead_bytes(next[i]);
    if (own + 96 > 256 && all > left) left = std::min(left, few_ahead_bytes(next[0]) + FEW_AHEAD_SHARED);
    // one matrix, or two read tile by tile (W1; per: the halves of W0's heads)
    auto take = [&](const void* W0, const void* W1, int N, int K, int q4, int rows, int tiles, int tile0, int per) {
        const unsigned row = q4 ? K / 2 : K, run = rows * row;
        const int two = per || W1 ? 2 : 1;
        const long long one = (long long)run * two * (q4 ? 9 : 8) / 8;
        int n = (int)std::min<long long>(tiles, left / one);
        if (n < tiles) n = n / 8 * 8;
        if (n <= 0 || a.n + two * (q4 ? 2 : 1) > FEW_REGIONS || (long long)N * row >= 1LL << 32) { left = 0; return; }
        for (int h = 0; h < two; h++) {
            const char* W = static_cast<const char*>(h && W1 ? W1 : W0);
            const unsigned skip = h && per ? per * run : 0;
            a.r[a.n++] = FewRegion{W + skip, run, N * row - skip, n, tile0, per};
            if (q4) a.r[a.n++] = FewRegion{W + (size_t)N * row + skip / 8, run / 8, (N * row - skip) / 8, n, tile0, per};
        }
        left = n < tiles ? 0 : left - n * one;
        bytes += n * one;
    };
    for (int i = 0; i < nNext; i++) {
        const FewNext& m = next[i];
        if (m.mode == FEW_QKV) {
            // (not in Q4_0, whose ten planes hold a fifteenth of a layer's bytes and take more turns than the other eight: 0.5B, without / with / nothing
            // read at all, 2 rows 760 / 798 / 757 us a call, 16 795 / 825 / 830, 37 behind 200 887 / 898 / 914, 301 1,637 / 1,656 / 1,633)
            if (m.q4) break;
            const int per = headDim / 32, tq = m.N / 32, tk = m.N1 / 32;
            take(m.W0, nullptr, m.N, m.K, m.q4, 16, tq, 0, per);
            take(m.W1, nullptr, m.N1, m.K, m.q4, 16, tk, tq, per);
            take(m.W2, nullptr, m.N1, m.K, m.q4, 32, tk, tq + tk, 0);
        } else {
            const int rows = tileRows(m);
            take(m.W0, m.W1, m.N, m.K, m.q4, rows, (m.N + rows - 1) / rows, 0, 0);
        }
    }
    if (a.n) {
        a.first = (int)own;
        a.readers = (int)std::min<long long>(room, (bytes / FEW_AHEAD_LEAST + 8) / 8 * 8);
    }
    return a;
}

// ---- which products take the integer form (few_gemm.hip) ----
// Eight waves sum a run of K each, whole chunks of 64, of products of two signed bytes in 32 bits.  Past this K a run of them
// could exceed those (K = 1,048,064 is the last that cannot); the tiled kernel's fp32 sums take any.
constexpr bool few_gemm_sums_fit(int K) { return (long long)(((K >> 6) + ((K & 63) ? 1 : 0) + 7) / 8) * 64 * (128 * 128) < (1LL << 31); }

// What it keeps of T rows, 16 at a time: three digit planes, and for each of the eight runs a scale and a mark a row.
constexpr size_t few_gemm_bytes(int T, int K) {
    const size_t blocks = ((size_t)(T > 0 ? T : 0) + 15) / 16, chunks = ((size_t)K + 63) / 64;
    return blocks * (chunks * 3 * 1024 + 8 * 16 * (sizeof(float) + 1));
}

// ---- which prefills take the few-row kernels, and which the tiled GEMMs (prefill.hip) ----
// Rows up to which some prefill takes them.  The tiled GEMMs want work for every CU, so the line falls with the weights of a
// layer.  Microseconds a layer, few-row / tiled, Q8 and Q4_0, nothing cached: 0.5B shape (15 million weights) 36 / 69 and
// 39 / 77 at 37 rows, 103 / 119 and 118 / 141 at 506, 138 / 136 and 156 / 154 at 625; 1.1B (44) 147 / 164 and 182 / 203 at
// 294, 161 / 173 and 203 / 211 at 346, 183 / 191 and 239 / 219 at 415; 8B (218) 236 / 243 and 286 / 297 at 124.  (Drawn before gate | up of
// many rows went through LDS (few_swiglu_kernel); with that the few-row kernels lead up to it everywhere and some way past it: 0.5B 78 / 110
// at 512 rows, 118 / 132 at 700, 157 / 157 at 1,024, Q4_0 131 / 166 at 700; 1.1B 122 / 152 at 301, 150 / 173 at 400, 237 / 231 at 600.)
inline int few_rows_most(int dim, int kvDim, int ffn) {
    const double millions = ((double)dim * (2.0 * dim + 2.0 * kvDim) + 3.0 * dim * ffn) * 1e-6;
    const int n = (int)(2300.0 / std::sqrt(millions));
    return n < 1500 ? n : 1500;
}
// T rows behind pos0 cached ones.
//   * The largest Q8 layers, past 128 rows: a third block of 64 rows through every few-row tile costs more than the half-filled second
//     tile of 128 rows does (dim 4096: ffn 11008 at 137 rows 299 / 322, 12288 at 132 300 / 291; 3584 x 14336 at 152 296 / 270;
//     4096 x 14336 at 132 315 / 275).  Q4_0 layers, whose conversions weigh more in the tiled GEMMs, keep the line above
//     (380 / 367 there, 352 / 347 at 3584 x 14336, 303 / 340 at 4096 x 11008); so do layers whose attention is one round
//     (below) behind a long cache (3584 x 14336, 28 heads, 144 rows: 270 / 262, behind 3,000 333 / 391).
//   * Cached rows: the few-row attention takes a workgroup a query head and 16 rows, 256 at a time, and each such round reads the
//     cache once; the tiled one splits the cache rows in a pass of its own and reads them once for 128 rows.  One or two
//     rounds cost less than that for every cached row (heads of 64: 0.011 us a round against 0.026; of 128: 0.020 against
//     0.042), so the line does not move: 8B at 128 rows behind 12,000 472 / 757, 1.1B at 256 391 / 447.  With three rounds the
//     projections' lead is used up after 400 (at the line) to 3,000 rows (at three quarters of it): 0.5B at 590 rows 133 / 136
//     with nothing cached, 154 / 150 behind 600, 331 / 283 behind 6,000; 1.1B at 301 167 / 184 behind 600, 247 / 246
//     behind 3,000, 350 / 324 behind 6,000; the toy shape at 1,034 107 / 123 and, behind 3,000, 208 / 202.
inline bool few_rows_pay(int T, int pos0, int dim, int kvDim, int ffn, int nHeads, bool q4) {
    const int most = few_rows_most(dim, kvDim, ffn);
    const int rounds = (int)(((long long)nHeads * ((T + 15) / 16) + 255) / 256);
    if (T > most || (!q4 && T > 128 && 3.0 * dim * ffn > 145e6 && (rounds > 1 || pos0 < 800))) return false;
    return rounds <= 2 || T <= most * (1.05 - pos0 / 8000.0);
}

}  // namespace mg
