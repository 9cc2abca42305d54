// few_rules.h -- where the few-row kernels (few_rows.hip) read a weight matrix, in plain C++: the kernels use these
// functions, and so does the host test that walks them over whole matrices.
#pragma once
#include <cstddef>

namespace mg {

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

}  // namespace mg
