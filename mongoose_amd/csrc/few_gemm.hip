// few_gemm.hip -- several rows of fp32 activations through one Q8 matrix (mongoose_q8_gemm up to some hundred rows), on the
// integer matrix instruction.
//
// Y[T,N] = A[T,K] . W[N,K]^T: an activation becomes a whole number of 24 bits times a scale, a = s (65536 d2 + 256 d1 + d0)
// with signed digits of a byte, so that v_mfma_i32_16x16x64_i8 multiplies the int8 weights as they are -- three products at
// twice the bf16 rate where two bf16 terms need two at the plain one, no conversion of a weight (which was a third of a
// workgroup's time: no other workgroup's conversions serve it), three bytes an activation instead of four.  (Operands split
// into small integers for an integer matrix unit: the Ozaki scheme, as in Ootomo, Ozaki and Yokota, "DGEMM on integer matrix
// multiplication unit", 2024.)  The sums of a wave are whole numbers, exact; scale, row scale, bias and the sum of the waves are
// fp32.  Bound by the operands a workgroup pulls through its CU's L1.  Microseconds a call, weights from memory, two bf16 terms
// / this: 77 x 5632 x 2048 19.7 / 14.1, 16 x 5632 x 2048 10.4 / 9.9, 37 x 896 x 4864 11.8 / 11.1, 300 x 5632 x 2048 36.5 / 31.9,
// 48 x 9000 x 8192 49.7 / 39.8, 500 x 9000 x 8192 240 / 207.
//
// Precision: the eight waves of a workgroup split K into eight runs, and every row has a scale for each run, the run's
// largest value / 8355584.  A value is off by half a step, 2^-24 of the run's largest one (by up to 1.4 steps next to that one,
// where the roundings of factor, product and scale weigh as much): no more than two bf16 terms leave of it (up to 2^-17 of
// itself) down to a 64th of the largest.  The smaller ones of a run (3 to 5 % of normal samples, 28 % of a SwiGLU's outputs) are
// weighed against each other in mean square, their share of the run times the digits' error against the error of two bf16 terms
// of them; where the digits lose -- a few large values among small ones, a part of the run on a scale of its own -- the run is a
// wide one, its small values go in as two bf16 terms instead, and so keep 2^-17 of themselves however large their neighbours
// are.  Against 64 bits, two bf16 terms / digits alone / as it is: normal samples, K 64 to 8192 2.5e-6 / 1.5e-7 / 1.5e-7; one
// value R times the others, seen through weights that are zero there, K = 2048 (eight runs, one of them wide) R = 30 2.5e-6 /
// 3.9e-7 / 3.9e-7, 100 2.5e-6 / 1.2e-6 / 7.7e-7, 1,000 2.5e-6 / 1.2e-5 / 8.8e-7, 10^5 2.5e-6 / 1.2e-3 / 8.7e-7, 10^20 2.5e-6 /
// 0.35 / 8.7e-7; K = 64 (one run) 100 2.4e-6 / 3.4e-6 / 2.1e-6, from 1,000 on two bf16 terms' own.
// A wide run costs its chunks a second time, with conversions, shared by the eight waves.  Microseconds a call with no wide
// run, one of eight, about half of them, all (two bf16 terms): 77 x 5632 x 2048 14.1, 15.7, 19.2, 23.2 (19.7), 48 x 9000 x 8192
// 40, 45, 54, 74 (50), 300 x 5632 x 2048 32, 38, 55, 86 (36), 500 x 9000 x 8192 209, 257, 386, 555 (241).
#include "few_rows.h"
#include "few_rules.h"
#include "kernels.h"
#include "device_util.h"
#include <cmath>

namespace mg {

typedef int int4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int FG_WAVES = 8, FG_WG = 64 * FG_WAVES;
constexpr int FG_TOP = 127 * 65536 + 127 * 256;             // three signed digits go to 127 more: a product may round up past it
constexpr float FG_KEPT = 131072.f;                         // whole numbers from here on keep 2^-17 of themselves, as two bf16 terms do
constexpr float FG_EVEN = 6.58e9f;                          // 2^37.2 / 24: 1 / 12 of a step^2 against twice 2^-37.2 of a value^2

// chunks of 64 k (a last half one counts), and of them a wave's
__host__ __device__ inline int fg_chunks(int K) { return (K + 63) >> 6; }
__host__ __device__ inline int fg_per_wave(int K) { return (fg_chunks(K) + FG_WAVES - 1) / FG_WAVES; }

// ---------------------------------------------------------------------------
// Digits and scales, a wave per row and run of K (a workgroup four rows): a lane holds pieces of four k.  A 16-row block of a
// chunk is 3 KB, a KB a digit, in each the operand of a lane (lane = 16 q + row: k 16 q .. + 15 of the chunk) at lane * 16.
// Rows past T and k past K are zeros.  A run with a NaN or an infinity gets the scale NaN (so did the two bf16 terms of an
// infinity); one whose values are below 2^-64 is brought up by 2^64 first, which a negative scale says.  wide: 1 for a row's
// wide run (see above), whose small values are zeros here.
// ---------------------------------------------------------------------------
constexpr int FG_PIECES = 4;                                // a lane's pieces: runs of up to 1024 k
__device__ __forceinline__ unsigned max_bits(unsigned m, float4 v) {
    auto bits = [](float x) { return __builtin_bit_cast(unsigned, x) & 0x7fffffffu; };
    return max(max(m, max(bits(v.x), bits(v.y))), max(bits(v.z), bits(v.w)));
}

__global__ __launch_bounds__(WG) void few_digits_kernel(const float* in, signed char* out, float* scales, unsigned char* wide, int T, int K) {
    const int run = blockIdx.y, t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int chunks = fg_chunks(K), per = fg_per_wave(K);
    const int c0 = run * per, pieces = max(0, min(per, chunks - c0)) * 16;      // (a last run may be empty)
    const float* row = in + (size_t)min(t, T - 1) * K;
    auto get = [&](int p) {
        const int k = c0 * 64 + p * 4;
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        if (p < pieces && k < K && t < T) a = *reinterpret_cast<const float4*>(row + k);
        return a;
    };
    float4 v[FG_PIECES];
    unsigned m = 0;
#pragma unroll
    for (int j = 0; j < FG_PIECES; j++) { v[j] = get(lane + 64 * j); m = max_bits(m, v[j]); }
    for (int p = lane + 64 * FG_PIECES; p < pieces; p += 64) m = max_bits(m, get(p));      // longer runs are read twice
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    const bool bad = m >= 0x7f800000u, tiny = m < 0x1f800000u;           // (2^-64)
    const float up = tiny ? 0x1p64f : 1.0f, top = __builtin_bit_cast(float, m) * up;
    const float inv = m == 0 || bad ? 0.f : (float)FG_TOP / top;
    const float s = bad ? __builtin_nanf("") : top / (float)FG_TOP;
    const size_t tb = (size_t)(t >> 4);
    const int r = t & 15;
    if (lane == 0) scales[(tb * FG_WAVES + run) * 16 + r] = tiny ? -s : s;
    // values below this are small; of the wave: values that are not zero, small ones among them, and of the lane their squares
    const float lim = tiny ? s * FG_KEPT * 0x1p-64f : s * FG_KEPT;
    int some = 0, small = 0;
    float squares = 0.f;
    auto weigh = [&](float4 a) {                            // (called by whole waves; pieces past the run are zeros)
        const float x[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const bool low = x[e] != 0.f && fabsf(x[e]) < lim;
            some += __popcll(__ballot(x[e] != 0.f));
            small += __popcll(__ballot(low));
            const float z = low ? x[e] * up * inv : 0.f;
            squares = fmaf(z, z, squares);
        }
    };
    auto put = [&](int p, float4 a, float least) {
        if (p >= pieces) return;
        const float x[4] = {a.x, a.y, a.z, a.w};
        unsigned d[3] = {0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float y = rintf(x[e] * up * inv);
            if (bad || fabsf(x[e]) < least) y = 0.f;
            const unsigned n = ((unsigned)(int)y + 0x808080u) ^ 0x808080u;          // bytes = signed digits, carries taken along
            d[0] |= (n & 0xffu) << (8 * e);
            d[1] |= ((n >> 8) & 0xffu) << (8 * e);
            d[2] |= ((n >> 16) & 0xffu) << (8 * e);
        }
        const int i = p & 15;
        signed char* o = out + ((tb * chunks + c0 + (p >> 4)) * 3) * 1024 + ((i >> 2) * 16 + r) * 16 + (i & 3) * 4;
#pragma unroll
        for (int g = 0; g < 3; g++) *reinterpret_cast<unsigned*>(o + g * 1024) = d[g];
    };
    // (digits of all values first, which hides the weighing; those of a wide run again)
#pragma unroll
    for (int j = 0; j < FG_PIECES; j++)
        if (64 * j < pieces) { weigh(v[j]); put(lane + 64 * j, v[j], 0.f); }
    for (int p = 64 * FG_PIECES; p < pieces; p += 64) { const float4 a = get(p + lane); weigh(a); put(p + lane, a, 0.f); }
    squares = wave_sum(squares);
    const float f = (float)small;
    const bool isWide = !bad && small * 8 > some && (float)some * squares < FG_EVEN * f * f;
    if (lane == 0) wide[(tb * FG_WAVES + run) * 16 + r] = isWide ? 1 : 0;
    if (!isWide) return;
#pragma unroll
    for (int j = 0; j < FG_PIECES; j++) put(lane + 64 * j, v[j], lim);
    for (int p = lane + 64 * FG_PIECES; p < pieces; p += 64) put(p, get(p), lim);
}

// ---------------------------------------------------------------------------
// The product.  A workgroup = 8 waves on a tile of 16 MT rows x 16 NB weight rows, each with a run of K of its own: operands
// go from memory into the matrix instruction, only the eight waves' sums meet in LDS (few_rows.hip has the same plan).  A
// lane loads 16 bytes of row 4 Q + R / 4 of a weight block (lane = 16 Q + R), so that a quarter wave reads whole 64-byte
// pieces of rows, and the pieces change lanes.
//   LOOP = 0: runs of at most two chunks, both requested at once.
// ---------------------------------------------------------------------------
template <int MT, int NB, int LOOP>
__global__ __launch_bounds__(FG_WG) void few_gemm_kernel(FewGemmParams p) {
    constexpr int D = !LOOP || MT * NB >= 6 || MT >= 4 ? 2 : (MT * NB >= 3 ? 3 : 4);
    constexpr int NCOL = 16 * NB, MROW = 16 * MT, LST = MROW + 4;
    static_assert(NCOL * (MROW / 4) <= FG_WG, "four results a thread");
    extern __shared__ __attribute__((aligned(16))) float part[];      // [wave][column][LST]: the waves' sums
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    const int numM = (p.T + MROW - 1) / MROW;
    const int L = blockIdx.x, grp = L / (8 * numM), rem = L % (8 * numM);
    const int nTile = grp * 8 + (rem & 7), mTile = rem >> 3;          // the row tiles of a weight tile on one XCD
    if (nTile >= p.nTiles) return;
    const int m0 = mTile * MROW, r0 = nTile * NCOL, K = p.K, T = p.T, N = p.N;
    const int chunks = fg_chunks(K), per = fg_per_wave(K), whole = K >> 6;
    const int c0 = wave * per, cEnd = min(c0 + per, whole), lastChunk = few_last_chunk(K);

    const int ldRow = few_load_row(fq, fr), ldPiece = few_piece(fr, K);
    const int from = 4 * (16 * (fr >> 2) + 4 * (fr & 3) + fq);        // (bytes: ds_bpermute's lane address)
    const signed char* wP[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) wP[b] = p.W + few_piece_at(min(r0 + b * 16 + ldRow, N - 1), ldPiece, K, 0);
    const signed char* aP[MT];
    const float* sP[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        // Blocks past the last row repeat the last one, and so do rows: half a block's lines where it has eight rows or fewer (1 to 8 rows
        // 896 x 4864 9.8 -> 8.9 us a call, 9000 x 8192 30.8 -> 28.0; 20 rows 35.0 -> 32.7, 72 49.3 -> 47.3).
        const size_t tb = (size_t)min((m0 >> 4) + i, (T - 1) >> 4);
        aP[i] = p.A + tb * chunks * 3072 + (fq * 16 + min(fr, T - 1 - (int)tb * 16)) * 16;
        sP[i] = p.aScales + (tb * FG_WAVES + wave) * 16 + 4 * fq;
    }
    // what the epilogue needs, requested before the operands: this thread's column n, rows mq .. mq + 3
    const int n = tid % NCOL, mq = (tid / NCOL) * 4, row = r0 + n, rowC = min(row, N - 1);
    const bool mine = mq < min(MROW, T - m0);
    const float sc = p.scales[rowC], bi = p.bias ? p.bias[rowC] : 0.f;
    float old[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.accumulate)
#pragma unroll
        for (int e = 0; e < 4; e++) old[e] = p.Y[(size_t)min(m0 + mq + e, T - 1) * N + rowC];
    float4_t aS[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) aS[i] = *reinterpret_cast<const float4_t*>(sP[i]);
    int wides[MT];                                                    // lane = 8 run + pair of rows: whether one of the two has a wide run
#pragma unroll
    for (int i = 0; i < MT; i++)
        wides[i] = *reinterpret_cast<const unsigned short*>(p.wide + (size_t)min((m0 >> 4) + i, (T - 1) >> 4) * FG_WAVES * 16 + lane * 2);

    int4_t acc[MT][NB][3];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int d = 0; d < 3; d++) acc[i][b][d] = int4_t{0, 0, 0, 0};
    int4_t va[D][MT][3], vw[D][NB];
    auto load = [&](int c, int4_t (&a)[MT][3], int4_t (&w)[NB]) __attribute__((always_inline)) {
        const int cc = min(c, lastChunk);                             // (unconditional: a load under a branch drains the ring)
#pragma unroll
        for (int b = 0; b < NB; b++) w[b] = *reinterpret_cast<const int4_t*>(wP[b] + (size_t)cc * few_chunk_bytes(0));
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int d = 0; d < 3; d++) a[i][d] = *reinterpret_cast<const int4_t*>(aP[i] + (size_t)cc * 3072 + d * 1024);
        asm volatile("" ::: "memory");
    };
    auto multiply = [&](const int4_t (&a)[MT][3], const int4_t (&w)[NB]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            int4_t x;
#pragma unroll
            for (int e = 0; e < 4; e++) x[e] = __builtin_amdgcn_ds_bpermute(from, w[b][e]);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int d = 0; d < 3; d++) acc[i][b][d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i][d], x, acc[i][b][d], 0, 0, 0);
        }
    };
    if (!LOOP) {
        load(c0, va[0], vw[0]);
        load(c0 + 1, va[1], vw[1]);
        if (c0 < cEnd) multiply(va[0], vw[0]);
        if (c0 + 1 < cEnd) multiply(va[1], vw[1]);
    } else {
#pragma unroll
        for (int j = 0; j < D - 1; j++) load(c0 + j, va[j], vw[j]);
        for (int c = c0; c < cEnd; c += D) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                constexpr int DM = D - 1;
                load(c + j + DM, va[(j + DM) % D], vw[(j + DM) % D]);
                if (c + j < cEnd) multiply(va[j], vw[j]);
            }
        }
    }
    if ((K & 32) && wave == whole / per) {                            // the last 32 k: the digits past them are zeros, the weights any
        int4_t a[MT][3], w[NB];
#pragma unroll
        for (int b = 0; b < NB; b++)
            w[b] = *reinterpret_cast<const int4_t*>(p.W + (size_t)min(r0 + b * 16 + ldRow, N - 1) * K + (size_t)whole * 64 + (ldPiece & 1) * 16);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int d = 0; d < 3; d++) a[i][d] = *reinterpret_cast<const int4_t*>(aP[i] + (size_t)whole * 3072 + d * 1024);
        multiply(a, w);
    }

    // C layout: lane holds column fr, rows 4 fq .. 4 fq + 3 of a block
    float4_t sum[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x = fmaf((float)acc[i][b][2][e], 65536.f, fmaf((float)acc[i][b][1][e], 256.f, (float)acc[i][b][0][e]));
                sum[i][b][e] = x * fabsf(aS[i][e]);
                if (aS[i][e] < 0.f) sum[i][b][e] *= 0x1p-64f;
            }
    // Wide runs: their small values, as two bf16 terms; all waves share a run's chunks, a chunk's weights are converted once for
    // all rows of the tile (the same lane of both operands holds the same 16 k, so they go in as two halves of 8 k of every lane).
    unsigned long long runs[MT], any = 0;                             // a byte a run
#pragma unroll
    for (int i = 0; i < MT; i++) { runs[i] = __ballot(wides[i] != 0); any |= runs[i]; }
    if (any) {
        float4_t left[MT][NB];
        const float* aRow[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) {
            aRow[i] = p.act + (size_t)min(min((m0 >> 4) + i, (T - 1) >> 4) * 16 + fr, T - 1) * K;
#pragma unroll
            for (int b = 0; b < NB; b++) left[i][b] = float4_t{0.f, 0.f, 0.f, 0.f};
        }
        for (int run = 0; run < FG_WAVES; run++) {
            if (((any >> (8 * run)) & 0xff) == 0) continue;
            float lim[MT];                                            // of a row whose run is not wide no value is small
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const size_t at = ((size_t)min((m0 >> 4) + i, (T - 1) >> 4) * FG_WAVES + run) * 16 + fr;
                const float s = p.aScales[at];
                lim[i] = !p.wide[at] ? 0.f : s < 0.f ? s * -FG_KEPT * 0x1p-64f : s * FG_KEPT;
            }
            for (int c = run * per + ((wave - run * per) & (FG_WAVES - 1)); c < min(run * per + per, chunks); c += FG_WAVES) {
                const int k = c * 64 + fq * 16, kA = k < K ? k : 0;
                int4_t w[NB];
                float4_t a[2][4];                                     // a block's values, and those of the next
                auto loadA = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                    for (int e = 0; e < 4; e++) a[i & 1][e] = *reinterpret_cast<const float4_t*>(aRow[i] + kA + 4 * e);
                };
#pragma unroll
                for (int b = 0; b < NB; b++)
                    w[b] = *reinterpret_cast<const int4_t*>(c < whole ? wP[b] + (size_t)c * few_chunk_bytes(0)
                        : p.W + (size_t)min(r0 + b * 16 + ldRow, N - 1) * K + (size_t)whole * 64 + (ldPiece & 1) * 16);
                loadA(0);
                asm volatile("" ::: "memory");
                bf16x8_t x[NB][2];
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int q = __builtin_amdgcn_ds_bpermute(from, w[b][e]);
#pragma unroll
                        for (int y = 0; y < 4; y++) x[b][e >> 1][(e & 1) * 4 + y] = (__bf16)(float)(q << (24 - 8 * y) >> 24);
                    }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    if (i + 1 < MT) loadA(i + 1);
                    asm volatile("" ::: "memory");
                    if (((runs[i] >> (8 * run)) & 0xff) == 0) continue;
                    const float below = k < K ? lim[i] : 0.f;
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        bf16x8_t hi, lo;
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {                      // (pairs: one conversion for two values)
                            float2_t v;
#pragma unroll
                            for (int y = 0; y < 2; y++) {
                                const float u = a[i & 1][2 * h + (e >> 2)][(e & 3) + y];
                                v[y] = fabsf(u) < below ? u : 0.f;
                            }
                            const bf16x2_t t = __builtin_convertvector(v, bf16x2_t);
                            const unsigned bits = __builtin_bit_cast(unsigned, t);
                            v[0] -= __builtin_bit_cast(float, bits << 16);
                            v[1] -= __builtin_bit_cast(float, bits & 0xffff0000u);
                            const bf16x2_t r = __builtin_convertvector(v, bf16x2_t);
                            hi[e] = t[0]; hi[e + 1] = t[1];
                            lo[e] = r[0]; lo[e + 1] = r[1];
                        }
#pragma unroll
                        for (int b = 0; b < NB; b++) {
                            left[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, x[b][h], left[i][b], 0, 0, 0);
                            left[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, x[b][h], left[i][b], 0, 0, 0);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int b = 0; b < NB; b++) sum[i][b] += left[i][b];
    }
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
            *reinterpret_cast<float4_t*>(&part[(wave * NCOL + b * 16 + fr) * LST + i * 16 + 4 * fq]) = sum[i][b];
    __syncthreads();
    if (!mine) return;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < FG_WAVES; w++) {
        const float4_t t = *reinterpret_cast<const float4_t*>(&part[(w * NCOL + n) * LST + mq]);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += t[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int m = m0 + mq + e;
        if (row < N && m < T) p.Y[(size_t)m * N + row] = old[e] + (v[e] * sc + bi);
    }
}

template <int MT, int NB, int LOOP>
static hipError_t launch_fg(const FewGemmParams& p, hipStream_t s) {
    constexpr int bytes = FG_WAVES * 16 * NB * (16 * MT + 4) * 4;
    if (bytes > 48 * 1024) {
        static bool raised = false;                                    // (more than the default cap on dynamic LDS)
        if (!raised) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_gemm_kernel<MT, NB, LOOP>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return e;
            raised = true;
        }
    }
    const unsigned grid = (unsigned)((p.nTiles + 7) / 8 * 8) * (unsigned)((p.T + 16 * MT - 1) / (16 * MT));
    hipLaunchKernelGGL((few_gemm_kernel<MT, NB, LOOP>), dim3(grid), dim3(FG_WG), bytes, s, p);
    return hipGetLastError();
}
template <int MT, int NB>
static hipError_t launch_fg_loop(FewGemmParams& p, hipStream_t s) {
    p.nTiles = (p.N + 16 * NB - 1) / (16 * NB);
    return fg_per_wave(p.K) <= 2 ? launch_fg<MT, NB, 0>(p, s) : launch_fg<MT, NB, 1>(p, s);
}

hipError_t launch_few_gemm(const float* act, FewGemmParams& p, void* ws, size_t wsBytes, hipStream_t s) {
    if (p.T <= 0 || p.N <= 0) return hipSuccess;
    if (p.K <= 0 || p.K % 32 || !few_gemm_sums_fit(p.K) || few_gemm_bytes(p.T, p.K) > wsBytes || ((uintptr_t)act & 15) || ((uintptr_t)p.W & 15) || ((uintptr_t)ws & 15)) return hipErrorInvalidValue;
    const unsigned tb = (unsigned)((p.T + 15) / 16);
    signed char* digits = static_cast<signed char*>(ws);
    float* scales = reinterpret_cast<float*>(digits + (size_t)tb * fg_chunks(p.K) * 3072);
    unsigned char* wide = reinterpret_cast<unsigned char*>(scales + (size_t)tb * FG_WAVES * 16);
    hipLaunchKernelGGL(few_digits_kernel, dim3(tb * 4, FG_WAVES), dim3(WG), 0, s, act, digits, scales, wide, p.T, p.K);
    p.act = act; p.A = digits; p.aScales = scales; p.wide = wide;
    // The tile (few_rows.hip's model without conversions): a workgroup's bytes at 80 a nanosecond and the sums it exchanges,
    // times the workgroups of the busiest CU, a quarter of which overlap evenly over the chip.  Against every tile in turn, 8
    // to 500 rows, twelve shapes: the best or within 6 % of it (77 x 5632 x 2048: 13.9 us, the best 13.1, the others 16 to 24).
    const int b16 = (int)tb;
    int mt = 1, nb = 1;
    double least = 1e30;
    for (int b = 1; b <= 8; b *= 2)
        for (int m = 1; m <= 4 && m <= b16 && m * b <= 8; m++) {
            const double wgs = (double)((p.N + 16 * b - 1) / (16 * b)) * ((b16 + m - 1) / m);
            const double each = (48.0 * m + 16.0 * b) * p.K / 80.0 + 25.0 * m * b;
            const double cost = (0.75 * ceil(wgs / 256.0) + 0.25 * wgs / 256.0) * each;
            if (cost < least) { least = cost; mt = m; nb = b; }
        }
#define FG_CASE(M, B) case M * 10 + B: return launch_fg_loop<M, B>(p, s)
    switch (mt * 10 + nb) {
        FG_CASE(1, 1); FG_CASE(2, 1); FG_CASE(3, 1); FG_CASE(4, 1); FG_CASE(1, 2); FG_CASE(2, 2); FG_CASE(3, 2); FG_CASE(4, 2);
        FG_CASE(1, 4); FG_CASE(2, 4); FG_CASE(1, 8);
    }
#undef FG_CASE
    return hipErrorInvalidValue;
}

}  // namespace mg
