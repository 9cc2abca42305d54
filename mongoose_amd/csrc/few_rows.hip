// few_rows.hip -- a layer over a handful of positions (short prompts, further turns of a conversation).
//
// Up to some hundred rows a projection is bound by its weight bytes and by launch latency, not by the matrix cores: what
// counts is that every weight byte is requested once and early, by enough workgroups, and that a layer is few launches.
// A layer is five here -- norm + q|k|v + RoPE + cache rows, attention, Wo + residual, norm + gate|up + SwiGLU, down +
// residual -- where the tiled GEMMs of prefill.hip with their K splits need ten (0.5B shape, 37 rows behind 200: 78 us a
// layer before).
//
// Arithmetic is that of prefill.hip: int8 weights (Q4_0: nibble - 8) exact in bf16, activations as two bf16 terms, fp32
// accumulation on v_mfma_f32_16x16x32_bf16.  The RMS factor is applied to the finished sums: whoever produces a row of
// the hidden state also leaves its split times the next gain and, per tile, the row's sum of squares.
#include "kernels.h"
#include "prefill.h"
#include "few_rows.h"
#include "few_rules.h"
#include "device_util.h"

namespace mg {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int FR_WAVES = 8, FR_WG = 64 * FR_WAVES;
constexpr int FEW_MT3 = 2;                 // row blocks of a tile with three terms (registers)

// two floats -> two bf16, round to nearest even
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
    const float2_t f = {a, b};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(f, bf16x2_t));
}
__device__ __forceinline__ unsigned short bf16_one(float a) { return (unsigned short)(bf16_pair(a, 0.f) & 0xffffu); }
__device__ __forceinline__ float bf16_value(unsigned short h) { return __builtin_bit_cast(float, (unsigned)h << 16); }
__device__ __forceinline__ unsigned pack_exact(float lo, float hi) {      // small whole numbers: truncation is exact
    return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, hi), __builtin_bit_cast(unsigned, lo), 0x07060302u);
}
// 8 int8 -> 8 bf16
__device__ __forceinline__ bf16x8_t frag_i8(int lo, int hi) {
    uint4 u;
    u.x = pack_exact((float)(signed char)(lo), (float)(signed char)(lo >> 8));
    u.y = pack_exact((float)(signed char)(lo >> 16), (float)(lo >> 24));
    u.z = pack_exact((float)(signed char)(hi), (float)(signed char)(hi >> 8));
    u.w = pack_exact((float)(signed char)(hi >> 16), (float)(hi >> 24));
    return __builtin_bit_cast(bf16x8_t, u);
}
// the low (sh = 4) or high (sh = 0) nibbles of 8 bytes, minus 8 -> 8 bf16, sixteen times too large: a nibble in the upper half of a
// byte, its highest bit flipped, is that as a signed byte, and a signed byte converts in one instruction (two with the subtraction; Q4_0
// 0.5B shape, 200 rows 1,621 -> 1,596 us, 77 1,070 -> 1,056)
__device__ __forceinline__ bf16x8_t frag_nib16(int2 w, unsigned sh) {
    auto bytes = [&](int x) { return (int)((((unsigned)x << sh) & 0xf0f0f0f0u) ^ 0x80808080u); };
    return frag_i8(bytes(w.x), bytes(w.y));
}
// The split planes of these kernels are stored as the MFMA operand is held: per 16 rows and 64 k two steps of 1 KB, in
// each the lane's 8 values at lane * 16 bytes (lane = 16 q + row % 16), so that an operand is one contiguous load.  (Row
// by row, a lane per row, every load touches 16 lines per quarter wave: 37 rows through an 896 x 4864 matrix 19.8 us
// instead of 12.3.)  The k of a step: 16 q + 8 s .. + 7 for int8 weights, whose row then is one 16-byte load a lane, or
// 32 s + 8 q .. + 7 for Q4_0, where a step has to be one block.
__device__ __forceinline__ size_t few_index(int t, int k, int K, int q4) {
    const int kk = k & 63;
    const int s = q4 ? kk >> 5 : (kk >> 3) & 1, q = q4 ? (kk >> 3) & 3 : kk >> 4;
    return ((size_t)(t >> 4) * ((K + 63) >> 6) + (k >> 6)) * 1024 + s * 512 + (q * 16 + (t & 15)) * 8 + (k & 7);
}

// A value's terms to element o of the planes: hi + lo, and what those leave of it in a third one.
template <bool THIRD>
__device__ __forceinline__ void put_split(unsigned short* hi, unsigned short* lo, unsigned short* ext, size_t o, float a) {
    const unsigned short h = bf16_one(a);
    const float r = a - bf16_value(h);
    const unsigned short l = bf16_one(r);
    hi[o] = h;
    lo[o] = l;
    if (THIRD) ext[o] = bf16_one(r - bf16_value(l));
}

// ---------------------------------------------------------------------------
// Y[T,N] = (Ahi + Alo)[T,K] . W[N,K]^T with the mode's epilogue.  A workgroup = 8 waves that split K: wave w takes the
// 64-k chunks w, w + 8, ...; a chunk of 16 weight rows is one 16-byte load a lane (Q4_0: two of 8 bytes), a chunk of 16
// activation rows two of each plane, straight from the blocked planes into MFMA operands -- no operand is wanted by two
// waves, so nothing goes through LDS before the sums of the eight waves do.  D register sets keep D - 1 chunks of loads
// in flight a wave.
//   MT: 16-row blocks of activations, NB: 16-row blocks of weights a workgroup.
// The k of a chunk an operand's quarter (lane / 16) holds: 16 q .. 16 q + 15 in two steps of 8 (Q8), or 8 q .. 8 q + 7 of
// each of the two Q4_0 blocks -- any order serves as long as both operands have the same.
// ---------------------------------------------------------------------------
//   LOOP = 0: K of at most 16 chunks, two a wave: both are requested at once, no ring.
//   TERMS: bf16 terms of an activation, one plane each: 2 (2^-17 of the value left over), or 3 -- all 24 bits of an fp32 value,
//   so that the products are those of the decode step and only the order of the fp32 sums differs.
template <int MODE, int MT, int NB, int Q4, int LOOP, int TERMS>
__global__ __launch_bounds__(FR_WG) void few_rows_kernel(FewParams p) {
    constexpr int D = !LOOP || MT * NB >= 6 || MT == 4 || (TERMS == 3 && MT * NB >= 4) ? 2 : (MT * NB >= 3 ? 3 : 4);
    constexpr int NCOL = 16 * NB, MROW = 16 * MT, LST = MROW + 4;
    static_assert(NCOL * (MROW / 4) <= FR_WG, "four results a thread");
    extern __shared__ __attribute__((aligned(16))) float part[];      // [wave][column][LST]: the waves' sums
    __shared__ float sumq[FR_WAVES][MROW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    const int numM = (p.T + MROW - 1) / MROW;
    const int L = blockIdx.x, grp = L / (8 * numM), rem = L % (8 * numM);
    const int nTile = grp * 8 + (rem & 7), mTile = rem >> 3;          // the row tiles of a weight tile on one XCD
    if (nTile >= p.nTiles) return;
    const int m0 = mTile * MROW, K = p.K, T = p.T;
    const int mRows = min(MROW, T - m0);

    // the tile's matrix, its first row there, and the distance of its two 16-row blocks
    int sgi = 0, r0 = nTile * NCOL, blk = 16;
    int head0 = 0, jj0 = 0;                                           // FEW_QKV: first element of the head, index in the half
    if (MODE == FEW_SWIGLU) r0 = nTile * (NCOL / 2);                   // the first NB/2 blocks are gate rows, the others the same up rows
    if (MODE == FEW_QKV) {
        const int half = p.headDim >> 1, tq = p.seg[0].N >> 5, tk = p.seg[1].N >> 5;
        const int t = nTile < tq ? nTile : (nTile < tq + tk ? nTile - tq : nTile - tq - tk);
        sgi = nTile < tq ? 0 : (nTile < tq + tk ? 1 : 2);
        if (sgi == 2) r0 = t * 32;
        else {
            const int per = half >> 4;
            head0 = (t / per) * p.headDim;
            jj0 = (t % per) * 16;
            r0 = head0 + jj0;
            blk = half;
        }
    }
    FewSeg sg = p.seg[0];
    if (MODE == FEW_QKV) { if (sgi == 1) sg = p.seg[1]; if (sgi == 2) sg = p.seg[2]; }
    const int N = sg.N;

    const int chunks = K >> 6, planeChunks = (K + 63) >> 6;           // whole chunks; a last half one is multiplied after them
    const int lastChunk = few_last_chunk(K);
    // A lane's weights of a chunk: row fr of the block, 16 of its 64 bytes (Q4_0: 8 bytes of each of two blocks).  Loaded
    // like that a quarter wave touches 16 rows; so lane 16 Q + R loads piece R % 4 of row 4 Q + R / 4 instead (whole
    // rows of 64 bytes) and the pieces change lanes (ds_bpermute).
    const signed char* wP[NB];
    const unsigned short* dP[NB];
    const int ldRow = few_load_row(fq, fr), ldPiece = few_piece(fr, K);
    const int from = 4 * (16 * (fr >> 2) + 4 * (fr & 3) + (Q4 ? fq & 1 : fq));      // (bytes: ds_bpermute's lane address)
    auto blockRow = [&](int b, int i) __attribute__((always_inline)) {
        return min((MODE == FEW_SWIGLU ? r0 + (b % (NB / 2 > 0 ? NB / 2 : 1)) * 16 : r0 + b * blk) + i, N - 1);
    };
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const signed char* W = (MODE == FEW_SWIGLU && b >= NB / 2) ? p.seg[1].W : sg.W;
        wP[b] = W + few_piece_at(blockRow(b, ldRow), ldPiece, K, Q4);
        dP[b] = Q4 ? reinterpret_cast<const unsigned short*>(W + (size_t)N * (K >> 1)) + few_scales_at(blockRow(b, fr), K) : nullptr;
    }
    const size_t aBlk = (size_t)planeChunks * 1024;                   // elements from one 16-row block to the next
    const unsigned short* aP[TERMS][MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        // Blocks past the last row repeat the last one, and so do rows: half a block's lines where it has eight rows or fewer (us a call,
        // eight 1.1B layers at 3 / 20 rows 370 / 387 -> 338 / 367, four of 8B 361 / 441 -> 332 / 422, Q4_0 385 / 495 -> 356 / 475).
        const int block = min((m0 >> 4) + i, (T - 1) >> 4);
        const size_t o = (size_t)block * aBlk + (fq * 16 + min(fr, T - 1 - block * 16)) * 8;
        aP[0][i] = p.Ahi + o;
        aP[1][i] = p.Alo + o;
        if constexpr (TERMS == 3) aP[2][i] = p.Ax + o;
    }

    // What the epilogue needs is requested before the products' operands: the rows' sums of squares (for the RMS factor;
    // 64 / MROW lanes share a row's parts), and this thread's scale, bias, gain, residual rows and RoPE factors.
    constexpr int G = MT == 1 ? 4 : (MT == 2 ? 2 : 1), SQN = 4;     // (MT = 3: lanes past the rows repeat the last one)
    const int sqRow = min(m0 + (G == 1 ? lane : lane % MROW), T - 1), sq0 = wave * G + (G == 1 ? 0 : lane / MROW);
    float sqv[SQN];
#pragma unroll
    for (int j = 0; j < SQN; j++) {
        const int i = sq0 + j * FR_WAVES * G;
        sqv[j] = 0.f;
        if (p.sumSq && i < p.sumParts) sqv[j] = p.sumSq[(size_t)i * p.sumStride + sqRow];
    }
    const int n = tid % NCOL, mq = (tid / NCOL) * 4;                  // this thread's results: column n, rows mq .. mq + 3
    const int b = n >> 4, i16 = n & 15;
    const bool isUp = MODE == FEW_SWIGLU && n >= NCOL / 2;
    const int row = MODE == FEW_SWIGLU ? r0 + n % (NCOL / 2) : r0 + b * blk + i16;      // row of the weight matrix = column of the result
    const bool okN = row < N, mine = mq < mRows;
    const float* scales = isUp ? p.seg[1].scales : sg.scales;
    const int rowC = min(row, N - 1);
    const float sc = Q4 ? 0.0625f : scales[rowC], bi = (MODE != FEW_SWIGLU && sg.bias) ? sg.bias[rowC] : 0.f;
    float gain = 1.0f, old[4] = {0.f, 0.f, 0.f, 0.f}, cs[4], sn[4];
    if (MODE == FEW_RESID) {
        if (p.nextGain) gain = p.nextGain[rowC];
#pragma unroll
        for (int e = 0; e < 4; e++) old[e] = sg.Y[(size_t)min(m0 + mq + e, T - 1) * N + rowC];
    }
    if (MODE == FEW_QKV) {
        const int half = p.headDim >> 1;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const size_t o = (size_t)(p.pos0 + min(m0 + mq + e, T - 1)) * half + jj0 + i16;
            cs[e] = p.cosTab[o];
            sn[e] = p.sinTab[o];
        }
    }

    // (three terms: the lower two have sums of their own, so that a sum is rounded once a step, not three times)
    constexpr bool SUMS2 = TERMS == 3 && !Q4;
    float4_t acc[MT][NB], acc2[SUMS2 ? MT : 1][SUMS2 ? NB : 1];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc[i][b][e] = 0.f;
                if constexpr (SUMS2) acc2[i][b][e] = 0.f;
            }

    uint4 va[D][TERMS][MT][2];
    int4 vw[D][NB];
    unsigned vd[D][NB];
    auto load = [&](int c, uint4 (&a)[TERMS][MT][2], int4 (&w)[NB], unsigned (&d)[NB]) __attribute__((always_inline)) {
        const int cc = min(c, lastChunk);
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (Q4) {
                const int2 x = *reinterpret_cast<const int2*>(wP[b] + cc * few_chunk_bytes(1));
                w[b] = make_int4(x.x, x.y, 0, 0);
                d[b] = (unsigned)dP[b][cc * 2] | ((unsigned)dP[b][cc * 2 + 1] << 16);
            } else {
                w[b] = *reinterpret_cast<const int4*>(wP[b] + cc * few_chunk_bytes(0));
            }
        }
        // (every load is unconditional: one under a branch, even a branch that is always taken, makes the compiler's waits
        // drain the ring; rows past T are the last one's again, and their results are dropped)
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int t = 0; t < TERMS; t++) a[t][i][s] = *reinterpret_cast<const uint4*>(aP[t][i] + cc * 1024 + s * 512);
        asm volatile("" ::: "memory");                                // (the loads stay here, ahead of the products before them)
    };
    // a 32-k step: weight fragments f (Q4_0: block scales d) against activation blocks
    auto product = [&](const bf16x8_t (&f)[NB], const float (&d)[NB], int i, const uint4 (&a)[TERMS]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (Q4) {
                // a Q4_0 block's sum, then its fp16 scale (not foldable into a bf16 weight without loss)
                float4_t t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < TERMS; k++) t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[k]), f[b], t, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) acc[i][b][e] = fmaf(d[b], t[e], acc[i][b][e]);
            } else {
#pragma unroll
                for (int k = 0; k < TERMS; k++) {
                    float4_t& sum = SUMS2 && k > 0 ? acc2[SUMS2 ? i : 0][SUMS2 ? b : 0] : acc[i][b];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[k]), f[b], sum, 0, 0, 0);
                }
            }
        }
    };
    auto multiply = [&](const uint4 (&a)[TERMS][MT][2], const int4 (&w)[NB], const unsigned (&d)[NB]) __attribute__((always_inline)) {
        int4 x[NB];                                                   // this lane's own pieces
#pragma unroll
        for (int b = 0; b < NB; b++) {
            x[b].x = __builtin_amdgcn_ds_bpermute(from, w[b].x);
            x[b].y = __builtin_amdgcn_ds_bpermute(from, w[b].y);
            x[b].z = __builtin_amdgcn_ds_bpermute(Q4 ? from + 8 : from, Q4 ? w[b].x : w[b].z);      // (Q4_0: pieces 2 and 3 are the second block)
            x[b].w = __builtin_amdgcn_ds_bpermute(Q4 ? from + 8 : from, Q4 ? w[b].y : w[b].w);
        }
#pragma unroll
        for (int s = 0; s < 2; s++) {
            bf16x8_t f[NB];
            float dd[NB];
#pragma unroll
            for (int b = 0; b < NB; b++) {
                f[b] = Q4 ? frag_nib16(s ? make_int2(x[b].z, x[b].w) : make_int2(x[b].x, x[b].y), fq >= 2 ? 0u : 4u)
                          : frag_i8(s ? x[b].z : x[b].x, s ? x[b].w : x[b].y);
                dd[b] = Q4 ? half_bits_to_float((unsigned short)(s ? d[b] >> 16 : d[b] & 0xffffu)) : 1.0f;
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                uint4 at[TERMS];
#pragma unroll
                for (int t = 0; t < TERMS; t++) at[t] = a[t][i][s];
                product(f, dd, i, at);
            }
        }
    };
    if (!LOOP) {
        load(wave, va[0], vw[0], vd[0]);
        load(wave + FR_WAVES, va[1], vw[1], vd[1]);
        if (wave < chunks) multiply(va[0], vw[0], vd[0]);
        if (wave + FR_WAVES < chunks) multiply(va[1], vw[1], vd[1]);
    } else {
#pragma unroll
        for (int j = 0; j < D - 1; j++) load(wave + j * FR_WAVES, va[j], vw[j], vd[j]);
        for (int c = wave; c < chunks; c += D * FR_WAVES) {
#pragma unroll
            for (int j = 0; j < D; j++) {
                constexpr int DM = D - 1;
                load(c + (j + DM) * FR_WAVES, va[(j + DM) % D], vw[(j + DM) % D], vd[(j + DM) % D]);
                if (c + j * FR_WAVES < chunks) multiply(va[j], vw[j], vd[j]);
            }
        }
    }

    if ((K & 32) && wave == (chunks & (FR_WAVES - 1))) {              // the last 32 k: 8 a quarter
        bf16x8_t f[NB];
        float dd[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (Q4) {
                const signed char* W = (MODE == FEW_SWIGLU && b >= NB / 2) ? p.seg[1].W : sg.W;
                f[b] = frag_nib16(*reinterpret_cast<const int2*>(W + (size_t)blockRow(b, fr) * (K >> 1) + chunks * 32 + (fq & 1) * 8), fq >= 2 ? 0u : 4u);
                dd[b] = half_bits_to_float(dP[b][chunks * 2 + few_own_scale(K)]);
            } else {
                const signed char* W = (MODE == FEW_SWIGLU && b >= NB / 2) ? p.seg[1].W : sg.W;
                const int2 x = *reinterpret_cast<const int2*>(W + (size_t)blockRow(b, fr) * K + chunks * 64 + 8 * fq);
                f[b] = frag_i8(x.x, x.y);
                dd[b] = 1.0f;
            }
        }
        const int at = chunks * 1024 + (Q4 ? 0 : (fq & 1) * 512 + ((fq >> 1) - fq) * 128);      // k = 8 q .. 8 q + 7
#pragma unroll
        for (int i = 0; i < MT; i++) {
            uint4 a[TERMS];
#pragma unroll
            for (int t = 0; t < TERMS; t++) a[t] = *reinterpret_cast<const uint4*>(aP[t][i] + at);
            product(f, dd, i, a);
        }
    }

    // C layout: lane holds column fr, rows 4 fq .. 4 fq + 3 of a block
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            float4_t v = acc[i][b];
            if constexpr (SUMS2) v += acc2[i][b];
            *reinterpret_cast<float4_t*>(&part[(wave * NCOL + b * 16 + fr) * LST + i * 16 + 4 * fq]) = v;
        }
    {
        float sq = (sqv[0] + sqv[1]) + (sqv[2] + sqv[3]);
        if (p.sumSq)
            for (int i = sq0 + SQN * FR_WAVES * G; i < p.sumParts; i += FR_WAVES * G) sq += p.sumSq[(size_t)i * p.sumStride + sqRow];
        if (G == 4) sq = rows_sum(sq);
        if (G == 2) sq += __shfl_xor(sq, 32, 64);
        if (lane < MROW) sumq[wave][lane] = sq;
    }
    __syncthreads();
    if (NB < 8 && !mine) return;                                      // (NB = 8: 128 columns x 16 rows, all threads have results)
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < FR_WAVES; w++) {
        const float4_t t = *reinterpret_cast<const float4_t*>(&part[(w * NCOL + n) * LST + mq]);
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] += t[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        float rs = 1.0f;
        if (p.sumSq) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < FR_WAVES; w++) t += sumq[w][mq + e];
            rs = 1.0f / sqrtf(t / (float)K + p.eps);
        }
        v[e] = v[e] * sc * rs + bi;
    }
    if (MODE == FEW_RESID) {
        float q2[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = m0 + mq + e;
            q2[e] = 0.f;
            if (okN && m < T) {
                const float x = old[e] + v[e];
                sg.Y[(size_t)m * N + row] = x;
                q2[e] = x * x;
                if (p.nextHi) {
                    const float a = x * gain;
                    put_split<TERMS == 3>(p.nextHi, p.nextLo, p.nextX, few_index(m, row, N, p.nextQ4), a);
                }
            }
        }
        if (p.nextSumSq) {
            // the tile's share of the rows' sums of squares: over the 16 lanes of a block, then the blocks
#pragma unroll
            for (int e = 0; e < 4; e++) {
                q2[e] = row_sum16(q2[e]);
                if (NB >= 2) q2[e] += __shfl_xor(q2[e], 16, 64);
                if (NB == 4) q2[e] += __shfl_xor(q2[e], 32, 64);
            }
            if (n == 0)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (m0 + mq + e < T) p.nextSumSq[(size_t)nTile * p.sumStride + m0 + mq + e] = q2[e];
        }
    } else if (MODE == FEW_SWIGLU) {
        // the up value of a gate value's column is NCOL / 2 threads away: in the wave, or (64 columns of each) in the next
        float up[4];
        if (NB < 8) {
#pragma unroll
            for (int e = 0; e < 4; e++) up[e] = __shfl_xor(v[e], NCOL / 2, 64);
        } else {
            __syncthreads();                                          // (all sums are read; every thread is here: see `mine`)
            *reinterpret_cast<float4_t*>(&part[(n * (MROW / 4) + mq / 4) * 4]) = float4_t{v[0], v[1], v[2], v[3]};
            __syncthreads();
            const float4_t t = *reinterpret_cast<const float4_t*>(&part[((n ^ (NCOL / 2)) * (MROW / 4) + mq / 4) * 4]);
#pragma unroll
            for (int e = 0; e < 4; e++) up[e] = t[e];
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float u = up[e];
            const int m = m0 + mq + e;
            if (!isUp && okN && m < T) {
                const float g = v[e];
                const float a = g * (1.0f / (1.0f + expf(-g))) * u;          // mongoose.cu:949-956
                put_split<TERMS == 3>(p.nextHi, p.nextLo, p.nextX, few_index(m, row, N, p.nextQ4), a);
            }
        }
    } else {
        // RoPE on the pairs (j, j + half) of q and k (mongoose.cu:991-1006): the partner is 16 lanes away
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float other = __shfl_xor(v[e], 16, 64);
            const int m = m0 + mq + e;
            if (m >= T) continue;
            const size_t pos = (size_t)(p.pos0 + m);
            float x = v[e];
            if (sgi < 2) x = b == 0 ? v[e] * cs[e] - other * sn[e] : other * sn[e] + v[e] * cs[e];
            if (sgi == 0) sg.Y[(size_t)m * N + row] = x;
            else {
                void* cache = sgi == 1 ? p.Kc : p.Vc;
                if (p.kvHalf) static_cast<_Float16*>(cache)[pos * N + row] = (_Float16)x;
                else static_cast<float*>(cache)[pos * N + row] = x;
            }
        }
    }
}

template <int MODE, int MT, int NB, int Q4, int LOOP, int TERMS>
static hipError_t launch_few_l(const FewParams& p, hipStream_t s) {
    constexpr int bytes = FR_WAVES * 16 * NB * (16 * MT + 4) * 4;
    if (bytes > 48 * 1024) {
        static bool raised = false;                                    // (more than the default cap on dynamic LDS)
        if (!raised) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_rows_kernel<MODE, MT, NB, Q4, LOOP, TERMS>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return e;
            raised = true;
        }
    }
    const int numM = (p.T + 16 * MT - 1) / (16 * MT);
    const unsigned grid = (unsigned)((p.nTiles + 7) / 8 * 8) * (unsigned)numM;
    hipLaunchKernelGGL((few_rows_kernel<MODE, MT, NB, Q4, LOOP, TERMS>), dim3(grid), dim3(FR_WG), bytes, s, p);
    return hipGetLastError();
}

template <int MODE, int MT, int NB, int Q4>
static hipError_t launch_few_t(const FewParams& p, hipStream_t s) {
    if constexpr (MT <= FEW_MT3)
        if (p.Ax) return p.K <= 64 * 2 * FR_WAVES ? launch_few_l<MODE, MT, NB, Q4, 0, 3>(p, s) : launch_few_l<MODE, MT, NB, Q4, 1, 3>(p, s);
    if (p.Ax) return hipErrorInvalidValue;
    return p.K <= 64 * 2 * FR_WAVES ? launch_few_l<MODE, MT, NB, Q4, 0, 2>(p, s) : launch_few_l<MODE, MT, NB, Q4, 1, 2>(p, s);
}

// The tile of a launch (16 MT activation rows x 16 NB weight rows a workgroup): the one with the shortest time by a model of
// a workgroup's nanoseconds -- the bytes it pulls (a CU gets some 80 a nanosecond, whether they come from its L2 or from
// beyond it), the weights it converts (no other workgroup's conversions serve it: a Q4_0 weight costs four int8 ones), its
// matrix instructions, the sums it exchanges -- times the workgroups of the busiest CU, a fifth of which overlap evenly over the
// chip.  A launch is made up to a multiple of eight weight tiles, and those count: they end at once, but until then another CU has
// two workgroups (Q4_0 0.5B shape, down at 400 rows: 252 workgroups of 3 x 2, 288 launched, 11 us longer than 196 of 4 x 2).  Short rows
// go through two workgroups a CU at once; tiles of more than four blocks take too many registers for that (1.5), which matters where
// there are two, and 128 weight rows at any number.  The constants are a fit to every tile of gate | up, Wo and down at 16 to 512
// rows of the benchmark shapes, both formats: what it picks is within 2 % of a prefill of the best one at all but one of 160 points (8B at
// 77 rows 3 %; without matrix instructions, made-up tiles and the line at one workgroup a CU 10 %: 0.5B shape, 301 rows 1,808 -> 1,718 us, Q4_0
// 400 rows 2,642 -> 2,330).
struct FewTile { int mt, nb; };
// With three terms an activation row is half as many bytes again, and a tile has at most FEW_MT3 row blocks.
static double few_tile_cost(int rowsN, int T, int K, int nbFirst, int nbLast, int q4, int terms, FewTile& best) {
    const int b16 = (T + 15) / 16;
    best = FewTile{1, nbFirst};
    double least = 1e30;
    for (int nb = nbFirst; nb <= nbLast; nb *= 2)
        for (int mt = 1; mt <= (terms == 3 ? FEW_MT3 : 4) && mt <= b16 && mt * nb <= 8; mt++) {
            const int nTiles = (rowsN + 16 * nb - 1) / (16 * nb), mTiles = (b16 + mt - 1) / mt;
            const double wgs = (double)nTiles * mTiles, launched = (double)((nTiles + 7) / 8 * 8) * mTiles;
            const double bytes = (32.0 * terms * mt + (q4 ? 9.0 : 16.0) * nb) * K;
            double each = bytes / 80.0 + (q4 ? 0.9 : 0.225) * nb * K + 0.03 * terms * mt * nb * K + 160.0 * mt * nb;
            if (K <= 64 * 2 * FR_WAVES && mt * nb > 4 && (nb > 4 || launched > 256)) each *= 1.5;
            const double cost = (0.8 * ceil(launched / 256.0) + 0.2 * wgs / 256.0) * each;
            if (cost < least) { least = cost; best = FewTile{mt, nb}; }
        }
    return least;
}
static FewTile few_tile(int rowsN, int T, int K, int nbFirst, int nbLast, int q4, int terms) {
    FewTile t;
    few_tile_cost(rowsN, T, K, nbFirst, nbLast, q4, terms, t);
    return t;
}
int few_rows_sum_parts(int N, int T, int K, int q4, int terms) {
    const int b = few_tile(N, T, K, 1, 4, q4, terms).nb;
    return (N + 16 * b - 1) / (16 * b);
}

// ---------------------------------------------------------------------------
// gate | up + SwiGLU of more rows.  few_rows_kernel reads an operand once a workgroup of at most 64 x 32 rows, all from L2: from some
// hundred rows on that is what a CU pulls (0.5B shape, 301 rows, 31 us of a layer's 72), with the matrix pipe mostly idle.  Here a
// workgroup takes BM = 64 or 128 activation rows x (64 gate + 64 up rows), eight waves as two halves of the rows x four quarters of the
// columns, and a chunk of 64 k of both operands comes through LDS, straight from memory (a ring of three, two chunks under way): 0.04 to
// 0.05 bytes a product instead of 0.14 and more.  Activations lie in LDS as the instruction holds them, weights as they are (a row's
// 16-byte pieces permuted so that 16 rows fall on different banks), converted by the wave that multiplies them.  A wave has the same 16
// columns of gate and of up, so SwiGLU stays in registers, and a tile's columns are one chunk of the down projection's input: its split
// is put together in LDS and leaves in whole lines.  Sums over K in one wave, in the order of k.  Bound by a wave's own chain in a chunk --
// LDS reads, conversions, products -- with two waves a SIMD: 64 rows 0.62 us a chunk with one workgroup on a CU, 0.50 with two (products
// 0.21, conversions 0.17), 128 rows 0.93; a ring of six changes nothing with one and keeps two from fitting (0.70), products ordered so that
// none waits for the one before 1 to 3 % slower.  Microseconds a launch: few_swiglu_rows.
//   K a multiple of 64, N K below 2^31, two terms.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned few_lds_offset(const void* p) {
    return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)(p);
}
constexpr int FS_RING = 3;
template <int Q4, int BM>
__global__ __launch_bounds__(FR_WG) void few_swiglu_kernel(FewParams p) {
    constexpr int MT = BM / 32, BLK = BM / 16, AB = BLK * 4096, WB = Q4 ? 4608 : 8192, STAGE = AB + WB, LA = BLK / 2, G = FR_WG / BM;
    extern __shared__ __attribute__((aligned(16))) float part[];
    __shared__ float sq[G][BM], rs[BM];
    unsigned char* const ring = reinterpret_cast<unsigned char*>(part);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4, wm = wave >> 2, wn = wave & 3;
    const int T = p.T, K = p.K, N = p.seg[0].N, numM = (T + BM - 1) / BM;
    const int L = blockIdx.x, grp = L / (8 * numM), rem = L % (8 * numM);
    const int nTile = grp * 8 + (rem & 7), mTile = rem >> 3;          // the row tiles of a weight tile on one XCD
    if (nTile >= p.nTiles) return;
    const int m0 = mTile * BM, n0 = nTile * 64, chunks = K >> 6;

    // what this wave brings of a chunk: LA KB of activations, a KB of weights (Q4_0: waves 0 .. 3 nibbles, 4 .. 7 block scales, twice)
    const size_t aBlk = (size_t)chunks * 1024;
    // (uniform bases, a byte offset a lane that stays)
    const int aBlock = BM == 128 ? wave : wave & 3;
    const unsigned aOff = ((unsigned)min((m0 >> 4) + aBlock, (T - 1) >> 4) * (unsigned)aBlk + lane * 8) * 2;      // (blocks past the last row repeat the last one)
    const unsigned short* const a0 = BM == 128 || wave < 4 ? p.Ahi : p.Alo;
    const unsigned aDst = aBlock * 4096 + (BM == 128 ? 0 : (wave >> 2) * 2048);
    const signed char* wBase;
    unsigned wOff, wDst;
    if (!Q4) {
        wBase = wave < 4 ? p.seg[0].W : p.seg[1].W;
        wOff = (unsigned)min(n0 + (wave & 3) * 16 + (lane >> 2), N - 1) * (unsigned)K + ((lane & 3) ^ fq) * 16;
        wDst = AB + wave * 1024;
    } else if (wave < 4) {
        wBase = wave < 2 ? p.seg[0].W : p.seg[1].W;
        wOff = (unsigned)min(n0 + (wave & 1) * 32 + (lane >> 1), N - 1) * (unsigned)(K >> 1) + ((lane & 1) ^ (fq & 1)) * 16;
        wDst = AB + wave * 1024;
    } else {
        wBase = (wave & 1 ? p.seg[1].W : p.seg[0].W) + (size_t)N * (K >> 1);
        wOff = (unsigned)min(n0 + lane, N - 1) * (unsigned)(K >> 4);
        wDst = AB + 4096 + (wave & 1) * 256;
    }
    // (written out, M0 the LDS address of the wave's first slot: the compiler's own form has every LDS read behind it wait for all loads)
    auto issue = [&](int c, int stage) __attribute__((always_inline)) {
        const int cc = min(c, chunks - 1);                            // past the end: a reload that keeps the count of loads
        const unsigned base = few_lds_offset(ring) + stage * STAGE;
#pragma unroll
        for (int t = 0; t < LA / 2; t++) {
            const unsigned short* const src = (t ? p.Alo : a0) + (size_t)cc * 1024;
            asm volatile(MG_SET_M0 "global_load_lds_dwordx4 %1, %2" : : "s"(base + aDst + t * 2048), "v"(aOff), "s"(src) : "memory");
            asm volatile(MG_SET_M0 "global_load_lds_dwordx4 %1, %2" : : "s"(base + aDst + t * 2048 + 1024), "v"(aOff), "s"(src + 512) : "memory");
        }
        if (Q4 && wave >= 4) asm volatile(MG_SET_M0 "global_load_lds_dword %1, %2" : : "s"(base + wDst), "v"(wOff), "s"(wBase + (size_t)cc * 4) : "memory");
        else asm volatile(MG_SET_M0 "global_load_lds_dwordx4 %1, %2" : : "s"(base + wDst), "v"(wOff), "s"(wBase + (size_t)cc * (Q4 ? 32 : 64)) : "memory");
    };
#pragma unroll
    for (int c = 0; c < FS_RING - 1; c++) issue(c, c);

    // the rows' RMS factors
    {
        const int row = tid % BM, g = tid / BM, t = min(m0 + row, T - 1);
        float v = 0.f;
        if (p.sumSq)
#pragma unroll 4
            for (int i = g; i < p.sumParts; i += G) v += p.sumSq[(size_t)i * p.sumStride + t];
        sq[g][row] = v;
        __syncthreads();
        if (tid < BM) {
            float x = 0.f;
#pragma unroll
            for (int j = 0; j < G; j++) x += sq[j][tid];
            rs[tid] = p.sumSq ? 1.0f / sqrtf(x / (float)K + p.eps) : 1.0f;
        }
    }
    const int col = n0 + wn * 16 + fr, colC = min(col, N - 1);
    const float scG = Q4 ? 0.0625f : p.seg[0].scales[colC], scU = Q4 ? 0.0625f : p.seg[1].scales[colC];

    float4_t acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < 2; b++) acc[i][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int stage) __attribute__((always_inline)) {
        const unsigned char* const A = ring + stage * STAGE + wm * (MT * 4096) + lane * 16;
        const unsigned char* const W = ring + stage * STAGE + AB;
        bf16x8_t f[2][2];
        unsigned d[2] = {0, 0};
#pragma unroll
        for (int b = 0; b < 2; b++) {
            if (!Q4) {
                const int4 x = *reinterpret_cast<const int4*>(W + (b * 4 + wn) * 1024 + fr * 64 + (fq ^ (fr >> 2)) * 16);
                f[b][0] = frag_i8(x.x, x.y);
                f[b][1] = frag_i8(x.z, x.w);
            } else {
#pragma unroll
                for (int s = 0; s < 2; s++)
                    f[b][s] = frag_nib16(*reinterpret_cast<const int2*>(W + (b * 4 + wn) * 512 + fr * 32 + (s ^ (fr >> 3)) * 16 + (fq & 1) * 8), fq >= 2 ? 0u : 4u);
                d[b] = *reinterpret_cast<const unsigned*>(W + 4096 + b * 256 + (wn * 16 + fr) * 4);
            }
        }
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const bf16x8_t hi = *reinterpret_cast<const bf16x8_t*>(A + i * 4096 + s * 1024);
                const bf16x8_t lo = *reinterpret_cast<const bf16x8_t*>(A + i * 4096 + 2048 + s * 1024);
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    if (Q4) {
                        // a Q4_0 block's sum, then its fp16 scale
                        float4_t t = {0.f, 0.f, 0.f, 0.f};
                        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, f[b][s], t, 0, 0, 0);
                        t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, f[b][s], t, 0, 0, 0);
                        const float dd = half_bits_to_float((unsigned short)(s ? d[b] >> 16 : d[b] & 0xffffu));
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][b][e] = fmaf(dd, t[e], acc[i][b][e]);
                    } else {
                        acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, f[b][s], acc[i][b], 0, 0, 0);
                        acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, f[b][s], acc[i][b], 0, 0, 0);
                    }
                }
            }
    };
    int stage = 0;
    for (int c = 0; c < chunks; c++) {
        // chunk c has landed (of what is under way only chunk c + 1's loads are younger), and nobody reads chunk c - 1 any more
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((FS_RING - 2) * (LA + 1)) : "memory");
        const int s2 = stage == 0 ? FS_RING - 1 : stage - 1;
        issue(c + FS_RING - 1, s2);
        multiply(stage);
        stage = stage + 1 == FS_RING ? 0 : stage + 1;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");      // the ring is nobody's any more

    // C layout: lane holds column fr, rows 4 fq .. 4 fq + 3 of a block
    unsigned short* const out = reinterpret_cast<unsigned short*>(part);      // [plane][block][1024], as few_index has a block's chunk
    const int kk = wn * 16 + fr, slot = (p.nextQ4 ? (kk >> 5) * 512 + ((kk >> 3) & 3) * 128 : ((kk >> 3) & 1) * 512 + (kk >> 4) * 128) + (kk & 7);
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int blk = wm * MT + i, t = 4 * fq + e;
            const float r = rs[blk * 16 + t];
            const float g = acc[i][0][e] * scG * r, u = acc[i][1][e] * scU * r;
            const float a = g * (1.0f / (1.0f + expf(-g))) * u;      // mongoose.cu:949-956
            put_split<false>(out, out + BLK * 1024, nullptr, (size_t)(blk * 1024 + slot + t * 8), a);
        }
    __syncthreads();
    const size_t o0 = (size_t)(m0 >> 4) * ((N + 63) >> 6) * 1024 + (size_t)nTile * 1024;
#pragma unroll
    for (int j = 0; j < 2 * BLK * 128 / FR_WG; j++) {
        const int x = tid + j * FR_WG, plane = x / (BLK * 128), blk = x / 128 % BLK, piece = x & 127;
        const int s = piece >> 6, q = (piece >> 4) & 3, k0 = n0 + (p.nextQ4 ? 32 * s + 8 * q : 16 * q + 8 * s);
        if (k0 >= N || m0 + blk * 16 + (piece & 15) >= T) continue;
        const uint4 v = *reinterpret_cast<const uint4*>(out + (size_t)x * 8);
        *reinterpret_cast<uint4*>((plane ? p.nextLo : p.nextHi) + o0 + (size_t)blk * ((N + 63) >> 6) * 1024 + piece * 8) = v;
    }
}

template <int Q4, int BM>
static hipError_t launch_few_swiglu(FewParams& p, hipStream_t s) {
    constexpr int bytes = FS_RING * (BM / 16 * 4096 + (Q4 ? 4608 : 8192));
    static bool raised = false;                                        // (more than the default cap on dynamic LDS)
    if (!raised) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_swiglu_kernel<Q4, BM>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        if (e != hipSuccess) return e;
        raised = true;
    }
    p.nTiles = (p.seg[0].N + 63) / 64;
    const unsigned grid = (unsigned)((p.nTiles + 7) / 8 * 8) * (unsigned)((p.T + BM - 1) / BM);
    hipLaunchKernelGGL((few_swiglu_kernel<Q4, BM>), dim3(grid), dim3(FR_WG), bytes, s, p);
    return hipGetLastError();
}
// 0: gate | up of T rows is few_rows_kernel's; else the activation rows of a workgroup's tile in few_swiglu_kernel.  The least of three
// models in microseconds: few_tile's, and for tiles of 64 and 128 rows a start and end and so much a chunk of 64 k, times the
// workgroups of the busiest CU (of 64 rows two run on it together and hide each other's waits).  Fitted to the launches of five
// shapes at 16 to 1,000 rows; what it picks is within 6 % of the best at all but three of 114 points (9, 12 and 15 %), and none of it is slower than
// few_rows_kernel.  Microseconds a launch, old / 64 / 128 rows, Q8 and Q4_0: 0.5B shape 77 rows 12.6 / 14.8 / 20.3 and 15.0 / 17.0 / 24.0, 301 31.6 / 20.7 / 21.5 and 36.0 / 24.6 / 24.8, 512 47.0 /
// 29.1 / 37.3 and 51.8 / 33.7 / 43.3; 1.1B 64 rows 19.1 / 23.0 / 34.2 and 27.7 / 27.6 / 42.8, 200 41.1 / 34.9 / 35.0 and 58.2 / 43.4 / 42.6; 8B
// 16 rows 32.4 / 46.1 / 71.0, 37 62.8 / 42.6 / 63.0, 128 109.5 / 69.8 / 67.6, Q4_0 144.1 / 87.0 / 83.0.
static int few_swiglu_rows(int N, int T, int K, int q4, int terms) {
    if (terms != 2 || K % 64 || (long long)N * K >= 1LL << 31) return 0;      // (offsets in 32 bits)
    FewTile t;
    const double cost = 1e-3 * few_tile_cost(2 * N, T, K, 2, 8, q4, terms, t), chunks = K / 64;
    const double old = q4 && K <= 64 * 2 * FR_WAVES ? 6.0 + 0.7 * cost : 4.0 + 0.9 * cost;
    const int launched = ((N + 63) / 64 + 7) / 8 * 8;
    auto busiest = [&](int bm) { return (launched * ((T + bm - 1) / bm) + 255) / 256; };
    const int c64 = busiest(64), c128 = busiest(128);
    const double t64 = c64 == 1 ? (q4 ? 6.5 + 0.75 * chunks : 5.5 + 0.62 * chunks) : 7.0 + (q4 ? 0.61 : 0.50) * chunks * c64;
    const double t128 = 7.0 + (q4 ? 1.18 : 0.93) * chunks * c128;
    if (old <= t64 && old <= t128) return 0;
    return t64 <= t128 ? 64 : 128;
}

template <int MODE, int MT, int NB>
static hipError_t launch_few_fmt(const FewParams& p, hipStream_t s) {
    return p.q4 ? launch_few_t<MODE, MT, NB, 1>(p, s) : launch_few_t<MODE, MT, NB, 0>(p, s);
}
template <int MODE, int NB>
static hipError_t launch_few_mt(int mt, const FewParams& p, hipStream_t s) {
    if (mt == 1) return launch_few_fmt<MODE, 1, NB>(p, s);
    if constexpr (NB <= 4)
        if (mt == 2) return launch_few_fmt<MODE, 2, NB>(p, s);
    if constexpr (NB <= 2) {
        if (mt == 3) return launch_few_fmt<MODE, 3, NB>(p, s);
        if (mt == 4) return launch_few_fmt<MODE, 4, NB>(p, s);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_few_rows(int mode, FewParams& p, hipStream_t s) {
    if (p.T <= 0) return hipSuccess;
    if (p.K <= 0 || p.K % 32 || !p.Ahi || !p.Alo || p.seg[0].N <= 0) return hipErrorInvalidValue;
    const int terms = p.Ax ? 3 : 2;
    if (terms == 3 && p.nextHi && !p.nextX) return hipErrorInvalidValue;
    const int N = p.seg[0].N;
    if (mode == FEW_RESID) {
        const FewTile t = few_tile(N, p.T, p.K, 1, 4, p.q4, terms);
        p.nTiles = (N + 16 * t.nb - 1) / (16 * t.nb);
        return t.nb == 1 ? launch_few_mt<FEW_RESID, 1>(t.mt, p, s) : t.nb == 2 ? launch_few_mt<FEW_RESID, 2>(t.mt, p, s) : launch_few_mt<FEW_RESID, 4>(t.mt, p, s);
    }
    if (mode == FEW_SWIGLU) {
        if (p.seg[1].N != N || !p.nextHi || !p.nextLo) return hipErrorInvalidValue;
        const int bm = few_swiglu_rows(N, p.T, p.K, p.q4, terms);
        if (bm == 64) return p.q4 ? launch_few_swiglu<1, 64>(p, s) : launch_few_swiglu<0, 64>(p, s);
        if (bm == 128) return p.q4 ? launch_few_swiglu<1, 128>(p, s) : launch_few_swiglu<0, 128>(p, s);
        const FewTile t = few_tile(2 * N, p.T, p.K, 2, 8, p.q4, terms);
        p.nTiles = (N + 8 * t.nb - 1) / (8 * t.nb);
        return t.nb == 2 ? launch_few_mt<FEW_SWIGLU, 2>(t.mt, p, s) : t.nb == 4 ? launch_few_mt<FEW_SWIGLU, 4>(t.mt, p, s) : launch_few_mt<FEW_SWIGLU, 8>(t.mt, p, s);
    }
    if (mode == FEW_QKV) {
        if ((p.headDim != 64 && p.headDim != 128) || N % p.headDim || p.seg[1].N <= 0 || p.seg[1].N % p.headDim ||
            p.seg[2].N != p.seg[1].N || !p.Kc || !p.Vc) return hipErrorInvalidValue;
        p.nTiles = (N + 2 * p.seg[1].N) / 32;
        return launch_few_mt<FEW_QKV, 2>(few_tile(N + 2 * p.seg[1].N, p.T, p.K, 2, 2, p.q4, terms).mt, p, s);
    }
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// Embedding rows, their split times the first gain, their sums of squares: one workgroup a row.  Rows of up to EV * 256
// elements have all of their loads under way at once.
// ---------------------------------------------------------------------------
constexpr int EV = 8;
__global__ __launch_bounds__(WG) void embed_split_kernel(int kind, const void* table, const float* scales, const int* tokens, float* x,
                                                         const float* gain, unsigned short* hi, unsigned short* lo, unsigned short* ext, float* sumSq,
                                                         int dim, int vocab, int q4) {
    __shared__ float red[4];
    const int t = blockIdx.x;
    int tok = tokens[t];
    tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
    float ss = 0.f;
    for (int i0 = threadIdx.x; i0 < dim; i0 += EV * WG) {
        float v[EV], g[EV];
#pragma unroll
        for (int j = 0; j < EV; j++) {
            const int i = min(i0 + j * WG, dim - 1);
            v[j] = embed_value(kind, table, scales, tok, dim, vocab, i);
            g[j] = gain[i];
        }
#pragma unroll
        for (int j = 0; j < EV; j++) {
            const int i = i0 + j * WG;
            if (i >= dim) continue;
            x[(size_t)t * dim + i] = v[j];
            ss += v[j] * v[j];
            const size_t o = few_index(t, i, dim, q4);
            if (ext) put_split<true>(hi, lo, ext, o, v[j] * g[j]);
            else put_split<false>(hi, lo, ext, o, v[j] * g[j]);
        }
    }
    ss = block_sum(ss, red);
    if (threadIdx.x == 0) sumSq[t] = ss;
}
hipError_t launch_embed_split(int kind, const void* table, const float* scales, const int* tokens, float* x, const float* gain,
                              unsigned short* hi, unsigned short* lo, unsigned short* ext, float* sumSq, int T, int dim, int vocab, int q4,
                              hipStream_t s) {
    if (T <= 0) return hipSuccess;
    hipLaunchKernelGGL(embed_split_kernel, dim3((unsigned)T), dim3(WG), 0, s, kind, table, scales, tokens, x, gain, hi, lo, ext, sumSq, dim, vocab, q4);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Causal attention over fp32 (or fp16) cache rows in fp32, on v_mfma_f32_16x16x4_f32: no split of the operands, no pass
// over the cache rows beforehand.  A workgroup = one query head x 16 queries x 1 / CS of the output's columns; its 8
// waves take the 16-position tiles in turn, each with a running maximum / sum / output of its own, combined through LDS at the end.
//   S^T[kpos][q] = K . Q^T   A = K rows (lane: row l%16), B = Q rows; the quarter l/16 of a lane holds the head elements
//                            HD/4 * (l/16) + s, s = 0 .. HD/4 - 1, of both
//   O^T[d][q]    = V^T . P^T a lane holds S^T rows 4 (l/16) + e of its query: as the B operand of step e it is position
//                            4 (l/16) + e, which is the V row the lane loads; its elements HD/16/CS * (l%16) + b of the
//                            workgroup's columns make up row l%16 of output block b
// A prompt of a few rows has fewer (head, 16 queries) than the chip has CUs, and each is bound by its own matrix products and
// V loads.  So CS = 2 or 4 workgroups share one as long as 256 are not exceeded: all of them form the scores (half of the
// products), each a share of the columns, by the same sums.  Microseconds a layer with 1 / 2 / 4, all five launches:
//   14 heads of 64 on 2: 37 rows behind 200 37.1 / 36.1 / 35.8, behind 1,000 46.2 / 43.8 / 42.9; 128 rows 47.2 / 46.7 / 47.2
//   32 heads of 128 on 8: 16 rows behind 500 113.4 / 109.6 / 107.9; 64 behind 1,000 188.4 / 182.8 / 198.0
// and past 256 workgroups the repeated scores cost more than they save: 14 heads, 256 rows behind 1,000 76.6 / 83.8 / 98.0.
// (16 waves a workgroup: 0.3 to 1.3 us more at every size.)
// ---------------------------------------------------------------------------
template <bool KVH>
__device__ __forceinline__ float4 ld_row4(const void* base, size_t i) {
    if (!KVH) return *reinterpret_cast<const float4*>(static_cast<const float*>(base) + i);
    const uint2 u = *reinterpret_cast<const uint2*>(static_cast<const unsigned short*>(base) + i);
    return make_float4(half_bits_to_float((unsigned short)(u.x & 0xffffu)), half_bits_to_float((unsigned short)(u.x >> 16)),
                       half_bits_to_float((unsigned short)(u.y & 0xffffu)), half_bits_to_float((unsigned short)(u.y >> 16)));
}

// n consecutive cache values
template <bool KVH, int N>
__device__ __forceinline__ void ld_row(const void* base, size_t i, float (&r)[N]) {
    if constexpr (N >= 4) {
#pragma unroll
        for (int j = 0; j < N; j += 4) {
            const float4 t = ld_row4<KVH>(base, i + j);
            r[j] = t.x; r[j + 1] = t.y; r[j + 2] = t.z; r[j + 3] = t.w;
        }
    } else if constexpr (!KVH) {
#pragma unroll
        for (int j = 0; j < N; j++) r[j] = static_cast<const float*>(base)[i + j];
    } else {
#pragma unroll
        for (int j = 0; j < N; j++) r[j] = half_bits_to_float(static_cast<const unsigned short*>(base)[i + j]);
    }
}

// Reading ahead.  The attention moves few bytes and leaves most CUs idle, and the projections behind it start cold, so workgroups
// behind its own read what those multiply -- Wo, gate | up, down, in Q8 the next layer's q|k|v -- into the L2s.  These are one an XCD: tile t
// of a launch runs on XCD t mod 8 (few_rows_kernel's mapping) and is read by workgroups there, a KB a wave and instruction, into
// LDS that nothing reads.  Microseconds a call, without / with: 0.5B, 24 layers, 16 rows 811 / 722, 37 behind 200 902 / 826, 128
// 1,180 / 1,100, 301 1,908 / 1,814, 512 2,641 / 2,440; Q4_0 16 rows 807 / 780, 301 1,906 / 1,902; 1.1B, eight layers, 77 rows 559 / 542, 200
// 859 / 824; 8B, four layers, within 1 %: a layer is far more than the L2s hold.
__device__ __forceinline__ void few_read_ahead(const FewAhead& a, float* scrap) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), xcd = (int)blockIdx.x & 7;
    const unsigned nW = (unsigned)(a.readers >> 3) * FR_WAVES, me = (((int)blockIdx.x - a.first) >> 3) * FR_WAVES + wave;
#pragma unroll                       // (arguments of a launch that are indexed at run time are copied to scratch memory first)
    for (int k = 0; k < FEW_REGIONS; k++) {
        if (k < a.n) {
            const FewRegion& r = a.r[k];
            const unsigned pieces = few_ahead_pieces(r, xcd);
            for (unsigned p = me; p < pieces; p += nW)
                __builtin_amdgcn_global_load_lds(reinterpret_cast<const int4*>(r.base + few_ahead_at(r, xcd, p, lane)), reinterpret_cast<int4*>(scrap), 16, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int HD, bool KVH, int CS>
__global__ __launch_bounds__(FR_WG) void few_attention_kernel(const float* q, const void* Kc, const void* Vc, unsigned short* hi,
                                                             unsigned short* lo, unsigned short* ext, int T, int pos0, int dim, int kvDim, int nHeads,
                                                             int nKVHeads, int q4, FewAhead ahead) {
    constexpr int KF = HD / 16, VF = HD / 16 / CS;         // K: float4 a lane and row (HD/4 elements); V: elements a lane and row
    constexpr int OST = 17;
    extern __shared__ float ob[];                          // [wave][HD][OST]
    __shared__ float wm[FR_WAVES][16], wl[FR_WAVES][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fq = lane >> 4;
    if ((int)blockIdx.x >= ahead.first) { few_read_ahead(ahead, ob); return; }
    const int blocks = (T + 15) / 16, item = blockIdx.x / CS, d0 = (int)blockIdx.x % CS * (HD / CS);
    const int head = item % nHeads, q0 = (blocks - 1 - item / nHeads) * 16;    // the longest ranges first
    if (q0 < 0) return;                                    // (workgroups that make their number a multiple of 8)
    const int kvh = head / (nHeads / nKVHeads);
    const int myq = min(q0 + fr, T - 1), qpos = pos0 + myq;
    const int last = pos0 + min(q0 + 15, T - 1), nTiles = last / 16 + 1;
    const float scale = 1.0f / sqrtf((float)HD);
    float4 qf[KF];
#pragma unroll
    for (int i = 0; i < KF; i++) {
        qf[i] = *reinterpret_cast<const float4*>(q + (size_t)myq * dim + (size_t)head * HD + (HD / 4) * fq + 4 * i);
        qf[i].x *= scale; qf[i].y *= scale; qf[i].z *= scale; qf[i].w *= scale;
    }
    float4_t o[VF];
#pragma unroll
    for (int b = 0; b < VF; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) o[b][e] = 0.f;
    float m = -INFINITY, l = 0.f;
    float4 kf[2][KF];
    float vf[2][4][VF];
    auto load = [&](int t, float4 (&k)[KF], float (&v)[4][VF]) __attribute__((always_inline)) {
        const int t0 = min(t, nTiles - 1) * 16;
        // K: whole rows at a time, HD/4 lanes a row (they change lanes through LDS when they are wanted)
#pragma unroll
        for (int i = 0; i < KF; i++)
            k[i] = ld_row4<KVH>(Kc, (size_t)min(t0 + i * (256 / HD) + lane / (HD / 4), last) * kvDim + (size_t)kvh * HD + 4 * (lane % (HD / 4)));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const size_t vr = (size_t)min(t0 + 4 * fq + e, last) * kvDim + (size_t)kvh * HD + d0 + VF * fr;
            ld_row<KVH>(Vc, vr, v[e]);
        }
    };
    float* kt = ob + wave * (HD * OST);                    // this wave's K tile: 16 rows of HD + HD/16 floats
    constexpr int KST = HD + HD / 16;
    auto step = [&](int t, const float4 (&kl)[KF], const float (&v)[4][VF]) __attribute__((always_inline)) {
        float4 k[KF];
#pragma unroll
        for (int i = 0; i < KF; i++)
            *reinterpret_cast<float4*>(&kt[(i * (256 / HD) + lane / (HD / 4)) * KST + 4 * (lane % (HD / 4))]) = kl[i];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < KF; i++) k[i] = *reinterpret_cast<const float4*>(&kt[fr * KST + (HD / 4) * fq + 4 * i]);
        __builtin_amdgcn_wave_barrier();
        float4_t s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};         // two chains for the matrix pipe
#pragma unroll
        for (int i = 0; i < KF; i++) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i].x, qf[i].x, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i].y, qf[i].y, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i].z, qf[i].z, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i].w, qf[i].w, s1, 0, 0, 0);
        }
        float sv[4], tmax = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int kpos = t * 16 + 4 * fq + e;
            sv[e] = kpos <= qpos ? s0[e] + s1[e] : -INFINITY;
            tmax = fmaxf(tmax, sv[e]);
        }
        tmax = rows_max(tmax);
        const float mNew = fmaxf(m, tmax);
        const float corr = m == -INFINITY ? 0.f : exp_neg(m - mNew);
        float ps = 0.f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            sv[e] = sv[e] == -INFINITY ? 0.f : exp_neg(sv[e] - mNew);
            ps += sv[e];
        }
        l = l * corr + rows_sum(ps);
        m = mNew;
#pragma unroll
        for (int b = 0; b < VF; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) o[b][e] *= corr;
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < VF; i++) o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e][i], sv[e], o[i], 0, 0, 0);
    };
    load(wave, kf[0], vf[0]);
    for (int t = wave; t < nTiles; t += 2 * FR_WAVES) {
        load(t + FR_WAVES, kf[1], vf[1]);
        step(t, kf[0], vf[0]);
        load(t + 2 * FR_WAVES, kf[0], vf[0]);
        if (t + FR_WAVES < nTiles) step(t + FR_WAVES, kf[1], vf[1]);
    }
    __builtin_amdgcn_wave_barrier();
    // O^T of block b: lane holds query fr, rows i = 4 fq + e, i.e. head element VF * i + b
#pragma unroll
    for (int b = 0; b < VF; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) ob[(wave * HD + VF * (4 * fq + e) + b) * OST + fr] = o[b][e];
    if (fq == 0) { wm[wave][fr] = m; wl[wave][fr] = l; }
    __syncthreads();
    for (int i = tid; i < 16 * (HD / CS); i += FR_WG) {
        const int qq = i / (HD / CS), d = i % (HD / CS);
        if (q0 + qq >= T) continue;
        float M = wm[0][qq];
#pragma unroll
        for (int w = 1; w < FR_WAVES; w++) M = fmaxf(M, wm[w][qq]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < FR_WAVES; w++) {
            const float g = wm[w][qq] == -INFINITY ? 0.f : exp_neg(wm[w][qq] - M);
            num = fmaf(g, ob[(w * HD + d) * OST + qq], num);
            den = fmaf(g, wl[w][qq], den);
        }
        const float a = num / den;
        const size_t ix = few_index(q0 + qq, head * HD + d0 + d, dim, q4);
        if (ext) put_split<true>(hi, lo, ext, ix, a);
        else put_split<false>(hi, lo, ext, ix, a);
    }
}

template <int HD, bool KVH, int CS>
static hipError_t launch_few_attn_t(unsigned grid, hipStream_t s, const float* q, const void* Kc, const void* Vc, unsigned short* hi,
                                    unsigned short* lo, unsigned short* ext, int T, int pos0, int dim, int kvDim, int nHeads, int nKVHeads, int q4, FewAhead ahead) {
    constexpr int bytes = FR_WAVES * HD * 17 * 4;
    if (bytes > 48 * 1024) {
        static bool raised = false;
        if (!raised) {
            hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&few_attention_kernel<HD, KVH, CS>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return e;
            raised = true;
        }
    }
    const unsigned wgs = ahead.n ? (unsigned)(ahead.first + ahead.readers) : grid * CS;
    hipLaunchKernelGGL((few_attention_kernel<HD, KVH, CS>), dim3(wgs), dim3(FR_WG), bytes, s, q, Kc, Vc, hi, lo, ext, T, pos0, dim, kvDim, nHeads, nKVHeads, q4, ahead);
    return hipGetLastError();
}

template <int HD, bool KVH, typename... A>
static hipError_t launch_few_attn(int cs, A... a) {
    return cs == 4 ? launch_few_attn_t<HD, KVH, 4>(a...) : (cs == 2 ? launch_few_attn_t<HD, KVH, 2>(a...) : launch_few_attn_t<HD, KVH, 1>(a...));
}

hipError_t launch_few_attention(const float* q, const void* Kc, const void* Vc, int kvHalf, unsigned short* hi, unsigned short* lo,
                                unsigned short* ext, int T, int pos0, int rowLimit, int dim, int kvDim, int nHeads, int nKVHeads, int headDim, int q4, const FewNext* next,
                                int nNext, int terms, hipStream_t s) {
    if (T <= 0) return hipSuccess;
    if (nKVHeads <= 0 || nHeads % nKVHeads || pos0 < 0 || pos0 + T > rowLimit || dim != nHeads * headDim || kvDim != nKVHeads * headDim ||
        (headDim != 64 && headDim != 128) || !hi || !lo) return hipErrorInvalidValue;
    const unsigned grid = (unsigned)nHeads * (unsigned)((T + 15) / 16);
    const int cs = grid <= 64 ? 4 : (grid <= 128 ? 2 : 1);              // workgroups a head's 16 queries are shared by: see the kernel
    const FewAhead ahead = few_plan(grid * cs, next, nNext, headDim, [&](const FewNext& m) {
        if (m.mode != FEW_SWIGLU) return 16 * few_tile(m.N, T, m.K, 1, 4, m.q4, terms).nb;
        return few_swiglu_rows(m.N, T, m.K, m.q4, terms) ? 64 : 8 * few_tile(2 * m.N, T, m.K, 2, 8, m.q4, terms).nb;
    });
    if (headDim == 64) return kvHalf ? launch_few_attn<64, true>(cs, grid, s, q, Kc, Vc, hi, lo, ext, T, pos0, dim, kvDim, nHeads, nKVHeads, q4, ahead)
                                     : launch_few_attn<64, false>(cs, grid, s, q, Kc, Vc, hi, lo, ext, T, pos0, dim, kvDim, nHeads, nKVHeads, q4, ahead);
    return kvHalf ? launch_few_attn<128, true>(cs, grid, s, q, Kc, Vc, hi, lo, ext, T, pos0, dim, kvDim, nHeads, nKVHeads, q4, ahead)
                  : launch_few_attn<128, false>(cs, grid, s, q, Kc, Vc, hi, lo, ext, T, pos0, dim, kvDim, nHeads, nKVHeads, q4, ahead);
}

}  // namespace mg
