// few_rows.h -- launchers of the few-row prefill kernels (few_rows.hip): a handful of positions through the layers.
#pragma once
#include <hip/hip_runtime.h>
#include "few_rules.h"

namespace mg {

struct FewSeg { const signed char* W; const float* scales; const float* bias; float* Y; int N; };
struct FewParams {
    FewSeg seg[3];
    const unsigned short* Ahi;       // split activations in the order few_rows.hip describes (for this launch's weight format)
    const unsigned short* Alo;
    const unsigned short* Ax;        // third terms (NULL: two terms)
    int T, K;
    int q4;                          // weights: 0 = int8 rows with scales, 1 = Q4_0 in the split layout
    // the rows' RMS factor, applied to the finished sums: sumSq holds sumParts partial sums of squares of every row,
    // sumStride floats apart (NULL: no factor)
    const float* sumSq;
    int sumParts, sumStride;
    float eps;
    // FEW_RESID (optional), FEW_SWIGLU
    const float* nextGain;
    unsigned short* nextHi;
    unsigned short* nextLo;
    unsigned short* nextX;           // with Ax
    int nextQ4;                      // weight format of the projection that reads them
    float* nextSumSq;                // [tiles of the launch][sumStride]; few_rows_sum_parts of them
    // FEW_QKV
    void* Kc;
    void* Vc;
    const float* cosTab;
    const float* sinTab;
    int pos0, headDim, kvHalf;
    // filled by the launcher
    int nTiles;
};
int few_rows_sum_parts(int N, int T, int K, int q4, int terms);
// K a multiple of 32, W and the planes 16-byte aligned; FEW_QKV: headDim 64 or 128, N multiples of it.
hipError_t launch_few_rows(int mode, FewParams& p, hipStream_t s);

// Rows of the embedding table (kinds as launch_embed_rows) into x, their split times `gain` and their sums of squares
// (one part).  tokens may be pinned host memory.  ext (here and below): the plane of the third terms, or NULL.
hipError_t launch_embed_split(int kind, const void* table, const float* scales, const int* tokens, float* x, const float* gain,
                              unsigned short* hi, unsigned short* lo, unsigned short* ext, float* sumSq, int T, int dim, int vocab, int q4,
                              hipStream_t s);
// Several rows through one Q8 matrix on the integer matrix instruction (few_gemm.hip): Y[T,N] (+)= act[T,K] . W[N,K]^T *
// scales[n] (+ bias[n]).  act, W and ws 16-byte aligned, K a multiple of 32; ws: few_gemm_bytes(T, K) (few_rules.h).
struct FewGemmParams {
    const signed char* W; const float* scales; const float* bias; float* Y;
    int T, N, K, accumulate;
    // filled by the launcher
    const float* act; const signed char* A; const float* aScales; const unsigned char* wide;
    int nTiles;
};
hipError_t launch_few_gemm(const float* act, FewGemmParams& p, void* ws, size_t wsBytes, hipStream_t s);

// Causal attention of T query rows (rotated) at positions pos0 .. over the cache rows [0, pos0 + T), all products and sums
// in fp32; the result goes out as the split the output projection reads.
hipError_t launch_few_attention(const float* q, const void* Kc, const void* Vc, int kvHalf, unsigned short* hi, unsigned short* lo,
                                unsigned short* ext, int T, int pos0, int rowLimit, int dim, int kvDim, int nHeads, int nKVHeads, int headDim, int q4,
                                const FewNext* next, int nNext, int terms, hipStream_t s);

}  // namespace mg
