// q4_dp4a.hip -- the integer form of the Q4_0 matvec: the activation vector is quantized to int8 blocks once and the
// dot products run on the packed int8 dot instruction (v_dot4_i32_i8), as the reference's dp4a kernels do
// (kernels.go:66-70, 985-1017; dispatch cuda_fused_infer_q4.go:611-673).
//
// The reference's CUDA bodies of these kernels are not in its tree; what its Go side fixes is the calling sequence and
// the size of the scratch buffer, (K/32)*40 bytes (cuda_fused_infer.go:176): 40 bytes per block of 32 activations,
// "Q8_1 blocks" (kernels.go:993).  The block here is GGML's Q8_1 with fp32 fields:
//     float d = max|x| / 127;  float s = d * sum(q);  int8 q[32] = round-half-away(x / d)      (zero block: d = s = 0)
// and a row of block_q4_0 weights against it is GGML's vec_dot_q4_0_q8_1:
//     out[r] = sum_b  f32(d4[r,b]) * ( d8[b] * sum_i nib[r,b,i] * q[b,i]  -  8 * s8[b] )
// with nib the unsigned nibbles in GGML element order (low nibble of byte j = element j, high nibble = element j+16).
// The integer sums are exact; only the activation rounding distinguishes the result from the fp32-activation matvec.
#include "kernels.h"
#include "device_util.h"

namespace mg {

// One thread per block of 32 activations (a vector has at most a few hundred blocks, a batch a few thousand).
__global__ __launch_bounds__(WG) void q8_quantize_act_kernel(const float* __restrict__ act, unsigned char* __restrict__ out, int nBlocks) {
    const int b = blockIdx.x * WG + threadIdx.x;
    if (b >= nBlocks) return;
    const float4* x4 = reinterpret_cast<const float4*>(act + (size_t)b * 32);
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = x4[i];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) amax = fmaxf(fmaxf(fmaxf(amax, fabsf(v[i].x)), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w)));
    const float d = amax / 127.0f;
    const float id = d != 0.f ? 1.0f / d : 0.f;
    int q[8];
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int a = (int)roundf(v[i].x * id), b1 = (int)roundf(v[i].y * id), c = (int)roundf(v[i].z * id), e = (int)roundf(v[i].w * id);
        sum += a + b1 + c + e;
        q[i] = (a & 0xff) | ((b1 & 0xff) << 8) | ((c & 0xff) << 16) | ((e & 0xff) << 24);
    }
    unsigned char* o = out + (size_t)b * 40;                  // 8-byte aligned (the buffer is, and 40 is a multiple of 8)
    *reinterpret_cast<float2*>(o) = make_float2(d, d * (float)sum);
    int2* oq = reinterpret_cast<int2*>(o + 8);
#pragma unroll
    for (int i = 0; i < 4; i++) oq[i] = make_int2(q[2 * i], q[2 * i + 1]);
}

// A wave per row, a lane per block and step of 64 blocks.  PLANAR: the split layout of the context's resident matrices
// (nibble groups [N, K/32] of 16 bytes, then fp16 d [N, K/32]); otherwise raw GGUF 18-byte blocks (2-byte aligned).
// grid.y = vectors of the batch: activations q8 + y * (K/32) * 40, results out + y * N.
template <bool PLANAR>
__global__ __launch_bounds__(WG) void q4_0_dp4a_kernel(const unsigned char* __restrict__ w, const unsigned char* __restrict__ q8,
                                                       float* __restrict__ out, int N, int K) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * (WG / 64) + (threadIdx.x >> 6);
    if (r >= N) return;
    const int nb = K >> 5;
    const unsigned char* a = q8 + (size_t)blockIdx.y * nb * 40;
    float acc = 0.f;
    for (int b = lane; b < nb; b += 64) {
        unsigned x[4];
        unsigned short hd;
        if (PLANAR) {
            const uint4 g = reinterpret_cast<const uint4*>(w)[(size_t)r * nb + b];
            x[0] = g.x; x[1] = g.y; x[2] = g.z; x[3] = g.w;
            hd = reinterpret_cast<const unsigned short*>(w + (size_t)N * (K >> 1))[(size_t)r * nb + b];
        } else {
            const unsigned short* h = reinterpret_cast<const unsigned short*>(w + ((size_t)r * nb + b) * 18);
            hd = h[0];
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = (unsigned)h[1 + 2 * i] | ((unsigned)h[2 + 2 * i] << 16);
        }
        const unsigned char* ab = a + (size_t)b * 40;
        const float2 ds = *reinterpret_cast<const float2*>(ab);
        const int2* aq = reinterpret_cast<const int2*>(ab + 8);
        int qv[8];
#pragma unroll
        for (int i = 0; i < 4; i++) { const int2 t = aq[i]; qv[2 * i] = t.x; qv[2 * i + 1] = t.y; }
        int sumi = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            sumi = __builtin_amdgcn_sdot4((int)(x[i] & 0x0f0f0f0fu), qv[i], sumi, false);             // elements 4i .. 4i+3
            sumi = __builtin_amdgcn_sdot4((int)((x[i] >> 4) & 0x0f0f0f0fu), qv[4 + i], sumi, false);   // elements 16+4i .. 16+4i+3
        }
        acc += half_bits_to_float(hd) * (ds.x * (float)sumi - 8.0f * ds.y);
    }
    acc = wave_sum(acc);
    if (lane == 0) out[(size_t)blockIdx.y * N + r] = acc;
}

// Vectors against raw GGUF rows: the integer matrix instruction v_mfma_i32_16x16x32_i8, whose 32 k are a block.  A workgroup
// = 8 waves over 16 NB weight rows x 16 MT vectors, K in chunks of CH blocks, CH / 8 a wave; the waves' sums meet in LDS.
// Rows of 18-byte blocks and vectors of 40-byte ones are a poor fit for operand loads (16 rows a load: 100 cycles each), so
// a chunk is loaded along its rows, a thread a block, the next two while this one is multiplied, and passes through LDS:
// weight nibbles and scales apart, the vectors' values and scales apart, rows padded so that 16 of them meet no bank twice.
// A weight is read once per 16 MT vectors, a vector's block (from the L2) once per 16 NB rows.  Bound by its vector
// instructions, 12 per 16 x 16 sums and block for scales and fp32 sums, and at one vector by its loads.
// us with the vectors' quantization, before (a wave a row, each vector its own pass) / now: 6584 x 5920, 8 vectors 48 / 17, 48 vectors 256 / 30;
// 14336 x 4096 68 / 18 and 375 / 33; 896 x 4864 10.7 / 11.8 and 37 / 22.
// Operand lane 16 q + i: row i, eight of a block's 32 values: low nibbles of bytes 8 (q & 1) .. + 7 for q < 2, else their
// high nibbles = elements 8 q .. 8 q + 7.  Result lane 16 q + i: vector i, weight rows 4 q .. 4 q + 3. 
typedef int q4v4i __attribute__((ext_vector_type(4)));
constexpr int Q4B_WAVES = 8, Q4B_WG = 64 * Q4B_WAVES;
template <int MT, int NB, int CH>
__global__ __launch_bounds__(Q4B_WG, 4) void q4_0_batch_kernel(const unsigned char* __restrict__ w, const unsigned char* __restrict__ q8,
                                                            float* __restrict__ out, int N, int K, int T) {
    constexpr int NR = 16 * NB, TR = 16 * MT;
    constexpr int WS = CH * 4 + 4, QS = CH * 8 + 8, DS = CH * 2 + 2, HS = CH + 2;      // LDS row strides: dwords, dwords, floats, halves
    struct Stage {
        unsigned wn[NR][WS];                 // nibbles
        unsigned aq[TR][QS];                 // int8 values
        float ad[TR][DS];                    // d8, s8
        unsigned short wd[NR][HS];           // d4
    };
    __shared__ union { Stage st; float part[Q4B_WAVES][TR][NR + 1]; } sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fi = lane & 15, fq = lane >> 4;
    const int n0 = blockIdx.x * NR, t0 = blockIdx.y * TR;
    const int nb = K >> 5;
    const unsigned nsh = fq >= 2 ? 4u : 0u;
    const int tRows = min(TR, T - t0);

    // A thread's share of a chunk: weight blocks (row, block) tid, tid + 512, ...; 8-byte pieces of the vectors' rows.  Where
    // they lie and where they go is worked out once (done for every chunk it costs several times the multiplications).  A
    // chunk's blocks past the end of a row are whatever follows, inside the matrix, and are not multiplied.
    constexpr int WPT = (NR * CH + Q4B_WG - 1) / Q4B_WG, APT = (TR * CH * 5 + Q4B_WG - 1) / Q4B_WG;
    const unsigned char *wBase = w + (size_t)n0 * nb * 18, *aBase = q8 + (size_t)t0 * nb * 40;
    const unsigned wLast = (unsigned)(((long long)min(NR, N - n0) * nb - 1) * 18), aLast = (unsigned)((long long)tRows * nb * 40 - 8);
    unsigned wOff[WPT], aOff[APT], aDst[APT];
#pragma unroll
    for (int i = 0; i < WPT; i++) { const int k = tid + i * Q4B_WG; wOff[i] = (unsigned)((min(k / CH, N - n0 - 1)) * nb + k % CH) * 18u; }
#pragma unroll
    for (int i = 0; i < APT; i++) {
        const int k = tid + i * Q4B_WG, row = k / (CH * 5), pc = k % (CH * 5), b = pc / 5, part = pc % 5;
        aOff[i] = (unsigned)((row * nb + b) * 40 + part * 8);
        const char* d = part == 0 ? reinterpret_cast<const char*>(&sh.st.ad[row][b * 2]) : reinterpret_cast<const char*>(&sh.st.aq[row][b * 8 + (part - 1) * 2]);
        aDst[i] = row < tRows ? (unsigned)(d - reinterpret_cast<const char*>(&sh)) : ~0u;
    }
    struct Share { uint4 w[WPT]; unsigned short d[WPT]; uint2 a[APT]; };
    auto load = [&](Share& g, int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WPT; i++) {
            const unsigned char* p = wBase + min(wOff[i] + (unsigned)c0 * 18u, wLast);
            g.d[i] = *reinterpret_cast<const unsigned short*>(p);
            __builtin_memcpy(&g.w[i], p + 2, 16);                                  // (2-byte aligned)
        }
#pragma unroll
        for (int i = 0; i < APT; i++)
            if (aDst[i] != ~0u) g.a[i] = *reinterpret_cast<const uint2*>(aBase + min(aOff[i] + (unsigned)c0 * 40u, aLast));
    };
    auto store = [&](const Share& g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WPT; i++) {
            const int k = tid + i * Q4B_WG;
            if (NR * CH % Q4B_WG && k >= NR * CH) continue;
            *reinterpret_cast<uint4*>(&sh.st.wn[k / CH][(k % CH) * 4]) = g.w[i];
            sh.st.wd[k / CH][k % CH] = g.d[i];
        }
#pragma unroll
        for (int i = 0; i < APT; i++)
            if (aDst[i] != ~0u) *reinterpret_cast<uint2*>(reinterpret_cast<char*>(&sh) + aDst[i]) = g.a[i];
    };
    float acc[MT][NB][4];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][b][e] = 0.f;
    auto multiply = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < CH / Q4B_WAVES; h++) {
            const int j = wave + h * Q4B_WAVES;
            if (c0 + j < nb) {                                            // uniform in the wave
                long av[MT];
                float2 ds[MT];
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    av[i] = __builtin_bit_cast(long, *reinterpret_cast<const uint2*>(&sh.st.aq[i * 16 + fi][j * 8 + 2 * fq]));
                    ds[i] = *reinterpret_cast<const float2*>(&sh.st.ad[i * 16 + fi][j * 2]);
                }
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    uint2 x = *reinterpret_cast<const uint2*>(&sh.st.wn[b * 16 + fi][j * 4 + 2 * (fq & 1)]);
                    x.x = (x.x >> nsh) & 0x0f0f0f0fu;
                    x.y = (x.y >> nsh) & 0x0f0f0f0fu;
                    float d4[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) d4[e] = half_bits_to_float(sh.st.wd[b * 16 + 4 * fq + e][j]);
#pragma unroll
                    for (int i = 0; i < MT; i++) {
                        const q4v4i z = {0, 0, 0, 0};
                        const q4v4i s = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, x), av[i], z, 0, 0, 0);
                        const float m8 = -8.0f * ds[i].y;
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[i][b][e] = fmaf(d4[e], fmaf(ds[i].x, (float)s[e], m8), acc[i][b][e]);
                    }
                }
            }
        }
    };
    auto chunk = [&](Share& g, int c0) __attribute__((always_inline)) {
        if (c0) __syncthreads();                                          // the chunk before has been multiplied
        store(g);
        __syncthreads();
        load(g, c0 + 2 * CH);                                             // (past the end: the last block again)
        multiply(c0);
    };
    Share g0, g1;
    load(g0, 0);
    load(g1, CH);
    for (int c0 = 0; c0 < nb; c0 += 2 * CH) {
        chunk(g0, c0);
        if (c0 + CH < nb) chunk(g1, c0 + CH);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) sh.part[wave][i * 16 + fi][b * 16 + 4 * fq + e] = acc[i][b][e];
    __syncthreads();
    for (int k = tid; k < tRows * NR; k += Q4B_WG) {
        const int t = k / NR, n = k % NR;
        float v = 0.f;
#pragma unroll
        for (int x = 0; x < Q4B_WAVES; x++) v += sh.part[x][t][n];
        if (n0 + n < N) out[(size_t)(t0 + t) * N + n0 + n] = v;
    }
}
template <int MT>
static hipError_t launch_q4_0_batch(const void* w, const void* q8, float* out, int N, int K, int T, hipStream_t s) {
    const unsigned char *wp = static_cast<const unsigned char*>(w), *qp = static_cast<const unsigned char*>(q8);
    const int my = (T + 16 * MT - 1) / (16 * MT);
    // one or two blocks of weight rows: what the busiest CU then has to load and to multiply
    auto cost = [&](int nbk) { return (double)(((long long)((N + 16 * nbk - 1) / (16 * nbk)) * my + 255) / 256) * (1.0 + 1.8 * MT * nbk + 1.1 * MT + 2.4 * nbk); };
    if (cost(2) < cost(1)) hipLaunchKernelGGL((q4_0_batch_kernel<MT, 2, 16>), dim3((unsigned)((N + 31) / 32), (unsigned)my), dim3(Q4B_WG), 0, s, wp, qp, out, N, K, T);
    else hipLaunchKernelGGL((q4_0_batch_kernel<MT, 1, MT == 1 ? 32 : 16>), dim3((unsigned)((N + 15) / 16), (unsigned)my), dim3(Q4B_WG), 0, s, wp, qp, out, N, K, T);
    return hipGetLastError();
}

hipError_t launch_q8_quantize_act(const float* act, void* q8out, int K, int batch, hipStream_t s) {
    if (K <= 0 || K % 32 || batch <= 0 || ((uintptr_t)act & 15) || ((uintptr_t)q8out & 7)) return hipErrorInvalidValue;
    const long long nBlocks = (long long)(K / 32) * batch;
    if (nBlocks > (1ll << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(q8_quantize_act_kernel, dim3((unsigned)((nBlocks + WG - 1) / WG)), dim3(WG), 0, s, act,
                       static_cast<unsigned char*>(q8out), (int)nBlocks);
    return hipGetLastError();
}

hipError_t launch_q4_0_dp4a(const void* w, bool planar, const void* q8, float* out, int N, int K, int batch, hipStream_t s) {
    if (N <= 0 || K <= 0 || K % 32 || batch <= 0 || batch > 65535 || ((uintptr_t)q8 & 7) || ((uintptr_t)w & (planar ? 15 : 1)))
        return hipErrorInvalidValue;
    // A wave a row and a pass a vector while all of it is in flight at once (48 x 220 x 832 7.2 us against 9.5, 8 x 896 x 4864
    // 10.7 against 11.8, 27 x 896 x 896 10.4 against 8.9); the chunks of long rows follow one another, so there the line is later.
    if (!planar && batch > 3 && (double)batch * N * K > 16e6 + 5e3 * K && (long long)K / 32 * 40 * 48 < (1ll << 31))
        return batch <= 16 ? launch_q4_0_batch<1>(w, q8, out, N, K, batch, s) : batch <= 32 ? launch_q4_0_batch<2>(w, q8, out, N, K, batch, s)
                                                                                          : launch_q4_0_batch<3>(w, q8, out, N, K, batch, s);
    const dim3 grid((unsigned)((N + WG / 64 - 1) / (WG / 64)), (unsigned)batch);
    if (planar) hipLaunchKernelGGL(q4_0_dp4a_kernel<true>, grid, dim3(WG), 0, s, static_cast<const unsigned char*>(w),
                                   static_cast<const unsigned char*>(q8), out, N, K);
    else hipLaunchKernelGGL(q4_0_dp4a_kernel<false>, grid, dim3(WG), 0, s, static_cast<const unsigned char*>(w),
                            static_cast<const unsigned char*>(q8), out, N, K);
    return hipGetLastError();
}

// (max, lowest index) of contiguous slices of a vector, one per workgroup: the partials argmax_finish takes.
__global__ __launch_bounds__(WG) void argmax_slices_kernel(const float* __restrict__ x, int n, float* __restrict__ pv, int* __restrict__ pi) {
    __shared__ float sv[WG / 64];
    __shared__ int si[WG / 64];
    const int per = (n + gridDim.x - 1) / gridDim.x;
    const int i0 = blockIdx.x * per, i1 = min(n, i0 + per);
    float v = -INFINITY;
    int idx = INT_MAX;
    for (int i = i0 + threadIdx.x; i < i1; i += WG) argmax_pick(v, idx, x[i], i);
    wave_argmax(v, idx);
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = v; si[threadIdx.x >> 6] = idx; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < WG / 64; k++) argmax_pick(v, idx, sv[k], si[k]);
        pv[blockIdx.x] = v;
        pi[blockIdx.x] = idx;
    }
}
hipError_t launch_argmax_slices(const float* x, int n, int nparts, float* pv, int* pi, hipStream_t s) {
    if (n <= 0 || nparts <= 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(argmax_slices_kernel, dim3((unsigned)nparts), dim3(WG), 0, s, x, n, pv, pi);
    return hipGetLastError();
}

}  // namespace mg
