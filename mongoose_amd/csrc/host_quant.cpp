// host_quant.cpp -- host-side weight preparation for the HIP backend: the Q8
// per-row quantizer the reference runs in Go before upload, the GGML Q4_0
// block quantizer, fp16 conversion, the split-layout repack for Q4_0 rows and a
// machine-independent synthetic weight generator.  No device code.
#pragma STDC FP_CONTRACT OFF
#include "../../include/mongoose_hip.h"
#include "host_util.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#include <immintrin.h>
#endif

namespace mg {

// A fixed set of worker threads shared by every host-side loop of the library (starting threads per
// loop costs more than the per-layer staging loops themselves).  One parallel region at a time; the
// calling thread takes jobs too.  Jobs must not start a region themselves.
// Regions come in runs (matrix after matrix, layer after layer), tens of microseconds of work each, and waking fifteen
// sleeping threads takes as long: a worker keeps looking for the next region for SPIN_US before it sleeps, and the
// caller watches the count of its jobs.
class WorkPool {
    // Each parallel region has its own state object: a worker that wakes late holds the region it was
    // woken for, finds its job counter exhausted and never touches a later region's function.
    struct Region {
        const std::function<void(size_t)>* fn;
        size_t total;
        std::atomic<size_t> next{0};
        std::atomic<size_t> remaining;
    };
    static constexpr int SPIN_US = 100;

public:
    static WorkPool& get() {
        static WorkPool* pool = new WorkPool();      // lives until the process ends
        return *pool;
    }
    void run(size_t njobs, const std::function<void(size_t)>& fn, const std::function<void()>& meanwhile) {
        if (njobs <= (meanwhile ? 0u : 1u) || nWorkers == 0) {
            if (meanwhile) meanwhile();
            for (size_t j = 0; j < njobs; j++) fn(j);
            return;
        }
        std::lock_guard<std::mutex> region(regionMutex);
        auto r = std::make_shared<Region>();
        r->fn = &fn; r->total = njobs; r->remaining.store(njobs);
        bool sleeping;
        {
            std::lock_guard<std::mutex> lk(m);
            current = r;
            generation.fetch_add(1, std::memory_order_release);
            sleeping = nSleeping > 0;
        }
        if (sleeping) wake.notify_all();
        if (meanwhile) meanwhile();
        work(*r);
        if (spin([&] { return r->remaining.load(std::memory_order_acquire) == 0; })) return;
        std::unique_lock<std::mutex> lk(m);
        done.wait(lk, [&] { return r->remaining.load() == 0; });
    }

private:
    WorkPool() {
        unsigned hw = std::thread::hardware_concurrency();
        if (hw == 0) hw = 1;
        if (hw > 16) hw = 16;
        nWorkers = hw - 1;
        for (unsigned t = 0; t < nWorkers; t++) std::thread([this] { loop(); }).detach();
    }
    template <class F>
    static bool spin(F ready) {
        const auto t0 = std::chrono::steady_clock::now();
        for (;;) {
            for (int i = 0; i < 64; i++) {
                if (ready()) return true;
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
                _mm_pause();
#endif
            }
            if (std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(SPIN_US)) return false;
        }
    }
    void work(Region& r) {
        for (;;) {
            const size_t j = r.next.fetch_add(1);
            if (j >= r.total) break;
            (*r.fn)(j);
            if (r.remaining.fetch_sub(1) == 1) {
                std::lock_guard<std::mutex> lk(m);
                done.notify_all();
            }
        }
    }
    void loop() {
        unsigned long seen = 0;
        for (;;) {
            std::shared_ptr<Region> r;
            (void)spin([&] { return generation.load(std::memory_order_acquire) != seen; });
            {
                std::unique_lock<std::mutex> lk(m);
                nSleeping++;
                wake.wait(lk, [&] { return generation.load() != seen; });
                nSleeping--;
                seen = generation.load();
                r = current;
            }
            if (r) work(*r);
        }
    }
    unsigned nWorkers = 0;
    std::mutex regionMutex, m;
    std::condition_variable wake, done;
    std::shared_ptr<Region> current;
    std::atomic<unsigned long> generation{0};
    unsigned nSleeping = 0;                          // under m
};

void parallel_jobs(size_t njobs, const std::function<void(size_t)>& fn, const std::function<void()>& meanwhile) { WorkPool::get().run(njobs, fn, meanwhile); }

void parallel_for(size_t n, size_t grain, const std::function<void(size_t, size_t)>& fn) {
    if (n == 0) return;
    if (grain == 0) grain = 1;
    const size_t chunks = (n + grain - 1) / grain;
    if (chunks <= 1) { fn(0, n); return; }
    parallel_jobs(chunks, [&](size_t c) { fn(c * grain, std::min(n, (c + 1) * grain)); });
}

// Split layout read by the fast Q4_0 kernel: all 16-byte nibble groups of the
// matrix (row-major), then all fp16 block scales.  Same bytes as GGUF, only
// regrouped so that both are reachable with aligned loads.
// Into page-locked memory that only the GPU reads: where it can, with stores that go past the caches (a layer of the 0.5B
// shape, 8.4 MB, in 58 us on 16 cores instead of 90).
static void repack_plain(const uint8_t* raw, size_t b0, size_t b1, uint8_t* qs, uint8_t* d) {
    for (size_t i = b0; i < b1; i++) {
        std::memcpy(qs + i * 16, raw + i * 18 + 2, 16);
        std::memcpy(d + i * 2, raw + i * 18, 2);
    }
}
void repack_q4_0_blocks(const uint8_t* raw, size_t nb, size_t b0, size_t b1, uint8_t* planar) {
    uint8_t* qs = planar;
    uint8_t* d = planar + nb * 16;
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
    if (((uintptr_t)qs & 15) == 0 && ((uintptr_t)(d + b0 * 2) & 15) == 0) {
        for (; b0 + 8 <= b1; b0 += 8) {
            alignas(16) uint16_t h[8];
            for (int k = 0; k < 8; k++) {
                const uint8_t* r = raw + (b0 + k) * 18;
                _mm_stream_si128(reinterpret_cast<__m128i*>(qs + (b0 + k) * 16), _mm_loadu_si128(reinterpret_cast<const __m128i*>(r + 2)));
                std::memcpy(&h[k], r, 2);
            }
            _mm_stream_si128(reinterpret_cast<__m128i*>(d + b0 * 2), _mm_load_si128(reinterpret_cast<const __m128i*>(h)));
        }
        _mm_sfence();
    }
#endif
    repack_plain(raw, b0, b1, qs, d);
}

// ---------------------------------------------------------------------------
// The quantizers.  The plain loops say what they compute; where the CPU has AVX2 the same operations run eight at a time,
// with the same bits: no operation is fused or reordered except the maximum of absolute values, which does not depend on
// the order, and the conversions saturate as the plain ones do (below).  The plain loops do some 0.9 weights a nanosecond a
// core; with AVX2 they keep up with the memory they read.
// ---------------------------------------------------------------------------
static void q8_row(const float* src, int c0, int cols, float s, float amax, int mode, int8_t* dst) {
    if (mode == 0) {
        const float inv = 1.0f / s;
        for (int c = c0; c < cols; c++) {
            const float t = src[c] * inv;
            // Go's int(): truncate; NaN/overflow (only when 1/s overflowed) -> most negative
            const bool inRange = t > -9.2233720368547758e18f && t < 9.2233720368547758e18f;
            const long long v = inRange ? (long long)t : (-9223372036854775807LL - 1);
            dst[c] = (int8_t)std::min(127LL, std::max(-128LL, v));
        }
    } else {
        const float inv = 127.0f / amax;
        for (int c = c0; c < cols; c++) {
            float v = std::min(127.0f, std::max(-127.0f, src[c] * inv));
            dst[c] = (int8_t)(v + (v > 0 ? 0.5f : -0.5f));
        }
    }
}
static float q8_absmax(const float* src, int c0, int cols, float amax) {
    for (int c = c0; c < cols; c++) {
        float v = std::fabs(src[c]);
        if (v > amax) amax = v;
    }
    return amax;
}
static void q4_0_block(const float* x, uint8_t* y) {
    float amax = 0.0f, vmax = 0.0f;
    for (int j = 0; j < 32; j++) {
        if (std::fabs(x[j]) > amax) { amax = std::fabs(x[j]); vmax = x[j]; }
    }
    const float d = vmax / -8.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    const uint16_t hd = mg_f32_to_f16(d);
    std::memcpy(y, &hd, 2);
    for (int j = 0; j < 16; j++) {
        int lo = (int8_t)(x[j] * id + 8.5f);
        int hi = (int8_t)(x[j + 16] * id + 8.5f);
        y[2 + j] = (uint8_t)(std::min(lo, 15) | (std::min(hi, 15) << 4));
    }
}

#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
#define MG_AVX2 __attribute__((target("avx2")))
// max_ps takes its second operand when one is NaN: the running maximum, as `if (v > amax)` does
MG_AVX2 static inline float hmax8(__m256 m) {
    __m128 a = _mm_max_ps(_mm256_castps256_ps128(m), _mm256_extractf128_ps(m, 1));
    a = _mm_max_ps(a, _mm_movehl_ps(a, a));
    a = _mm_max_ss(a, _mm_shuffle_ps(a, a, 1));
    return _mm_cvtss_f32(a);
}
MG_AVX2 static float q8_absmax_avx2(const float* src, int cols) {
    const __m256 mask = _mm256_castsi256_ps(_mm256_set1_epi32(0x7fffffff));
    __m256 m0 = _mm256_setzero_ps(), m1 = m0, m2 = m0, m3 = m0;
    int c = 0;
    for (; c + 32 <= cols; c += 32) {
        m0 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(src + c), mask), m0);
        m1 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(src + c + 8), mask), m1);
        m2 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(src + c + 16), mask), m2);
        m3 = _mm256_max_ps(_mm256_and_ps(_mm256_loadu_ps(src + c + 24), mask), m3);
    }
    return q8_absmax(src, c, cols, hmax8(_mm256_max_ps(_mm256_max_ps(m0, m1), _mm256_max_ps(m2, m3))));
}
// 32 values -> 32 int8.  cvttps gives INT_MIN for NaN and what does not fit, the packs saturate: -128, as the plain loop's
// most negative value does.  (A finite value past 2^31 does not occur: |x * inv| is at most 127 but for rounding, or inv is
// infinite.)
MG_AVX2 static inline __m256i pack32(__m256i a, __m256i b, __m256i c, __m256i d) {
    const __m256i p = _mm256_packs_epi16(_mm256_packs_epi32(a, b), _mm256_packs_epi32(c, d));
    return _mm256_permutevar8x32_epi32(p, _mm256_setr_epi32(0, 4, 1, 5, 2, 6, 3, 7));
}
MG_AVX2 static void q8_row_avx2(const float* src, int cols, float s, float amax, int mode, int8_t* dst) {
    int c = 0;
    const __m256 inv = _mm256_set1_ps(mode == 0 ? 1.0f / s : 127.0f / amax);
    if (mode == 0) {
        for (; c + 32 <= cols; c += 32) {
            __m256i v[4];
            for (int k = 0; k < 4; k++) v[k] = _mm256_cvttps_epi32(_mm256_mul_ps(_mm256_loadu_ps(src + c + 8 * k), inv));
            _mm256_storeu_si256(reinterpret_cast<__m256i*>(dst + c), pack32(v[0], v[1], v[2], v[3]));
        }
    } else {
        const __m256 lo = _mm256_set1_ps(-127.0f), hi = _mm256_set1_ps(127.0f), up = _mm256_set1_ps(0.5f), dn = _mm256_set1_ps(-0.5f), z = _mm256_setzero_ps();
        for (; c + 32 <= cols; c += 32) {
            __m256i v[4];
            for (int k = 0; k < 4; k++) {
                const __m256 t = _mm256_min_ps(_mm256_max_ps(_mm256_mul_ps(_mm256_loadu_ps(src + c + 8 * k), inv), lo), hi);
                v[k] = _mm256_cvttps_epi32(_mm256_add_ps(t, _mm256_blendv_ps(dn, up, _mm256_cmp_ps(t, z, _CMP_GT_OQ))));
            }
            _mm256_storeu_si256(reinterpret_cast<__m256i*>(dst + c), pack32(v[0], v[1], v[2], v[3]));
        }
    }
    q8_row(src, c, cols, s, amax, mode, dst);
}
MG_AVX2 static void q4_0_block_avx2(const float* x, uint8_t* y) {
    const __m256 mask = _mm256_castsi256_ps(_mm256_set1_epi32(0x7fffffff));
    __m256 v[4], a[4], m = _mm256_setzero_ps();
    for (int k = 0; k < 4; k++) {
        v[k] = _mm256_loadu_ps(x + 8 * k);
        a[k] = _mm256_and_ps(v[k], mask);
        m = _mm256_max_ps(a[k], m);
    }
    const float amax = hmax8(m);
    const __m256 am = _mm256_set1_ps(amax);
    unsigned eq = 0;                               // the first value of that size gives the sign
    for (int k = 0; k < 4; k++) eq |= (unsigned)_mm256_movemask_ps(_mm256_cmp_ps(a[k], am, _CMP_EQ_OQ)) << (8 * k);
    const float vmax = amax > 0.0f ? x[__builtin_ctz(eq)] : 0.0f;
    const float d = vmax / -8.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    const uint16_t hd = mg_f32_to_f16(d);
    std::memcpy(y, &hd, 2);
    const __m256 idv = _mm256_set1_ps(id), off = _mm256_set1_ps(8.5f);
    const __m256i fifteen = _mm256_set1_epi32(15);
    __m256i n[4];
    for (int k = 0; k < 4; k++) {
        n[k] = _mm256_cvttps_epi32(_mm256_add_ps(_mm256_mul_ps(v[k], idv), off));
        n[k] = _mm256_min_epi32(_mm256_srai_epi32(_mm256_slli_epi32(n[k], 24), 24), fifteen);      // (int8_t), then at most 15
    }
    const __m256i b0 = _mm256_and_si256(_mm256_or_si256(n[0], _mm256_slli_epi32(n[2], 4)), _mm256_set1_epi32(255));
    const __m256i b1 = _mm256_and_si256(_mm256_or_si256(n[1], _mm256_slli_epi32(n[3], 4)), _mm256_set1_epi32(255));
    const __m256i p = _mm256_permute4x64_epi64(_mm256_packus_epi32(b0, b1), 0xd8);
    _mm_storeu_si128(reinterpret_cast<__m128i*>(y + 2), _mm_packus_epi16(_mm256_castsi256_si128(p), _mm256_extracti128_si256(p, 1)));
}
// The same with sixteen a time (saturating conversions as above; the scale of a block as the CPU rounds to fp16: to nearest
// even, as mg_f32_to_f16 does for everything but NaN, and a scale is none).
#define MG_AVX512 __attribute__((target("avx512f,avx512bw,avx512vl,avx2,f16c")))
MG_AVX512 static float q8_absmax_avx512(const float* src, int cols) {
    __m512 m0 = _mm512_setzero_ps(), m1 = m0, m2 = m0, m3 = m0;
    int c = 0;
    for (; c + 64 <= cols; c += 64) {
        m0 = _mm512_max_ps(_mm512_abs_ps(_mm512_loadu_ps(src + c)), m0);
        m1 = _mm512_max_ps(_mm512_abs_ps(_mm512_loadu_ps(src + c + 16)), m1);
        m2 = _mm512_max_ps(_mm512_abs_ps(_mm512_loadu_ps(src + c + 32)), m2);
        m3 = _mm512_max_ps(_mm512_abs_ps(_mm512_loadu_ps(src + c + 48)), m3);
    }
    return q8_absmax(src, c, cols, _mm512_reduce_max_ps(_mm512_max_ps(_mm512_max_ps(m0, m1), _mm512_max_ps(m2, m3))));
}
MG_AVX512 static void q8_row_avx512(const float* src, int cols, float s, float amax, int mode, int8_t* dst) {
    int c = 0;
    const __m512 inv = _mm512_set1_ps(mode == 0 ? 1.0f / s : 127.0f / amax);
    if (mode == 0) {
        for (; c + 16 <= cols; c += 16)
            _mm_storeu_si128(reinterpret_cast<__m128i*>(dst + c), _mm512_cvtsepi32_epi8(_mm512_cvttps_epi32(_mm512_mul_ps(_mm512_loadu_ps(src + c), inv))));
    } else {
        const __m512 lo = _mm512_set1_ps(-127.0f), hi = _mm512_set1_ps(127.0f), up = _mm512_set1_ps(0.5f), dn = _mm512_set1_ps(-0.5f);
        for (; c + 16 <= cols; c += 16) {
            const __m512 t = _mm512_min_ps(_mm512_max_ps(_mm512_mul_ps(_mm512_loadu_ps(src + c), inv), lo), hi);
            const __m512 r = _mm512_mask_blend_ps(_mm512_cmp_ps_mask(t, _mm512_setzero_ps(), _CMP_GT_OQ), dn, up);
            _mm_storeu_si128(reinterpret_cast<__m128i*>(dst + c), _mm512_cvtsepi32_epi8(_mm512_cvttps_epi32(_mm512_add_ps(t, r))));
        }
    }
    q8_row(src, c, cols, s, amax, mode, dst);
}
MG_AVX512 static void q4_0_blocks_avx512(const float* w, size_t b0, size_t b1, uint8_t* blocks) {
    const __m512 off = _mm512_set1_ps(8.5f);
    const __m512i fifteen = _mm512_set1_epi32(15);
    for (size_t b = b0; b < b1; b++) {
        const float* x = w + b * 32;
        uint8_t* y = blocks + b * 18;
        const __m512 v0 = _mm512_loadu_ps(x), v1 = _mm512_loadu_ps(x + 16), a0 = _mm512_abs_ps(v0), a1 = _mm512_abs_ps(v1);
        const float amax = _mm512_reduce_max_ps(_mm512_max_ps(a1, _mm512_max_ps(a0, _mm512_setzero_ps())));
        const __m512 am = _mm512_set1_ps(amax);
        const unsigned eq = (unsigned)_mm512_cmp_ps_mask(a0, am, _CMP_EQ_OQ) | ((unsigned)_mm512_cmp_ps_mask(a1, am, _CMP_EQ_OQ) << 16);
        const float vmax = amax > 0.0f ? x[__builtin_ctz(eq)] : 0.0f;      // the first value of that size gives the sign
        const float d = vmax / -8.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const uint16_t hd = (uint16_t)_mm_cvtsi128_si32(_mm_cvtps_ph(_mm_set_ss(d), _MM_FROUND_TO_NEAREST_INT));
        std::memcpy(y, &hd, 2);
        const __m512 idv = _mm512_set1_ps(id);
        __m512i n0 = _mm512_cvttps_epi32(_mm512_add_ps(_mm512_mul_ps(v0, idv), off)), n1 = _mm512_cvttps_epi32(_mm512_add_ps(_mm512_mul_ps(v1, idv), off));
        n0 = _mm512_min_epi32(_mm512_srai_epi32(_mm512_slli_epi32(n0, 24), 24), fifteen);
        n1 = _mm512_min_epi32(_mm512_srai_epi32(_mm512_slli_epi32(n1, 24), 24), fifteen);
        _mm_storeu_si128(reinterpret_cast<__m128i*>(y + 2), _mm512_cvtepi32_epi8(_mm512_or_si512(n0, _mm512_slli_epi32(n1, 4))));
    }
}
static bool have_avx2() { static const bool h = __builtin_cpu_supports("avx2"); return h; }
static bool have_avx512() {
    static const bool h = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") && __builtin_cpu_supports("avx512vl") && __builtin_cpu_supports("f16c");
    return h;
}
#else
static bool have_avx2() { return false; }
static bool have_avx512() { return false; }
static float q8_absmax_avx512(const float* src, int cols) { return q8_absmax(src, 0, cols, 0.f); }
static void q8_row_avx512(const float* src, int cols, float s, float amax, int mode, int8_t* dst) { q8_row(src, 0, cols, s, amax, mode, dst); }
static void q4_0_blocks_avx512(const float*, size_t, size_t, uint8_t*) {}
static float q8_absmax_avx2(const float* src, int cols) { return q8_absmax(src, 0, cols, 0.f); }
static void q8_row_avx2(const float* src, int cols, float s, float amax, int mode, int8_t* dst) { q8_row(src, 0, cols, s, amax, mode, dst); }
static void q4_0_block_avx2(const float* x, uint8_t* y) { q4_0_block(x, y); }
#endif

void quantize_q8_rows(const float* w, int cols, int mode, int8_t* q, float* scales, size_t r0, size_t r1) {
    const bool wide = have_avx2(), wider = have_avx512();
    for (size_t r = r0; r < r1; r++) {
        const float* src = w + r * (size_t)cols;
        int8_t* dst = q + r * (size_t)cols;
        const float amax = wider ? q8_absmax_avx512(src, cols) : wide ? q8_absmax_avx2(src, cols) : q8_absmax(src, 0, cols, 0.0f);
        const float s = amax / 127.0f;
        scales[r] = s;
        if (!(s > 0.0f)) { std::memset(dst, 0, (size_t)cols); continue; }
        if (wider) q8_row_avx512(src, cols, s, amax, mode, dst);
        else if (wide) q8_row_avx2(src, cols, s, amax, mode, dst);
        else q8_row(src, 0, cols, s, amax, mode, dst);
    }
}
void quantize_q4_0_blocks(const float* w, size_t b0, size_t b1, uint8_t* blocks) {
    if (have_avx512()) { q4_0_blocks_avx512(w, b0, b1, blocks); return; }
    const bool wide = have_avx2();
    for (size_t b = b0; b < b1; b++) {
        if (wide) q4_0_block_avx2(w + b * 32, blocks + b * 18);
        else q4_0_block(w + b * 32, blocks + b * 18);
    }
}

}  // namespace mg

extern "C" {

// IEEE binary16 <-> binary32, round to nearest even (what GGML's
// GGML_FP32_TO_FP16 does; not the truncating helper of conductor.go:27-35).
uint16_t mg_f32_to_f16(float f) {
    uint32_t x;
    std::memcpy(&x, &f, 4);
    const uint32_t sign = (x >> 16) & 0x8000u;
    x &= 0x7fffffffu;
    if (x > 0x7f800000u) return (uint16_t)(sign | 0x7e00u | ((x >> 13) & 0x1ffu));   // NaN, payload kept
    if (x >= 0x477ff000u) return (uint16_t)(sign | 0x7c00u);                          // overflow -> inf
    if (x < 0x33000001u) return (uint16_t)sign;                                       // <= 2^-25 -> 0 (tie to even)
    uint32_t mant, shift, expBits;
    if (x < 0x38800000u) {            // subnormal half
        mant = (x & 0x7fffffu) | 0x800000u;
        shift = 126u - (x >> 23);
        expBits = 0;
    } else {
        mant = x & 0x7fffffu;
        shift = 13;
        expBits = ((x >> 23) - 112u) << 10;
    }
    uint32_t keep = mant >> shift;
    uint32_t dropped = mant & ((1u << shift) - 1u);
    uint32_t halfway = 1u << (shift - 1);
    uint32_t r = expBits + keep;                     // '+' so a mantissa carry bumps the exponent
    if (dropped > halfway || (dropped == halfway && (keep & 1u))) r++;
    return (uint16_t)(sign | r);
}

float mg_f16_to_f32(uint16_t h) {
    const uint32_t sign = ((uint32_t)h & 0x8000u) << 16;
    uint32_t e = (h >> 10) & 0x1fu, m = h & 0x3ffu, x;
    if (e == 31) x = sign | 0x7f800000u | (m << 13);
    else if (e != 0) x = sign | ((e + 112u) << 23) | (m << 13);
    else if (m == 0) x = sign;
    else {
        // value = m * 2^-24; normalise
        int lz = __builtin_clz(m) - 21;              // shifts needed to bring bit 10 up
        m = (m << lz) & 0x3ffu;
        x = sign | ((uint32_t)(113 - lz) << 23) | (m << 13);
    }
    float f;
    std::memcpy(&f, &x, 4);
    return f;
}

// quantizeQ8, cuda_fused_infer.go:363-390 (mode 0), or the Metal loader's
// rounding, metal_impl_darwin.m:5765-5780 (mode 1).  scale = absmax/127.
void mg_quantize_q8(const float* w, int rows, int cols, int mode, int8_t* q, float* scales) {
    mg::parallel_for((size_t)rows, std::max(1, 16384 / std::max(cols, 1)), [&](size_t r0, size_t r1) { mg::quantize_q8_rows(w, cols, mode, q, scales, r0, r1); });
}

// GGML quantize_row_q4_0 (the block format cuda_q4_0.go:13-17 uploads).
void mg_quantize_q4_0(const float* w, int rows, int cols, uint8_t* blocks) {
    const size_t nb = (size_t)rows * (cols / 32);
    mg::parallel_for(nb, 1 << 9, [&](size_t b0, size_t b1) { mg::quantize_q4_0_blocks(w, b0, b1, blocks); });
}

// ---------------------------------------------------------------------------
// Synthetic inputs.  Identical on every machine: integer generator
// (splitmix64 -> xoshiro256**), Marsaglia's polar method, and a logarithm
// written out in plain IEEE double operations (no libm call whose last bit
// could depend on the host CPU).
// ---------------------------------------------------------------------------
namespace {
inline uint64_t splitmix64(uint64_t& s) {
    uint64_t z = (s += 0x9e3779b97f4a7c15ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
struct Xoshiro {
    uint64_t s[4];
    Xoshiro(uint64_t seed, uint64_t idx, uint64_t blk) {
        uint64_t k = seed * 0x9e3779b97f4a7c15ull ^ (idx + 0x632be59bd9b4e019ull) * 0xd1342543de82ef95ull ^ (blk << 1 | 1) * 0xa0761d6478bd642full;
        for (int i = 0; i < 4; i++) s[i] = splitmix64(k);
    }
    static inline uint64_t rotl(uint64_t x, int k) { return (x << k) | (x >> (64 - k)); }
    inline uint64_t next() {
        const uint64_t r = rotl(s[1] * 5, 7) * 9, t = s[1] << 17;
        s[2] ^= s[0]; s[3] ^= s[1]; s[1] ^= s[2]; s[0] ^= s[3]; s[2] ^= t; s[3] = rotl(s[3], 45);
        return r;
    }
    inline double unit() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); }   // [0,1)
};
// ln(x) for x in (0, 1]: x = m*2^e, m in [sqrt(.5), sqrt(2)); ln m = 2*atanh((m-1)/(m+1))
inline double det_log(double x) {
    int e;
    double m = std::frexp(x, &e);               // exact
    if (m < 0.70710678118654752440) { m *= 2.0; e -= 1; }
    const double s = (m - 1.0) / (m + 1.0);
    const double z = s * s;
    double p = 1.0 / 23.0;
    p = p * z + 1.0 / 21.0; p = p * z + 1.0 / 19.0; p = p * z + 1.0 / 17.0; p = p * z + 1.0 / 15.0;
    p = p * z + 1.0 / 13.0; p = p * z + 1.0 / 11.0; p = p * z + 1.0 / 9.0;  p = p * z + 1.0 / 7.0;
    p = p * z + 1.0 / 5.0;  p = p * z + 1.0 / 3.0;  p = p * z + 1.0;
    return (double)e * 0.69314718055994530942 + 2.0 * s * p;
}
constexpr size_t kSynthBlock = 4096;
}  // namespace

void mg_synth_normal(uint64_t seed, uint64_t idx, float stdv, float* out, size_t n) {
    const size_t nblk = (n + kSynthBlock - 1) / kSynthBlock;
    mg::parallel_for(nblk, 8, [&](size_t b0, size_t b1) {
        for (size_t b = b0; b < b1; b++) {
            Xoshiro g(seed, idx, b);
            size_t a = b * kSynthBlock, e = std::min(n, a + kSynthBlock);
            size_t i = a;
            while (i < e) {
                double u = 2.0 * g.unit() - 1.0, v = 2.0 * g.unit() - 1.0;
                double s = u * u + v * v;
                if (s >= 1.0 || s == 0.0) continue;
                double f = std::sqrt(-2.0 * det_log(s) / s);
                out[i++] = (float)(u * f * (double)stdv);
                if (i < e) out[i++] = (float)(v * f * (double)stdv);
            }
        }
    });
}

void mg_synth_tokens(uint64_t seed, uint64_t idx, int bound, int* out, size_t n) {
    Xoshiro g(seed, idx, 0x7fffffffull);
    for (size_t i = 0; i < n; i++) out[i] = (int)((g.next() >> 11) % (uint64_t)bound);
}

}  // extern "C"
