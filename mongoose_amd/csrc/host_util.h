// host_util.h -- host helpers shared inside libmongoose_hip.so.
#pragma once
#include <cstddef>
#include <cstdint>
#include <functional>

namespace mg {

// fn(job) for job in [0, njobs) on the library's worker threads (up to 16 with the caller); returns when
// all are done.  One region at a time; fn must not start another.  meanwhile: what the caller does once the workers have
// been set going, before it takes jobs itself.
void parallel_jobs(size_t njobs, const std::function<void(size_t)>& fn, const std::function<void()>& meanwhile = nullptr);
// fn(begin, end) over [0, n) in pieces of `grain`, through parallel_jobs.
void parallel_for(size_t n, size_t grain, const std::function<void(size_t, size_t)>& fn);

// mg_quantize_q8's rows [r0, r1) and mg_quantize_q4_0's blocks [b0, b1), on the calling thread
void quantize_q8_rows(const float* w, int cols, int mode, int8_t* q, float* scales, size_t r0, size_t r1);
void quantize_q4_0_blocks(const float* w, size_t b0, size_t b1, uint8_t* blocks);
// GGUF block_q4_0 -> nibble plane + fp16 scale plane (16 and 2 bytes a block): blocks [b0, b1) of a matrix of nb blocks,
// on the calling thread
void repack_q4_0_blocks(const uint8_t* raw, size_t nb, size_t b0, size_t b1, uint8_t* planar);

}  // namespace mg
