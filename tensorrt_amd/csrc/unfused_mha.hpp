// What unfused_mha.hip asks of the other kernels of the unfused attention path (inside the library only).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace trtamd
{

// Binary32 attention with the keys split between wavefronts: the tiles of 16 rows need S >= 16 and a head size that is a
// multiple of 16 (of 16-byte aligned rows), the scores of a wavefront's keys fit in registers up to S = 1024, and offsets
// into Q, K and V are 32 bits.
bool attention_split_keys_takes(int32_t S, int32_t B, int32_t N, int32_t d, float const* qkv, float const* output);
int attention_split_keys(hipStream_t stream, int32_t S, int32_t B, int32_t N, int32_t d, float const* qkv,
    int32_t const* maskIdx, float* output);

} // namespace trtamd
