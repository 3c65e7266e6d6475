// What the native encoder passes ask of the kernels beyond the public entry points (inside the library only): what only a
// caller that knows the next launch can say, or can leave to it.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "trtamd_encoder_ops.h"

namespace trtamd
{

// Weights that an INT8 linear launch should bring into the caches beside its own work, for a later launch that is bound by the
// latency of its weights: few tokens, or long rows.  The CUs that the launches before it leave idle can fetch them.
// `units` KB of a 32-interleaved matrix, each 32 output channels of one k-slab; the 32-channel block with number c is read
// on XCD c % 8 and fetched there.  data == nullptr: nothing.
struct WeightPrefetch
{
    void const* data;
    uint32_t units;
};
WeightPrefetch prefetch_of(trtamd_int8_linear_params const& next);

// trtamd_int8_linear with a prefetch beside it.
int int8_linear(trtamd_stream_t stream, trtamd_int8_linear_params const& p, WeightPrefetch const& prefetch);

// A linear layer of few tokens and long rows whose k range is shared by `parts` workgroups each: instead of its output it
// leaves `parts` sums of accumulators [parts][T][N] (INT32 / binary32), which the SkipLayerNorm behind it adds up.
// 1: not worth it (the layer has enough workgroups, or a short k loop); at most kMaxLinearParts.
constexpr int kMaxLinearParts = 4;
int linear_parts(trtamd_int8_linear_params const& p);
int linear_parts(trtamd_fp16_linear_params const& p);
// Bytes that the partial sums of any such layer fit in: they come from one workgroup per CU at most, 32 x 32 of them each.
size_t linear_partial_bytes();
// linear_parts is 1 for more tokens than these and for layers of fewer bytes of k.
constexpr int kLinearPartialTokens = 255, kLinearPartialK = 2048;
// `parts`: what linear_parts said.  The parameters are checked as the public calls check theirs.
int int8_linear_partial(trtamd_stream_t stream, trtamd_int8_linear_params const& p, int parts, int32_t* partial,
    WeightPrefetch const& prefetch);
int fp16_linear_partial(trtamd_stream_t stream, trtamd_fp16_linear_params const& p, int parts, float* partial);
// The checks of trtamd_fp16_linear without its launch, for a pass that is refused before its first launch.
int fp16_linear_check(trtamd_fp16_linear_params const& p);

// trtamd_skipln_interleaved_{small,large}_hface with the input given as the partial sums of an affine INT8 layer (alpha,
// beta as in trtamd_int8_linear_params): the same bytes as the layer's output through memory would give.
int skipln_interleaved_from_partial(trtamd_stream_t stream, bool large, int32_t ld, int32_t total, int32_t const* partial,
    int parts, float const* alpha, float const* beta, int8_t const* skip, trtamd_half_t const* lnBeta,
    trtamd_half_t const* lnGamma, int8_t* output, float dqScaleIn, float dqScaleSkip, float qScale);

// trtamd_skip_layer_norm_fp16 likewise, behind an affine FP16 layer.
int skip_layer_norm_fp16_from_partial(trtamd_stream_t stream, int32_t ld, int32_t rows, float const* partial, int parts,
    float const* alpha, float const* beta, trtamd_half_t const* skip, trtamd_half_t const* lnBeta,
    trtamd_half_t const* lnGamma, trtamd_half_t* output, trtamd_half_t const* bias);

} // namespace trtamd
