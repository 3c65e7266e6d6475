// The fixed-length EmbLayerNorm with the mask output of the plugin in the same launch (inside the library only).
#pragma once

#include <stdint.h>

#include "trtamd_bert_kernels.h"

namespace trtamd
{

// What the extra workgroups of the embedding launch write.  warpsM == 0: maskIdx[b], as trtamd_compute_mask_idx;
// otherwise the packed mask of that geometry, as trtamd_convert_mask with warps_k = 1.
struct EmbMask
{
    int32_t const* mask; // [S, B]
    void* out;
    uint32_t warpsM, warpsN;
};

// trtamd_emb_layer_norm_fp32 / _fp16 (type 0 / 1) followed by the mask call, as one launch.
int emb_layer_norm_with_mask(trtamd_stream_t stream, int32_t type, int32_t ld, int32_t B, int32_t S,
    int32_t const* inputIds, int32_t const* tokenIds, float const* beta, float const* gamma, void const* wordEmb,
    void const* posEmb, void const* tokEmb, int32_t wordSize, int32_t tokSize, void* output, EmbMask const& mask);

} // namespace trtamd
