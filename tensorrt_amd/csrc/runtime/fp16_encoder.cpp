// One pass of the FP16 encoder of include/trtamd_encoder_runtime.h: the launches that tensorrt_amd/encoder_fp16.py used to
// make one by one from Python, 10 to 12 us of host time each where the kernels of a short request take 4 to 8.  The plugin
// objects, weights and buffers are the caller's; nothing is allocated or synchronised.
#include "plugin_common.h"
#include "trtamd_encoder_runtime.h"

#include "../host_utils.hpp"
#include "../network_ops.hpp"

#include <string>

namespace trtamd
{
namespace runtime
{
namespace
{

using namespace trtamd::plugin;

PluginTensorDesc half(std::initializer_list<int64_t> dims)
{
    PluginTensorDesc d{};
    for (int64_t v : dims)
    {
        d.dims.d[d.dims.nbDims++] = v;
    }
    d.type = DataType::kHALF;
    d.format = TensorFormat::kLINEAR;
    d.scale = 1.f;
    return d;
}

PluginTensorDesc int32(std::initializer_list<int64_t> dims)
{
    PluginTensorDesc d = half(dims);
    d.type = DataType::kINT32;
    return d;
}

IPluginV3OneRuntime* runtimeOf(void* plugin, char const* what)
{
    TRTAMD_VALIDATE_MSG(plugin != nullptr, std::string(what) + ": no plugin object");
    auto* rt = static_cast<IPluginV3OneRuntime*>(
        static_cast<IPluginV3*>(plugin)->getCapabilityInterface(PluginCapabilityType::kRUNTIME));
    TRTAMD_VALIDATE_MSG(rt != nullptr, std::string(what) + ": no runtime capability");
    return rt;
}

void run(void* plugin, char const* what, PluginTensorDesc const* in, int32_t nbIn, PluginTensorDesc const* out, int32_t nbOut,
    void const* const* inputs, void* const* outputs, hipStream_t stream)
{
    IPluginV3OneRuntime* rt = runtimeOf(plugin, what);
    int32_t st = rt->onShapeChange(in, nbIn, out, nbOut);
    if (st == 0)
    {
        st = rt->enqueue(in, out, inputs, outputs, nullptr, stream);
    }
    TRTAMD_VALIDATE_MSG(st == 0, std::string(what) + " failed with status " + std::to_string(st));
}

int enqueue(trtamd_fp16_encoder_config const& c, trtamd_fp16_encoder_layer const* layers, trtamd_fp16_encoder_batch const& b,
    hipStream_t stream)
{
    TRTAMD_VALIDATE(c.hidden > 0 && c.ffn > 0 && c.layers >= 0 && c.max_seqlen > 0 && (layers != nullptr || c.layers == 0));
    TRTAMD_VALIDATE(b.batch > 0 && b.tokens > 0 && b.ids && b.segment_ids && b.cu_seqlens && b.x && b.qkv && b.ctx && b.ao
        && b.h && b.m && b.f && b.mask && b.longest && b.emb2);
    int64_t const T = b.tokens, B = b.batch, E = c.hidden;
    int32_t const tokens = b.tokens;
    PluginTensorDesc const tIds = int32({T}), tCu = int32({B + 1}), tLongest = int32({c.max_seqlen}), tOne = int32({1});
    PluginTensorDesc const act = half({T, E, 1, 1}), qkvAct = half({T, 3 * E, 1, 1}), row = half({T, 1, E, 1, 1});

    auto params = [&](trtamd_fp16_encoder_linear const& l, void const* a, void* out, int32_t K, int32_t N, int32_t epilogue) {
        trtamd_fp16_linear_params p{};
        p.a = static_cast<trtamd_half_t const*>(a);
        p.w = l.w;
        p.alpha = l.alpha;
        p.beta = l.beta;
        p.out = static_cast<trtamd_half_t*>(out);
        p.T = tokens;
        p.K = K;
        p.N = N;
        p.epilogue = epilogue;
        return p;
    };
    // Few tokens: the second feed-forward layer, whose k loop is the longest, shares it between workgroups, and the
    // normalisation behind it adds up the sums, if what that takes beside the plugins is there.
    int parts = 1;
    if (c.layers > 0 && c.hidden % 8 == 0 && c.hidden > 32 && c.hidden <= 1024 && b.partial && aligned16(b.partial)
        && b.partial_bytes >= linear_partial_bytes())
    {
        parts = linear_parts(params(layers[0].ffn2, b.m, b.f, c.ffn, c.hidden, TRTAMD_LINEAR_AFFINE));
    }
    // everything that can be refused is refused before the first launch
    auto check = [&](trtamd_fp16_linear_params const& p) { checkKernelStatus(fp16_linear_check(p), "linear layer"); };
    for (int32_t i = 0; i < c.layers; ++i)
    {
        trtamd_fp16_encoder_layer const& L = layers[i];
        check(params(L.qkv, b.x, b.qkv, c.hidden, 3 * c.hidden, TRTAMD_LINEAR_AFFINE));
        check(params(L.proj, b.ctx, b.ao, c.hidden, c.hidden, TRTAMD_LINEAR_AFFINE));
        check(params(L.ffn1, b.h, b.m, c.hidden, c.ffn, TRTAMD_LINEAR_GELU));
        check(params(L.ffn2, b.m, b.f, c.ffn, c.hidden, TRTAMD_LINEAR_AFFINE));
        for (trtamd_half_t const* v : {L.ln2_gamma, L.ln2_beta, L.ln2_bias})
        {
            parts = v && aligned16(v) ? parts : 1;
        }
    }
    auto linear = [&](trtamd_fp16_linear_params const& p) {
        checkKernelStatus(trtamd_fp16_linear(stream, &p), "linear layer");
    };
    auto skipln = [&](void* plugin, void const* x, void const* skip, void* out) {
        PluginTensorDesc const in[2] = {row, row};
        void const* inputs[2] = {x, skip};
        run(plugin, "skipLayerNorm", in, 2, &row, 1, inputs, &out, stream);
    };
    {
        PluginTensorDesc const in[4] = {tIds, tIds, tCu, tLongest}, out[2] = {act, int32({})};
        void const* inputs[4] = {b.ids, b.segment_ids, b.cu_seqlens, b.longest};
        void* outputs[2] = {b.x, b.emb2};
        run(c.embedding, "embeddings", in, 4, out, 2, inputs, outputs, stream);
    }
    for (int32_t i = 0; i < c.layers; ++i)
    {
        trtamd_fp16_encoder_layer const& L = layers[i];
        linear(params(L.qkv, b.x, b.qkv, c.hidden, 3 * c.hidden, TRTAMD_LINEAR_AFFINE));
        {
            PluginTensorDesc const in[4] = {qkvAct, tOne, tCu, tLongest};
            void const* inputs[4] = {b.qkv, b.mask, b.cu_seqlens, b.longest};
            void* outputs[1] = {b.ctx};
            run(L.attention, "attention", in, 4, &act, 1, inputs, outputs, stream);
        }
        linear(params(L.proj, b.ctx, b.ao, c.hidden, c.hidden, TRTAMD_LINEAR_AFFINE));
        skipln(L.ln1, b.ao, b.x, b.h);
        linear(params(L.ffn1, b.h, b.m, c.hidden, c.ffn, TRTAMD_LINEAR_GELU));
        auto const f2 = params(L.ffn2, b.m, b.f, c.ffn, c.hidden, TRTAMD_LINEAR_AFFINE);
        if (parts > 1)
        {
            checkKernelStatus(fp16_linear_partial(stream, f2, parts, b.partial), "linear layer");
            checkKernelStatus(skip_layer_norm_fp16_from_partial(stream, c.hidden, tokens, b.partial, parts, f2.alpha, f2.beta, b.h,
                                  L.ln2_beta, L.ln2_gamma, b.x, L.ln2_bias),
                "skipLayerNorm");
        }
        else
        {
            linear(f2);
            skipln(L.ln2, b.f, b.h, b.x);
        }
    }
    return TRTAMD_STATUS_SUCCESS;
}

} // namespace
} // namespace runtime
} // namespace trtamd

extern "C" int trtamd_fp16_encoder_enqueue(trtamd_fp16_encoder_config const* config, trtamd_fp16_encoder_layer const* layers,
    trtamd_fp16_encoder_batch const* batch, trtamd_stream_t stream)
{
    try
    {
        TRTAMD_VALIDATE(config != nullptr && batch != nullptr);
        return trtamd::runtime::enqueue(*config, layers, *batch, trtamd::as_stream(stream));
    }
    catch (std::exception const& e)
    {
        return trtamd::set_error(TRTAMD_STATUS_FAILURE, "fp16_encoder_enqueue: %s", e.what());
    }
}
