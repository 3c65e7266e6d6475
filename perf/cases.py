"""What a program that uses this library asks of it, as measurable cases.

    int8_encoder       the INT8 encoder through the native runner (trtamd_encoder_enqueue / _enqueue_concurrent)
    fp16_encoder       the FP16 encoder (tensorrt_amd.encoder_fp16), called with the host arrays of a new batch
    attention_var      QKV-to-context on packed sequences: v5 in FP16, v6 (32-interleaved) in INT8
    attention_fixed    QKV-to-context v4 on padded sequences with a packed mask, FP16 and INT8
    attention_unfused  QKV-to-context v4 where no fused kernel exists: FP32, or FP16 at lengths of its own
    skipln             SkipLayerNorm v6 with bias, FP32 and FP16
    embln              EmbLayerNorm v6 with mask, FP32 and FP16

Models, plugin objects and workspaces are kept from call to call, as a serving program keeps them; what is new for
every seed are the contents of the sequences and the order in which their lengths come.  The models are the two of the benchmark configurations: 24 layers
of 1024 channels in INT8 and 12 layers of 768 channels in FP16, random-initialised.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from tensorrt_amd import capi
from tensorrt_amd.encoder import EMBLN, QKV, SKIPLN, EncoderConfig, Int8BertEncoder
from tensorrt_amd.encoder_fp16 import Fp16BertEncoder
from tensorrt_amd.plugin import (DataType, PluginField, PluginFieldType, TensorDesc, TensorFormat, TensorRTPhase,
                                 get_plugin_registry)

VOCAB = 30522
HEAD = 64
FUSED_LENGTHS = (64, 96, 128, 384)  # padded lengths that have a packed mask
TORCH = {"fp32": torch.float32, "fp16": torch.float16, "int8": torch.int8}
TRT = {"fp32": DataType.FLOAT, "fp16": DataType.HALF, "int8": DataType.INT8}
SIZE = {"fp32": 4, "fp16": 2, "int8": 1}


def listed():
    return [
        # one short question to a loaded model: nothing but latency, weights and launches
        dict(name="int8 encoder, one request", kind="int8_encoder", batch=1, max_len=48, parts=1),
        # a few queued requests of sentence length
        dict(name="int8 encoder, small batch", kind="int8_encoder", batch=7, max_len=128, parts=1),
        # a server's ordinary dynamic batch
        dict(name="int8 encoder, batch of 32", kind="int8_encoder", batch=32, max_len=256, parts=1),
        # throughput: the benchmark batch as two concurrent halves
        dict(name="int8 encoder, batch of 128", kind="int8_encoder", batch=128, max_len=384, parts=2),
        # one request to the FP16 model
        dict(name="fp16 encoder, one request", kind="fp16_encoder", batch=1, max_len=128),
        # the FP16 model on long sequences
        dict(name="fp16 encoder, batch of 32", kind="fp16_encoder", batch=32, max_len=384),
        # an engine's attention layer on packed sequences
        dict(name="attention fp16, packed", kind="attention_var", dtype="fp16", batch=32, heads=12, max_len=384),
        # the padded layout with the mask that the embedding layer packs
        dict(name="attention fp16, padded", kind="attention_fixed", dtype="fp16", batch=16, heads=12, seq=128),
        # full precision at a length that is a multiple of nothing
        dict(name="attention fp32, odd length", kind="attention_unfused", dtype="fp32", batch=8, heads=12, seq=197, head=64),
        # residual + LayerNorm of a small FP32 engine
        dict(name="skipln fp32, small", kind="skipln", dtype="fp32", seq=128, batch=8, hidden=768),
        # the same in FP16 on a batch that no cache holds
        dict(name="skipln fp16, large", kind="skipln", dtype="fp16", seq=384, batch=171, hidden=768),
        # the first layer of a padded FP16 engine
        dict(name="embln fp16", kind="embln", dtype="fp16", seq=128, batch=32, hidden=768),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("int8_encoder", "int8_encoder", "fp16_encoder", "fp16_encoder", "attention_var",
                       "attention_fixed", "attention_unfused", "skipln", "embln"))
    if kind == "int8_encoder":
        batch = _log(rng, 1, 128)
        # a server splits a batch in two only where both halves are worth a launch sequence of their own
        return dict(kind=kind, batch=batch, max_len=_log(rng, 16, 384), parts=2 if batch >= 64 else 1)
    if kind == "fp16_encoder":
        return dict(kind=kind, batch=_log(rng, 1, 64), max_len=_log(rng, 16, 384))
    if kind == "attention_var":
        return dict(kind=kind, dtype=rng.choice(("fp16", "int8")), batch=_log(rng, 1, 128), heads=rng.choice((12, 16)),
                    max_len=_log(rng, 16, 512))
    if kind == "attention_fixed":
        return dict(kind=kind, dtype=rng.choice(("fp16", "int8")), batch=_log(rng, 1, 64), heads=rng.choice((12, 16)),
                    seq=rng.choice(FUSED_LENGTHS))
    if kind == "attention_unfused":
        seq = _log(rng, 16, 1024)
        while seq in FUSED_LENGTHS:
            seq += 1
        return dict(kind=kind, dtype=rng.choice(("fp32", "fp32", "fp16")), batch=_log(rng, 1, max(1, 8192 // seq)),
                    heads=rng.choice((4, 12, 16)), seq=seq, head=rng.choice((32, 64, 80)))
    if kind == "skipln":
        return dict(kind=kind, dtype=rng.choice(("fp32", "fp16")), seq=_log(rng, 16, 512), batch=_log(rng, 1, 192),
                    hidden=rng.choice((384, 512, 768, 1024)))
    return dict(kind=kind, dtype=rng.choice(("fp32", "fp16")), seq=_log(rng, 16, 512), batch=_log(rng, 1, 128),
                hidden=rng.choice((768, 1024)))


# ---- models and plugin objects, kept as a serving program keeps them ---------------------------------------------

@functools.lru_cache(maxsize=None)
def _int8_model():
    """The INT8 model, calibrated, with two execution contexts."""
    enc = Int8BertEncoder(EncoderConfig(hidden=1024, heads=16, ffn=4096, layers=24))
    r = np.random.default_rng(1)
    cu = _prefix_sums(r.integers(64, 257, 8))
    enc.calibrate(r.integers(0, VOCAB, cu[-1]).astype(np.int32), r.integers(0, 2, cu[-1]).astype(np.int32), cu)
    handle = enc.build_native()
    enc.api.check(enc.api.encoder_reserve_contexts(handle, 2))
    return enc, handle


@functools.lru_cache(maxsize=None)
def _fp16_model():
    return Fp16BertEncoder(EncoderConfig(hidden=768, heads=12, ffn=3072, layers=12))


def _i32(name, v):
    return PluginField(name, np.array([v], np.int32), PluginFieldType.INT32)


def _f32(name, v):
    return PluginField(name, np.asarray(v, np.float32), PluginFieldType.FLOAT32)


def _plugin(name, version, fields, ins=None, outs=None):
    """Build phase, configuration and the runtime-phase object, as an engine file gives them."""
    creator = get_plugin_registry().get_creator(name, version)
    built = creator.create_plugin("layer", fields)
    if ins is not None and built.configure_plugin(ins, outs) != 0:
        raise RuntimeError(f"{name} {version}: configurePlugin failed")
    workspace = built.get_workspace_size(ins, outs) if ins is not None else 0
    plugin = creator.create_plugin("layer", built.get_fields_to_serialize(), TensorRTPhase.RUNTIME)
    return plugin, workspace


def _attention_fields(dtype, heads, head, extra=()):
    return [_i32("type_id", int(TRT[dtype])), _i32("hidden_size", heads * head), _i32("num_heads", heads),
            _i32("has_mask", 1), *extra]


@functools.lru_cache(maxsize=None)
def _skipln_plugin(dtype, hidden):
    r = np.random.default_rng(2)
    return _plugin(SKIPLN, "6", [_i32("type_id", int(TRT[dtype])), _f32("beta", 0.1 * r.standard_normal(hidden)),
                                 _f32("gamma", r.uniform(0.5, 1.5, hidden)),
                                 _f32("bias", 0.02 * r.standard_normal(hidden))])[0]


@functools.lru_cache(maxsize=None)
def _embln_plugin(dtype, hidden):
    r = np.random.default_rng(3)
    table = lambda n: 0.02 * r.standard_normal((n, hidden), np.float32)
    return _plugin(EMBLN, "6", [
        _f32("bert_embeddings_layernorm_beta", 0.1 * r.standard_normal(hidden)),
        _f32("bert_embeddings_layernorm_gamma", r.uniform(0.5, 1.5, hidden)),
        _f32("bert_embeddings_word_embeddings", table(VOCAB)),
        _f32("bert_embeddings_token_type_embeddings", table(2)),
        _f32("bert_embeddings_position_embeddings", table(512)),
        _i32("output_fp16", 1 if dtype == "fp16" else 0), _i32("mha_type_id", int(TRT[dtype]))])[0]


# ---- inputs ------------------------------------------------------------------------------------------------------

def _prefix_sums(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _lengths_of(case):
    n = case.get("max_len") or case["seq"]
    lo = -(-n // 3)  # lengths spread over a factor of three, as in the encoder benchmark
    return np.random.default_rng([case["batch"], n]).integers(lo, n + 1, case["batch"])


def _lengths(case, seed):
    """The case's lengths in the order in which this seed's requests came."""
    return np.random.default_rng(seed).permutation(_lengths_of(case))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _tokens(g, shape):
    ids = torch.randint(0, VOCAB, shape, generator=g, device="cuda", dtype=torch.int32)
    segs = torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.int32)
    return ids, segs


def _activations(g, shape, dtype):
    """Normal activations; INT8 with the scale amax / 127 that a calibrator finds.  Returns (tensor, scale)."""
    x = torch.randn(shape, generator=g, device="cuda")
    if dtype != "int8":
        return x.to(TORCH[dtype]), 1.0
    scale = float(x.abs().max()) / 127
    return (x / scale).round_().clamp_(-127, 127).to(torch.int8), scale


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _plugin_call(plugin, ins, outs, inputs, outputs, workspace=0):
    """A plugin layer ready to be enqueued: descriptors and addresses stay from pass to pass."""
    if plugin.on_shape_change(ins, outs) != 0:
        raise RuntimeError("onShapeChange failed")
    ws = torch.empty((max(workspace, 1),), dtype=torch.uint8, device="cuda")
    return dict(plugin=plugin, ins=ins, outs=outs, inputs=[t.data_ptr() for t in inputs],
                outputs=[t.data_ptr() for t in outputs], workspace=ws.data_ptr(), stream=_stream(),
                result=list(outputs), keep=(inputs, ws))


def _prepare_int8_encoder(case, seed):
    enc, handle = _int8_model()
    api, hidden = enc.api, enc.cfg.hidden
    lens = _lengths(case, seed)
    cu = _prefix_sums(lens)
    total = int(cu[-1])
    ids, segs = _tokens(_generator(seed), (total,))
    out = torch.empty((total, hidden), dtype=torch.float16, device="cuda")
    cut = int(np.argmin(np.abs(cu - total / 2))) if case["parts"] == 2 else 0
    runs = [(0, cut), (cut, len(lens))] if 0 < cut < len(lens) else [(0, len(lens))]
    batches = (capi.EncoderBatch * len(runs))()
    keep = []
    for q, (lo, hi) in zip(batches, runs):
        t0, n = int(cu[lo]), int(cu[hi] - cu[lo])
        sub = torch.from_numpy(cu[lo:hi + 1] - cu[lo]).cuda()
        ws = torch.empty((api.encoder_workspace_size(handle, n),), dtype=torch.uint8, device="cuda")
        keep += [sub, ws]
        q.ids, q.segment_ids, q.cu_seqlens = ids.data_ptr() + 4 * t0, segs.data_ptr() + 4 * t0, sub.data_ptr()
        q.batch, q.tokens, q.workspace, q.out = hi - lo, n, ws.data_ptr(), out.data_ptr() + 2 * hidden * t0
    return dict(api=api, handle=handle, batches=batches, stream=_stream(), result=out, keep=(ids, segs, keep))


def _prepare_fp16_encoder(case, seed):
    r = np.random.default_rng(seed)
    cu = _prefix_sums(_lengths(case, seed))
    # a request arrives as host arrays
    return dict(model=_fp16_model(), ids=r.integers(0, VOCAB, cu[-1]).astype(np.int32),
                segs=r.integers(0, 2, cu[-1]).astype(np.int32), cu=cu)


def _prepare_attention_var(case, seed):
    dtype, heads, hidden = case["dtype"], case["heads"], case["heads"] * HEAD
    cu = _prefix_sums(_lengths(case, seed))
    total, batch = int(cu[-1]), case["batch"]
    qkv, scale = _activations(_generator(seed), (total, 3 * hidden), dtype)
    cu_dev = torch.from_numpy(cu).cuda()
    longest = torch.zeros((case["max_len"],), dtype=torch.int32, device="cuda")
    tail = [TensorDesc([batch + 1], DataType.INT32), TensorDesc([case["max_len"]], DataType.INT32)]
    if dtype == "int8":
        qkv = qkv.view(total, 3 * hidden // 32, 32).transpose(0, 1).contiguous()
        ins = [TensorDesc([1, 3 * hidden, total, 1], DataType.INT8, TensorFormat.CHW32, scale), *tail]
        outs = [TensorDesc([1, hidden, total, 1], DataType.INT8, TensorFormat.CHW32, scale)]
        out = torch.empty((hidden // 32, total, 32), dtype=torch.int8, device="cuda")
        plugin, ws = _plugin(QKV, "6", [_i32("hidden_size", hidden), _i32("num_heads", heads),
                                        _f32("dq_probs", [1 / 127])], ins, outs)
        return _plugin_call(plugin, ins, outs, [qkv, cu_dev, longest], [out], ws)
    mask = torch.zeros((1,), dtype=torch.int32, device="cuda")
    ins = [TensorDesc([total, 3 * hidden, 1, 1], DataType.HALF), TensorDesc([1], DataType.INT32), *tail]
    outs = [TensorDesc([total, hidden, 1, 1], DataType.HALF)]
    out = torch.empty((total, hidden), dtype=torch.float16, device="cuda")
    plugin, ws = _plugin(QKV, "5", _attention_fields(dtype, heads, HEAD, [_i32("var_seqlen", 1)]), ins, outs)
    return _plugin_call(plugin, ins, outs, [qkv, mask, cu_dev, longest], [out], ws)


def _prepare_attention_fixed(case, seed):
    dtype, seq, batch, hidden = case["dtype"], case["seq"], case["batch"], case["heads"] * HEAD
    lens = torch.from_numpy(_lengths(case, seed)).cuda()
    mask = (torch.arange(seq, device="cuda")[:, None] < lens[None, :]).to(torch.int32)
    packed = torch.zeros((batch, 6144 if seq == 384 else 512), dtype=torch.int32, device="cuda")
    api = capi.api()
    warps = (1, 8) if seq == 384 else (2, 2)
    api.check(api.convert_mask(seq, batch, *warps, 1, mask.data_ptr(), packed.data_ptr(), _stream()))
    qkv, scale = _activations(_generator(seed), (seq, batch, 3 * hidden), dtype)
    fmt = TensorFormat.CHW32 if dtype == "int8" else TensorFormat.LINEAR
    ins = [TensorDesc([seq, batch, 3 * hidden, 1, 1], TRT[dtype], fmt, scale),
           TensorDesc([batch, packed.shape[1]], DataType.INT32)]
    outs = [TensorDesc([seq, batch, hidden, 1, 1], TRT[dtype], fmt, scale)]
    out = torch.empty((seq, batch, hidden), dtype=TORCH[dtype], device="cuda")
    plugin, ws = _plugin(QKV, "4", _attention_fields(dtype, case["heads"], HEAD), ins, outs)
    return _plugin_call(plugin, ins, outs, [qkv, packed], [out], ws)


@functools.lru_cache(maxsize=None)
def _unfused_plugin(dtype, seq, batch, heads, head):
    """Configured once for its shape: the configuration times the routes that the shape has."""
    hidden = heads * head
    ins = [TensorDesc([seq, batch, 3 * hidden, 1, 1], TRT[dtype]), TensorDesc([batch, 1], DataType.INT32)]
    outs = [TensorDesc([seq, batch, hidden, 1, 1], TRT[dtype])]
    return (*_plugin(QKV, "4", _attention_fields(dtype, heads, head), ins, outs), ins, outs)


def _prepare_attention_unfused(case, seed):
    dtype, seq, batch, heads, head = (case[k] for k in ("dtype", "seq", "batch", "heads", "head"))
    plugin, ws, ins, outs = _unfused_plugin(dtype, seq, batch, heads, head)
    qkv, _ = _activations(_generator(seed), (seq, batch, 3 * heads * head), dtype)
    valid = torch.from_numpy(_lengths(case, seed).astype(np.int32)).cuda()
    out = torch.empty((seq, batch, heads * head), dtype=TORCH[dtype], device="cuda")
    return _plugin_call(plugin, ins, outs, [qkv, valid], [out], ws)


def _prepare_skipln(case, seed):
    dtype, shape = case["dtype"], (case["seq"], case["batch"], case["hidden"])
    g = _generator(seed)
    x, skip = _activations(g, shape, dtype)[0], _activations(g, shape, dtype)[0]
    d = TensorDesc([*shape, 1, 1], TRT[dtype])
    return _plugin_call(_skipln_plugin(dtype, case["hidden"]), [d, d], [d], [x, skip], [torch.empty_like(x)])


def _prepare_embln(case, seed):
    dtype, seq, batch, hidden = (case[k] for k in ("dtype", "seq", "batch", "hidden"))
    plugin = _embln_plugin(dtype, hidden)
    ids, segs = _tokens(_generator(seed), (seq, batch))
    lens = torch.from_numpy(_lengths(case, seed)).cuda()
    mask = (torch.arange(seq, device="cuda")[:, None] < lens[None, :]).to(torch.int32)
    ins = [TensorDesc([seq, batch], DataType.INT32)] * 3
    shapes = plugin.get_output_shapes(ins)
    outs = [TensorDesc(shapes[0], TRT[dtype]), TensorDesc(shapes[1], DataType.INT32)]
    out = torch.empty((seq, batch, hidden), dtype=TORCH[dtype], device="cuda")
    packed = torch.zeros(shapes[1], dtype=torch.int32, device="cuda")
    return _plugin_call(plugin, ins, outs, [ids, segs, mask], [out, packed])


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state):
    kind = state["kind"]
    if kind == "int8_encoder":
        api, b = state["api"], state["batches"]
        if len(b) == 1:
            q = b[0]
            api.check(api.encoder_enqueue(state["handle"], q.ids, q.segment_ids, q.cu_seqlens, q.batch, q.tokens,
                                          q.workspace, q.out, state["stream"]))
        else:
            api.check(api.encoder_enqueue_concurrent(state["handle"], b, len(b), state["stream"]))
        return state["result"]
    if kind == "fp16_encoder":
        return state["model"].enqueue(state["ids"], state["segs"], state["cu"])
    if state["plugin"].enqueue(state["ins"], state["outs"], state["inputs"], state["outputs"], state["workspace"],
                               state["stream"]) != 0:
        raise RuntimeError("enqueue failed")
    return state["result"]


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def _moments(case):
    """Sum of the lengths and of their squares."""
    lens = _lengths_of(case).astype(np.float64)
    return float(lens.sum()), float((lens * lens).sum())


def work(case):
    kind = case["kind"]
    if kind in ("int8_encoder", "fp16_encoder"):
        hidden, layers, size = (1024, 24, 1) if kind == "int8_encoder" else (768, 12, 2)
        tokens, squares = _moments(case)
        weights = 12 * hidden * hidden * layers
        return dict(bytes=weights * size + tokens * (8 + 3 * hidden * 2 + hidden * 2),
                    flops=2 * tokens * weights + 4 * squares * hidden * layers)
    if kind == "attention_var":
        hidden = case["heads"] * HEAD
        tokens, squares = _moments(case)
        return dict(bytes=4 * tokens * hidden * SIZE[case["dtype"]], flops=4 * squares * hidden)
    if kind in ("attention_fixed", "attention_unfused"):
        hidden, rows = case["heads"] * case.get("head", HEAD), case["seq"] * case["batch"]
        return dict(bytes=4 * rows * hidden * SIZE[case["dtype"]], flops=4 * case["seq"] * _moments(case)[0] * hidden)
    rows, hidden, size = case["seq"] * case["batch"], case["hidden"], SIZE[case["dtype"]]
    if kind == "skipln":
        return dict(bytes=3 * rows * hidden * size + 3 * hidden * size, flops=9 * rows * hidden)
    # every gathered row once, but no more rows than the tables have
    gathered = min(rows, VOCAB) + min(case["seq"], 512) + 2
    return dict(bytes=(rows + gathered) * hidden * size + 12 * rows, flops=9 * rows * hidden)


def tolerance(case):
    kind = case["kind"]
    if kind == "int8_encoder":
        # a probability or activation that rounds the other way moves an INT8 value by one step of amax / 127, and the
        # layers behind pass it on
        return {"rel": 1e-2, "max": 0.3}
    if kind == "fp16_encoder":
        return {"rel": 5e-3}
    if case["dtype"] == "int8":
        return {"rel": 1e-5, "differ": 1e-3}
    return {"rel": 2e-3 if case["dtype"] == "fp16" else 1e-5}
