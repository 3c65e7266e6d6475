"""The FP16 encoder chain (embedding -> [QKV GEMM, fused FP16 attention v5, projection, SkipLayerNorm v6 with bias,
FFN + GELU, FFN, SkipLayerNorm v6] x L) on the GPU, every operation checked against the CPU oracle applied to that
operation's own GPU inputs (|a - b| <= 2e-3 + 1e-2 |b|)."""
import numpy as np
import pytest

import oracle
from helpers import assert_fp_close, dev, dev_empty, host, ptr, rng, stream, sync
from tensorrt_amd.encoder import EncoderConfig
from tensorrt_amd.encoder_fp16 import Fp16BertEncoder

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    cfg = EncoderConfig(hidden=768, heads=12, ffn=3072, layers=2, vocab=1000, max_pos=512, max_seqlen=384, seed=11)
    enc = Fp16BertEncoder(cfg)
    r = rng(12)
    lens = np.array([50, 128, 7, 101, 1, 384])
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    ids = r.integers(0, cfg.vocab, T).astype(np.int32)
    segs = r.integers(0, 2, T).astype(np.int32)
    cap = {}
    out = enc.enqueue(ids, segs, cu, capture=cap)
    import torch
    torch.cuda.synchronize()
    return cfg, enc, ids, segs, cu, cap, out.cpu().numpy()


def test_embedding(setup):
    cfg, enc, ids, segs, cu, cap, _ = setup
    w = enc.emb_weights
    tabs = {k: w[k].astype(np.float16) for k in ("word", "pos", "tok")}
    ref, _, _ = oracle.embln(1, ids, segs, cu, w["beta"], w["gamma"], tabs["word"], tabs["pos"], tabs["tok"],
                             cfg.max_seqlen, len(cu) - 1)
    assert_fp_close(cap["emb"], ref, what="embedding")


@pytest.mark.parametrize("layer", [0, 1])
def test_layer_operations(setup, layer):
    cfg, enc, ids, segs, cu, cap, _ = setup
    E, N = cfg.hidden, cfg.heads
    L = enc.layers[layer]
    g = lambda k: cap[f"l{layer}.{k}"]
    x = cap["emb"] if layer == 0 else cap[f"l{layer - 1}.out"]

    def linear(name, src):
        lin = L[name]
        return oracle.fp16_linear(src, lin.w_h, lin.alpha_h, lin.bias_h, gelu=lin.gelu)

    def skipln(ln, src, skip):
        h = lambda a: a.astype(np.float16)
        return oracle.skipln(src, skip, h(L[ln + "_beta"]), h(L[ln + "_gamma"]), h(L[ln + "_bias"]))

    assert_fp_close(g("qkv"), linear("qkv", x), what="QKV projection")
    assert_fp_close(g("ctx"), oracle.mha_fused_f16_packed(g("qkv"), cu, N, 64), what="attention")
    assert_fp_close(g("ao"), linear("proj", g("ctx")), what="output projection")
    assert_fp_close(g("h"), skipln("ln1", g("ao"), x), what="SkipLayerNorm 1")
    assert_fp_close(g("m"), linear("ffn1", g("h")), what="feed-forward 1 + GELU")
    assert_fp_close(g("f"), linear("ffn2", g("m")), what="feed-forward 2")
    assert_fp_close(g("out"), skipln("ln2", g("f"), g("h")), what="SkipLayerNorm 2")


def test_output_is_finite_and_repeatable(setup):
    import torch
    cfg, enc, ids, segs, cu, cap, out = setup
    assert np.isfinite(out.astype(np.float32)).all() and float(np.abs(out.astype(np.float32)).max()) > 1.0
    again = enc.enqueue()
    torch.cuda.synchronize()
    assert np.array_equal(again.cpu().numpy().view(np.uint16), out.view(np.uint16))


@pytest.mark.parametrize("lens", [[1], [31], [33], [64, 1], [97], [128, 2], [257, 1, 3]])
def test_few_tokens_against_single_operations(setup, lens):
    """The native pass with few tokens (partial sums of the second feed-forward layer, added up in the normalisation)
    against the same network one operation at a time: the order of binary32 sums is all that differs."""
    import torch
    cfg, enc, ids, segs, cu, cap, out = setup
    r = rng(41 + sum(lens))
    c = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = int(c[-1])
    i, s = r.integers(0, cfg.vocab, t).astype(np.int32), r.integers(0, 2, t).astype(np.int32)
    want = enc.enqueue(i, s, c, capture={}).cpu().numpy()
    got = enc.enqueue(i, s, c)
    torch.cuda.synchronize()
    assert_fp_close(got.cpu().numpy(), want, atol=1e-2, what="native pass")   # a few binary16 steps of values up to ~4
    enc.enqueue(ids, segs, cu)


@pytest.fixture(scope="module")
def one_layer():
    """One-layer models: their intermediate buffers still hold that layer's values after a native pass."""
    made = {}

    def get(hidden, ffn):
        if hidden not in made:
            made[hidden] = Fp16BertEncoder(EncoderConfig(hidden=hidden, heads=hidden // 64, ffn=ffn, layers=1, vocab=500,
                                                         max_pos=512, max_seqlen=384, seed=13))
        return made[hidden]
    return get


@pytest.mark.parametrize("hidden,ffn", [(768, 3072), (1024, 4096), (512, 2048), (320, 2048)])
@pytest.mark.parametrize("lens", [[1], [32], [20, 13], [64], [70, 26]])
def test_normalisation_of_partial_sums(one_layer, hidden, ffn, lens):
    """Few tokens: the partial sums of the second feed-forward layer add up to that layer's accumulators, and the
    normalisation that reads them is the oracle's SkipLayerNorm of the layer's output."""
    import torch
    enc = one_layer(hidden, ffn)
    r = rng(44 + sum(lens))
    c = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    t = int(c[-1])
    enc._partial.zero_()   # at most four parts: the sums of parts that do not exist are 0
    out = enc.enqueue(r.integers(0, 500, t).astype(np.int32), r.integers(0, 2, t).astype(np.int32), c)
    torch.cuda.synchronize()
    sums = enc._partial.view(torch.float32)[:4 * t * hidden].cpu().numpy().reshape(4, t, hidden)
    assert np.abs(sums[1]).max() > 0, "more than one part"
    m, h = (enc.buf[k].cpu().numpy() for k in ("m", "h"))
    L = enc.layers[0]
    lin = L["ffn2"]
    acc = m.astype(np.float64) @ lin.w_h.astype(np.float64).T
    total = sums.astype(np.float64).sum(0)
    # ffn products of binary32 accumulations in any order: |error| <= ffn * 2^-24 * sum |m w|, far below that in practice
    bound = ffn * 2.0 ** -24 * (np.abs(m).astype(np.float64) @ np.abs(lin.w_h).astype(np.float64).T)
    assert (np.abs(total - acc) <= bound + 1e-12).all()
    f = oracle.fp16_linear(m, lin.w_h, lin.alpha_h, lin.bias_h)
    half = lambda a: a.astype(np.float16)
    want = oracle.skipln(f, h, half(L["ln2_beta"]), half(L["ln2_gamma"]), half(L["ln2_bias"]))
    assert_fp_close(out.cpu().numpy(), want, what="SkipLayerNorm of partial sums")


@pytest.mark.parametrize("hidden,ffn", [(768, 3072), (1024, 4096), (512, 2048), (320, 2048)])
@pytest.mark.parametrize("scaled", [False, True])
def test_normalisation_of_partial_sums_rounds_as_the_layer_and_the_normalisation_do(one_layer, hidden, ffn, scaled):
    """The bytes of the normalisation that reads partial sums are those of the normalisation by itself behind a layer with
    the same sums: the layer's multiply-add rounded to binary16 once (`scaled`: by an alpha and a beta that leave something
    to round), the normalisation's rounded to binary32 first."""
    import torch
    enc = one_layer(hidden, ffn)
    api, L = enc.api, enc.layers[0]
    r = rng(48 + hidden)
    c = np.array([0, 20, 64], np.int32)
    t = int(c[-1])
    ids, segs = r.integers(0, 500, t).astype(np.int32), r.integers(0, 2, t).astype(np.int32)
    alpha, beta = np.ones(hidden, np.float32), np.zeros(hidden, np.float32)
    if scaled:
        alpha, beta = r.uniform(0.5, 1.5, hidden).astype(np.float32), (0.1 * r.standard_normal(hidden)).astype(np.float32)
    lin = L["ffn2"]
    d = [dev(L[k].astype(np.float16)) for k in ("ln2_beta", "ln2_gamma", "ln2_bias")]
    got, want = [], []
    lin.alpha.copy_(torch.from_numpy(alpha))
    lin.beta.copy_(torch.from_numpy(beta))
    try:
        for _ in range(8):   # one result in some 10^4 depends on how often it was rounded
            enc._partial.zero_()
            ids = np.roll(ids, 1)
            out = enc.enqueue(ids, segs, c)
            sync()
            got.append(host(out))
            sums = enc._partial.view(torch.float32)[:4 * t * hidden].cpu().numpy().reshape(4, t, hidden)
            assert np.abs(sums[1]).max() > 0, "more than one part"
            total = ((sums[0] + sums[1]) + sums[2]) + sums[3]   # binary32, in the kernel's order
            f = (total.astype(np.float64) * alpha + beta).astype(np.float16)
            o, d_f = dev_empty((t, hidden), np.float16), dev(f)
            api.check(api.skip_layer_norm_fp16(stream(), hidden, t * hidden, ptr(d_f), ptr(enc.buf["h"]), ptr(d[0]), ptr(d[1]),
                                               ptr(o), ptr(d[2])))
            sync()
            want.append(host(o))
    finally:
        lin.alpha.fill_(1.0)
        lin.beta.zero_()
    got, want = np.array(got).view(np.uint16), np.array(want).view(np.uint16)
    assert np.array_equal(got, want), f"{int((got != want).sum())} of {got.size} values differ"


def test_passes_asked_for_on_another_stream(setup):
    """Passes of changing sizes asked for while another stream is current, one after the other without waiting: memory that
    a pass reads or writes is not given to a later one before it is through with it."""
    import torch
    cfg, enc, ids, segs, cu, cap, out = setup
    r = rng(43)
    batches, want = [], []
    for n in (300, 20, 300, 7, 129, 300, 20, 64):
        c = np.array([0, n // 2, n], np.int32)
        batches.append((r.integers(0, cfg.vocab, n).astype(np.int32), r.integers(0, 2, n).astype(np.int32), c))
        want.append(enc.enqueue(*batches[-1]).cpu().numpy())
    home, other = torch.cuda.current_stream(), torch.cuda.Stream()
    got = []
    with torch.cuda.stream(other):
        for b in batches:
            x = enc.enqueue(*b)
            # what the caching allocator hands out on this stream is no memory of a pass in flight
            junk = [torch.full((n, c), 7, dtype=torch.float16, device="cuda") for n in (300, 129, 64) for c in (768, 3072)]
            junk += [torch.full((1 << k,), 7, dtype=torch.int32, device="cuda") for k in range(2, 11)]
            with torch.cuda.stream(home):
                got.append(x.clone())
            del junk
    torch.cuda.synchronize()
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy().view(np.uint16), w.view(np.uint16))
    enc.enqueue(ids, segs, cu)
