"""Host-side logic of the encoder builder and of the native passes that needs no GPU."""
import ctypes as C

import numpy as np
import pytest

from tensorrt_amd import capi
from tensorrt_amd.encoder import split_runs


def _cu(lens):
    return np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def test_split_runs_balances_tokens_on_sequence_boundaries():
    lens = np.random.default_rng(1).integers(128, 385, 128)
    cu = _cu(lens)
    runs = split_runs(cu, 2)
    assert runs[0][0] == 0 and runs[-1][1] == 128 and runs[0][1] == runs[1][0]
    a, b = (int(cu[hi] - cu[lo]) for lo, hi in runs)
    assert abs(a - b) <= int(lens.max())          # within one sequence of the middle
    three = split_runs(cu, 3)
    assert [r[0] for r in three[1:]] == [r[1] for r in three[:-1]] and len(three) == 3
    sizes = [int(cu[hi] - cu[lo]) for lo, hi in three]
    assert max(sizes) - min(sizes) <= 2 * int(lens.max())


def test_split_runs_degenerate_batches():
    assert split_runs(_cu([77]), 2) == [(0, 1)]                 # one sequence cannot be cut
    assert split_runs(_cu([5, 9]), 4) == [(0, 1), (1, 2)]       # never more runs than sequences
    assert split_runs(_cu([0, 0, 150, 40]), 2) == [(0, 3), (3, 4)]
    assert split_runs(_cu([90, 60, 0, 0]), 2) == [(0, 1), (1, 4)]
    assert split_runs(_cu([0, 0, 0, 12]), 2) == [(1, 4)]        # a run of empty sequences is left out
    assert split_runs(_cu([0, 0]), 2) == []                     # nothing to compute
    whole = split_runs(_cu([3, 4, 5]), 1)
    assert whole == [(0, 3)]


# ---- trtamd_fp16_encoder_enqueue: what it refuses, with addresses that nothing is ever launched on (no plugin objects) ----

def _fp16_pass(tokens=32, hidden=768, ffn=3072, layers=2):
    """Arguments of a pass whose pointers are all in order; 16-byte aligned addresses that are never read."""
    address = lambda: 0x10000
    config = capi.Fp16EncoderConfig(hidden=hidden, ffn=ffn, layers=layers, max_seqlen=128, embedding=None)
    lays = (capi.Fp16EncoderLayer * layers)()
    for d in lays:
        for name in ("qkv", "proj", "ffn1", "ffn2"):
            setattr(d, name, capi.Fp16EncoderLinear(address(), address(), address()))
        d.ln2_gamma = d.ln2_beta = d.ln2_bias = address()
    batch = capi.Fp16EncoderBatch(batch=1, tokens=tokens, partial=address(), partial_bytes=2 << 20)
    for name in ("ids", "segment_ids", "cu_seqlens", "mask", "longest", "x", "qkv", "ctx", "ao", "h", "m", "f", "emb2"):
        setattr(batch, name, address())
    return config, lays, batch


def _refusal(config, lays, batch):
    api = capi.api()
    assert api.fp16_encoder_enqueue(C.byref(config), lays, C.byref(batch), None) != 0
    return api.last_error_str()


@pytest.mark.parametrize("tokens", [32, 1000])
def test_fp16_pass_checks_every_layer_before_its_first_launch(tokens):
    """A short pass (partial sums) refuses what a long one does: missing or misaligned weights and vectors of any layer."""
    assert "no plugin object" in _refusal(*_fp16_pass(tokens))     # nothing else is wrong with these arguments
    for layer in (0, 1):
        for name in ("qkv", "proj", "ffn1", "ffn2"):
            for field in ("w", "alpha", "beta"):
                for value, what in ((None, "null pointer"), (0x10004, "aligned")):
                    args = _fp16_pass(tokens)
                    setattr(getattr(args[1][layer], name), field, value)
                    assert what in _refusal(*args), (layer, name, field, value)
    config, lays, batch = _fp16_pass(tokens)
    config.ffn = 3080                                              # no multiple of 32
    assert "multiples of 32" in _refusal(config, lays, batch)


@pytest.mark.parametrize("spoil", [
    lambda config, lays, batch: setattr(lays[1], "ln2_bias", None),
    lambda config, lays, batch: setattr(lays[1], "ln2_gamma", 0x10002),
    lambda config, lays, batch: setattr(batch, "partial", 0x10004),
    lambda config, lays, batch: setattr(batch, "partial", None),
    lambda config, lays, batch: setattr(batch, "partial_bytes", 4096),
])
def test_fp16_pass_without_what_partial_sums_need_is_not_refused(spoil):
    args = _fp16_pass()
    spoil(*args)
    assert "no plugin object" in _refusal(*args)
