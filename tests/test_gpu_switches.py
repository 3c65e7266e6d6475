"""Every tuning switch of the library (README, "Tuning switches") selects a kernel variant other than the default one.
Each setting is put through the parity checks of the kernel it changes, in this process, through the test hook that
stands in for the environment variable of the same name (include/trtamd_test_hooks.h): the variants must give what
the default choice gives, to the same bar against the oracle."""
import contextlib
import ctypes as C

import numpy as np
import pytest

import oracle
from helpers import (assert_fp_close, assert_int8_close, attention_f64, dev, dev_empty, half2_bits, host,
                     int8_attention_parity, ptr, quantize_amax, rng, stream, sync)
from tensorrt_amd import capi
from test_attention_routes_host import STREAM, TURNS, WHOLE, decode
from test_gpu_linear import interleave, problem, run_fp16, run_gpu

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def tuning(name, value):
    api = capi.api()
    api.check(api.test_set_tuning(name.encode(), value))
    try:
        yield
    finally:
        api.check(api.test_reset_tuning(name.encode()))


def route(dtype, p):
    """What the launcher makes of a call's parameters."""
    return decode(capi.api().test_fmha_route(dtype, C.byref(p)))


def test_unknown_switch_is_refused():
    api = capi.api()
    assert api.test_set_tuning(b"TRTAMD_NO_SUCH_SWITCH", 1) == 2
    assert "unknown tuning switch" in api.last_error_str()
    assert api.test_reset_tuning(b"TRTAMD_NO_SUCH_SWITCH") == 2


LINEAR_SETTINGS = [("TRTAMD_LINEAR_DIRECT", 0), ("TRTAMD_LINEAR_PERSISTENT", 0), ("TRTAMD_LINEAR_PARTIAL_ROUND", 0),
                   ("TRTAMD_LINEAR_PARTIAL_ROUND", 100)]


@pytest.mark.parametrize("T", [67 * 256 + 60, 133 * 256 + 60])
def test_remainder_pieces_against_remainder_tiles(T):
    """Large tiles as a partial round with 60 tokens behind them, and as a whole round with 1340: those go in 64 x 64
    pieces whose wavefronts split k, with TRTAMD_LINEAR_PIECES=0 in 128 x 128 tiles; both must give the oracle's
    accumulator-exact results and the same bytes."""
    with tuning("TRTAMD_LINEAR_PLAN", 0):   # the cost model may prefer smaller tiles for all of it
        _remainder_pieces_against_remainder_tiles(T, 256, 512)


def _remainder_pieces_against_remainder_tiles(T, K, N):
    a, w, alpha, beta = problem(93, T, K, N)
    ref = oracle.int8_linear(a, w, alpha, beta, oracle.LINEAR_AFFINE, out_interleaved=True)
    pieces = run_gpu(a, w, alpha, beta, capi.LINEAR_AFFINE, a_il=True, out_il=True, w_il=True)
    with tuning("TRTAMD_LINEAR_PIECES", 0):
        tiles = run_gpu(a, w, alpha, beta, capi.LINEAR_AFFINE, a_il=True, out_il=True, w_il=True)
    assert_int8_close(pieces, ref, what="pieces", max_frac_off=1e-3)
    assert np.array_equal(pieces, tiles)
    q = float(np.float32(127.0 / 4.0))
    al, be = (alpha * 0.06).astype(np.float32), (beta * 0.02).astype(np.float32)
    ref = oracle.int8_linear(a, w, al, be, oracle.LINEAR_GELU, out_scale=q, out_interleaved=True)
    pieces = run_gpu(a, w, al, be, capi.LINEAR_GELU, out_scale=q, a_il=True, out_il=True, w_il=True)
    with tuning("TRTAMD_LINEAR_PIECES", 0):
        tiles = run_gpu(a, w, al, be, capi.LINEAR_GELU, out_scale=q, a_il=True, out_il=True, w_il=True)
    assert_int8_close(pieces, ref, what="pieces, GELU", max_frac_off=2e-3)
    assert np.array_equal(pieces, tiles)


@pytest.mark.parametrize("name,value", LINEAR_SETTINGS)
@pytest.mark.parametrize("il", [True, False])
@pytest.mark.parametrize("T,K,N", [(777, 1024, 512), (70 * 256 + 9, 256, 512)])
def test_linear_variants(T, K, N, name, value, il):
    """Ragged token counts with whole 256-token tiles and a remainder, N and K multiples of 256: less than half a round of
    large tiles (which run only with TRTAMD_LINEAR_PARTIAL_ROUND=0) and more (which run unless it is 100).  Accumulators
    bit-exact, affine and GELU outputs to the oracle's bar and equal to the default setting's bytes."""
    with tuning("TRTAMD_LINEAR_PLAN", 0):   # large tiles wherever the setting allows them
        _linear_variants(T, K, N, name, value, il)


def _linear_variants(T, K, N, name, value, il):
    a, w, alpha, beta = problem(91, T, K, N, full_range=True)
    with tuning(name, value):
        raw = run_gpu(a, w, None, None, capi.LINEAR_RAW_INT32, a_il=il, w_il=il)
    assert np.array_equal(raw, oracle.int8_linear(a, w, epilogue=oracle.LINEAR_RAW_INT32))
    a, w, alpha, beta = problem(92, T, K, N)
    for epi, oepi, frac in ((capi.LINEAR_AFFINE, oracle.LINEAR_AFFINE, 1e-3), (capi.LINEAR_GELU, oracle.LINEAR_GELU, 2e-3)):
        # GELU: pre-activations of a few units either side of zero, as in test_gpu_linear.test_gelu_int8
        scale = 1.0 if epi == capi.LINEAR_AFFINE else float(np.float32(127.0 / 4.0))
        al = alpha if epi == capi.LINEAR_AFFINE else (alpha * 0.06).astype(np.float32)
        be = beta if epi == capi.LINEAR_AFFINE else (beta * 0.02).astype(np.float32)
        default = run_gpu(a, w, al, be, epi, out_scale=scale, a_il=il, out_il=il, w_il=il)
        with tuning(name, value):
            got = run_gpu(a, w, al, be, epi, out_scale=scale, a_il=il, out_il=il, w_il=il)
        ref = oracle.int8_linear(a, w, al, be, oepi, out_scale=scale, out_interleaved=il)
        assert_int8_close(got, ref, what=f"{name}={value} epilogue {epi}", max_frac_off=frac)
        assert np.array_equal(got, default), f"{name}={value}: bytes differ from the default kernel choice"


# large tiles: 132 of 256 CUs with one token behind them, 136 with 255, a round with 80 tiles' worth of smaller ones behind
LARGE_TILE_SHAPES = [(33 * 256 + 1, 256, 1024), (34 * 256 + 255, 512, 1024), (84 * 256 + 33, 256, 1024)]


@pytest.mark.parametrize("plan,T,K,N", [(plan, *shape) for plan in range(1, 10) for shape in
                                        [(1, 64, 32), (33, 192, 96), (130, 448, 160), (259, 768, 288)]]
                         + [(0, *shape) for shape in LARGE_TILE_SHAPES])
def test_linear_plans(plan, T, K, N):
    """Every tile shape of the linear layers at the edges of its tiles (one token, one past a block, channels and k that
    are no multiple of a tile; k shorter than the ring of stages), both layouts, INT8 and FP16: the oracle's bar, and
    INT8 bytes equal to the register-staged kernel's."""
    a, w, alpha, beta = problem(95 + T, T, K, N)
    for il in (True, False):
        for epi, oepi, frac, q in ((capi.LINEAR_AFFINE, oracle.LINEAR_AFFINE, 1e-3, 1.0),
                                   (capi.LINEAR_GELU, oracle.LINEAR_GELU, 2e-3, float(np.float32(127.0 / 4.0)))):
            al, be = (alpha, beta) if q == 1.0 else ((alpha * 0.06).astype(np.float32), (beta * 0.02).astype(np.float32))
            with tuning("TRTAMD_LINEAR_DIRECT", 0):
                want = run_gpu(a, w, al, be, epi, out_scale=q, a_il=il, out_il=il, w_il=il)
            with tuning("TRTAMD_LINEAR_PLAN", plan):
                got = run_gpu(a, w, al, be, epi, out_scale=q, a_il=il, out_il=il, w_il=il)
            ref = oracle.int8_linear(a, w, al, be, oepi, out_scale=q, out_interleaved=il)
            # one value of a small output is more than the allowed share
            assert_int8_close(got, ref, what=f"plan {plan} epilogue {epi}", max_frac_off=max(frac, 1.5 / got.size))
            assert np.array_equal(got, want)
    r = rng(96 + T)
    x = r.standard_normal((T, K)).astype(np.float16)
    w = (0.05 * r.standard_normal((N, K))).astype(np.float16)
    for gelu in (0, 1):
        with tuning("TRTAMD_LINEAR_PLAN", plan):
            got = run_fp16(x, w, np.ones(N, np.float32), beta * 0.1, bool(gelu))
        ref = oracle.fp16_linear(x, w, np.ones(N, np.float32), beta * 0.1, gelu=bool(gelu))
        assert_fp_close(got, ref, what=f"plan {plan} FP16")


@pytest.mark.parametrize("plan,T", [(9, 65535 * 32), (9, 65535 * 32 + 1), (8, 65535 * 32 + 1)])
def test_pieces_up_to_the_extent_of_their_grid(plan, T):
    """More pieces of tokens than the second extent of a grid holds are left to another plan."""
    a, w, alpha, beta = problem(99, T, 64, 32)
    want = run_gpu(a, w, alpha, beta, capi.LINEAR_AFFINE, a_il=True, out_il=True, w_il=True)
    with tuning("TRTAMD_LINEAR_PLAN", plan):
        got = run_gpu(a, w, alpha, beta, capi.LINEAR_AFFINE, a_il=True, out_il=True, w_il=True)
    assert np.array_equal(got, want)


# tiles of linear operands: stages of 128 bytes of k (64 FP16 values), rings of two to five of them.  One stage, as many as
# the ring has and one more; token and channel counts on both sides of a tile's edge.
WHOLE_LINES = [(plan, *shape) for plan in (2, 4, 5, 10, 11, 12, 13, 14) for shape in
               [(1, 64, 32), (63, 128, 96), (191, 192, 128), (193, 256, 160), (257, 384, 288)]]
# rows that end within a line: stages of 64 bytes and tiles of their own, k longer than their rings (three and four stages) and
# as long as one stage
HALF_LINES = [(plan, *shape) for plan in (1, 2, 3, 4) for shape in
              [(1, 32, 32), (65, 160, 64), (130, 608, 224), (257, 96, 160), (255, 288, 128)]]


@pytest.mark.parametrize("plan,T,K,N", WHOLE_LINES + HALF_LINES)
def test_linear_tiles_of_linear_operands(plan, T, K, N):
    """FP16 against binary64 and against the pieces' results; INT8 with linear operands byte for byte against the
    register-staged kernel; every shape through the kernel that it is listed for."""
    with tuning("TRTAMD_LINEAR_PLAN", plan):
        assert capi.api().test_linear_plan(0, T, 2 * K, N, 0) == plan == capi.api().test_linear_plan(0, T, 2 * K, N, 1)
    r = rng(97 + T)
    x = r.standard_normal((T, K)).astype(np.float16)
    w = (0.05 * r.standard_normal((N, K))).astype(np.float16)
    alpha, beta = r.uniform(0.5, 1.5, N).astype(np.float32), (0.1 * r.standard_normal(N)).astype(np.float32)
    exact = (x.astype(np.float64) @ w.astype(np.float64).T) * alpha + beta
    for gelu in (False, True):
        with tuning("TRTAMD_LINEAR_PLAN", plan):
            got = run_fp16(x, w, alpha, beta, gelu)
        with tuning("TRTAMD_LINEAR_PLAN", 9):
            pieces = run_fp16(x, w, alpha, beta, gelu)
        assert_fp_close(got, oracle.fp16_linear(x, w, alpha, beta, gelu=gelu), what=f"plan {plan}")
        # either kernel rounds a binary32 sum once: they differ by a unit in the last place where the sums straddle a tie
        assert_fp_close(got, pieces, atol=2.0 ** -14, rtol=2.0 ** -10, what=f"plan {plan} against the pieces")
        if not gelu:
            assert_fp_close(got, exact, what=f"plan {plan} against binary64")
    a, w8, al, be = problem(98 + T, T, 2 * K, N)
    for out_il in (False, True):
        with tuning("TRTAMD_LINEAR_DIRECT", 0):
            want = run_gpu(a, w8, al, be, capi.LINEAR_AFFINE, out_il=out_il)
        with tuning("TRTAMD_LINEAR_PLAN", plan):
            got = run_gpu(a, w8, al, be, capi.LINEAR_AFFINE, out_il=out_il)
        assert np.array_equal(got, want)


# pieces of linear operands: whole lines (K a multiple of 64 FP16 values; four wavefronts, rings of two and three stages) and
# rows that end within a line (eight, rings of three and four).  Fewer stages than wavefronts, as many as their rings have and
# one more, wavefronts with fewer than the others or none.
@pytest.mark.parametrize("plan", [8, 9])
@pytest.mark.parametrize("T,K,N", [(1, 64, 32), (33, 256, 96), (64, 512, 32), (65, 576, 160), (31, 832, 64), (70, 1600, 96),
                                   (32, 3072, 128), (33, 32, 64), (63, 608, 96), (65, 1056, 32)])
def test_pieces_of_linear_operands(plan, T, K, N):
    """FP16 against binary64 and the oracle; INT8 byte for byte against the register-staged kernel."""
    r = rng(92 + T)
    x = r.standard_normal((T, K)).astype(np.float16)
    w = (0.05 * r.standard_normal((N, K))).astype(np.float16)
    alpha, beta = r.uniform(0.5, 1.5, N).astype(np.float32), (0.1 * r.standard_normal(N)).astype(np.float32)
    with tuning("TRTAMD_LINEAR_PLAN", plan):
        assert capi.api().test_linear_plan(0, T, 2 * K, N, 0) == plan
        got = run_fp16(x, w, alpha, beta, False)
        gelu = run_fp16(x, w, alpha, beta, True)
    assert_fp_close(got, (x.astype(np.float64) @ w.astype(np.float64).T) * alpha + beta, what=f"plan {plan} against binary64")
    assert_fp_close(gelu, oracle.fp16_linear(x, w, alpha, beta, gelu=True), what=f"plan {plan} GELU")
    a, w8, al, be = problem(93 + T, T, 2 * K, N)
    for out_il in (False, True):
        with tuning("TRTAMD_LINEAR_DIRECT", 0):
            want = run_gpu(a, w8, al, be, capi.LINEAR_AFFINE, out_il=out_il)
        with tuning("TRTAMD_LINEAR_PLAN", plan):
            got = run_gpu(a, w8, al, be, capi.LINEAR_AFFINE, out_il=out_il)
        assert np.array_equal(got, want)


# the same tiles of interleaved operands: stages of 64 bytes, rings of four and five
@pytest.mark.parametrize("plan", [7, 10, 11, 12])
@pytest.mark.parametrize("T,K,N", [(1, 64, 32), (191, 256, 128), (193, 320, 160), (257, 384, 288), (130, 1088, 224)])
def test_linear_tiles_of_interleaved_operands(plan, T, K, N):
    """Byte for byte against the register-staged kernel, affine and GELU, either output layout."""
    a, w, alpha, beta = problem(94 + T, T, K, N)
    for epi, scale, f in ((capi.LINEAR_AFFINE, 1.0, 1.0), (capi.LINEAR_GELU, float(np.float32(127.0 / 4.0)), 0.06)):
        al, be = (alpha * f).astype(np.float32), (beta * f / 3).astype(np.float32)
        for out_il in (False, True):
            with tuning("TRTAMD_LINEAR_DIRECT", 0):
                want = run_gpu(a, w, al, be, epi, out_scale=scale, a_il=True, w_il=True, out_il=out_il)
            with tuning("TRTAMD_LINEAR_PLAN", plan):
                got = run_gpu(a, w, al, be, epi, out_scale=scale, a_il=True, w_il=True, out_il=out_il)
            assert np.array_equal(got, want)


def test_fp16_tiles_write_nothing_behind_the_last_row():
    import torch
    api = capi.api()
    T, K, N = 130, 128, 96
    r = rng(99)
    x, w = dev(r.standard_normal((T, K)).astype(np.float16)), dev(r.standard_normal((N, K)).astype(np.float16))
    one, zero = dev(np.ones(N, np.float32)), dev(np.zeros(N, np.float32))
    for plan in (2, 4, 5, 10, 11, 12, 13, 14):
        out = dev_empty((T + 200, N), np.float16, fill=-7)
        p = capi.Fp16LinearParams(ptr(x), ptr(w), ptr(one), ptr(zero), ptr(out), T, K, N, capi.LINEAR_AFFINE)
        with tuning("TRTAMD_LINEAR_PLAN", plan):
            api.check(api.fp16_linear(stream(), C.byref(p)))
        torch.cuda.synchronize()
        assert (host(out)[T:] == -7).all() and (host(out)[:T] != -7).any()


FMHA_SETTINGS = [("TRTAMD_FMHA_GENERIC", 1), ("TRTAMD_FMHA_QSPLIT", 1), ("TRTAMD_FMHA_QSPLIT", 2),
                 ("TRTAMD_FMHA_QSPLIT", 3), ("TRTAMD_FMHA_QSPLIT", 4), ("TRTAMD_FMHA_RANKED", 0),
                 ("TRTAMD_FMHA_RANKED", 1)]


@pytest.mark.parametrize("name,value", FMHA_SETTINGS)
@pytest.mark.parametrize("interleaved", [False, True])
def test_int8_attention_variants(name, value, interleaved):
    r = rng(1200 + value)
    B, N, S = 5, 3, 384
    lens = np.array([384, 1, 200, 65, 129])
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv, s_q = quantize_amax(r.standard_normal((T, 3 * N * 64)).astype(np.float32))
    s1, ss, s2 = np.float32(s_q * s_q * 0.125), np.float32(127.0), np.float32(s_q / 127.0 / 0.02)
    default = int8_attention_parity(qkv, cu, N, s1, ss, s2, interleaved, S=S)
    with tuning(name, value):
        int8_attention_parity(qkv, cu, N, s1, ss, s2, interleaved, S=S, expect=default)


# In FP16 only the kernel of many units of more than 384 keys shares a unit's queries by the launch size; where K and V take
# turns in LDS a workgroup has 64 of them.
@pytest.mark.parametrize("name,value,S,lens", [(n, v, 512, [512, 7, 385, 130] * 22) for n, v in FMHA_SETTINGS]
                         + [(n, v, 384, [384, 7, 250, 130]) for n, v in FMHA_SETTINGS if n != "TRTAMD_FMHA_QSPLIT"])
def test_fp16_attention_variants(name, value, S, lens):
    api = capi.api()
    r = rng(1300 + value)
    B, N = len(lens), 3
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv = (r.standard_normal((T, N, 3, 64)) * 0.7).astype(np.float16)
    d_qkv, d_cu = dev(qkv), dev(cu)

    def run():
        out = dev_empty((T, N * 64), np.float16, fill=0)
        p = capi.FmhaParams()
        p.qkv_ptr, p.o_ptr, p.cu_seqlens = ptr(d_qkv), ptr(out), ptr(d_cu)
        p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * N * 64, 2 * N * 64
        p.b, p.h, p.s, p.d = B, N, S, 64
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(0.125), half2_bits(1.0), half2_bits(1.0)
        api.check(api.fused_mha_run(stream(), 1, C.byref(p)))
        sync()
        return host(out)

    default = run()
    with tuning(name, value):
        got = run()
    for b in range(B):
        lo, hi = int(cu[b]), int(cu[b + 1])
        for n in range(N):
            want = attention_f64(qkv[lo:hi, n, 0], qkv[lo:hi, n, 1], qkv[lo:hi, n, 2], 0.125)
            assert_fp_close(got[lo:hi, n * 64:(n + 1) * 64], want, what=f"{name}={value} sequence {b} head {n}")
    # the specialised and the general kernel sum in different orders; the other switches only move work around
    if name == "TRTAMD_FMHA_GENERIC":
        assert_fp_close(got, default, atol=1e-3, rtol=2e-3, what="general kernel vs prefix kernel")
    else:
        assert np.array_equal(got.view(np.uint16), default.view(np.uint16)), f"{name}={value}: bits differ from the default"


@pytest.mark.parametrize("B", [1, 63, 64, 65, 127, 128, 129])
def test_longest_first_order_reaches_every_sequence(B):
    """The longest-first order on either side of what a wavefront keeps in its registers, with empty sequences, many of one
    length and one longer than the kernel serves whole: the bytes of the natural order."""
    r = rng(1500 + B)
    lens = r.integers(0, 40, B)
    lens[:: 3] = 17
    lens[B // 2] = 70
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T, N, S = int(cu[-1]), 2, 64
    qkv, s_q = quantize_amax(r.standard_normal((T, 3 * N * 64)).astype(np.float32))
    d_qkv, d_cu = dev(interleave(qkv)), dev(cu)
    api = capi.api()
    outs = []
    for ranked in (0, 1):
        out = dev_empty((N * 2, T, 32), np.int8, fill=55)
        p = capi.FmhaParams()
        p.qkv_ptr, p.o_ptr, p.cu_seqlens = ptr(d_qkv), ptr(out), ptr(d_cu)
        p.qkv_stride_in_bytes = p.o_stride_in_bytes = T
        p.b, p.h, p.s, p.d, p.interleaved = B, N, S, 64, 1
        bits = lambda x: int(np.float32(x).view(np.uint32))
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = bits(s_q * s_q * 0.125), bits(127.0), bits(s_q / 127.0 / 0.02)
        with tuning("TRTAMD_FMHA_RANKED", ranked):
            api.check(api.fused_mha_run(stream(), 2, C.byref(p)))
            sync()
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1])
    assert all((outs[0][:, cu[b]:cu[b + 1]] != 55).any() for b in range(B) if lens[b])


# (data type, sequences, heads, longest), the workgroups whose rounds change places, longest first: whole pairs of rounds, some
# workgroups more and one pair short, FP16 with 64 and with 128 queries per workgroup, INT8 units in one, two and four parts; INT8
# sequences that all have the length in natural order; and launches without any such rounds.
@pytest.mark.parametrize("dtype,B,N,S,backwards,ranked", [
    (1, 128, 1, 256, 512, False), (1, 255, 1, 200, 512, False), (1, 257, 1, 256, 1024, False), (1, 65, 1, 450, 512, False),
    (1, 43, 2, 321, 512, True), (1, 127, 1, 384, 512, True), (1, 192, 2, 190, 512, True), (1, 511, 1, 192, 512, True),
    (1, 513, 1, 192, 1024, True), (1, 128, 1, 512, 512, True), (1, 171, 1, 384, 512, True), (1, 342, 1, 384, 1024, True),
    (1, 1537, 1, 192, 3072, False), (1, 769, 1, 448, 3072, False),
    (2, 129, 1, 384, 512, True), (2, 192, 2, 190, 512, True), (2, 400, 1, 190, 512, True), (2, 144, 2, 330, 512, True),
    (2, 160, 5, 128, 512, True), (2, 1025, 1, 128, 1024, True), (2, 768, 1, 192, 512, True), (2, 193, 1, 256, 512, False),
    (2, 255, 1, 250, 512, False), (2, 400, 1, -192, 512, False), (2, 200, 3, -384, 1024, False),
    (1, 513, 1, 64, 0, False), (1, 240, 1, 320, 512, True), (1, 256, 1, 384, 0, True), (1, 1024, 1, 384, 0, False),
    (2, 100, 1, 384, 0, False), (2, 257, 1, 190, 0, True), (2, 800, 1, -192, 0, False)])
def test_rounds_that_go_backwards_reach_every_unit(dtype, B, N, S, backwards, ranked):
    """The order that the launcher chooses writes the bytes of the sequences' own order, and of every unit."""
    r = rng(1800 + B + abs(S))
    if S < 0: # all of this length
        S = -S
        lens = np.full(B, S)
    else:
        lens = r.integers(1, min(S, 40 if B > 600 else S) + 1, B)
        lens[0], lens[B // 2], lens[-1] = S, 0, 1
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv = r.standard_normal((T, 3 * N * 64)).astype(np.float32)
    bits = lambda x: int(np.float32(x).view(np.uint32))
    p = capi.FmhaParams()
    if dtype == 2:
        q, s_q = quantize_amax(qkv)
        d_qkv = dev(interleave(q))
        p.qkv_stride_in_bytes = p.o_stride_in_bytes = T
        p.interleaved = 1
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = bits(s_q * s_q * 0.125), bits(127.0), bits(s_q / 127.0 / 0.02)
    else:
        d_qkv = dev(qkv.astype(np.float16))
        p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * N * 64, 2 * N * 64
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(0.125), half2_bits(1.0), half2_bits(1.0)
    d_cu = dev(cu)
    p.qkv_ptr, p.cu_seqlens = ptr(d_qkv), ptr(d_cu)
    p.b, p.h, p.s, p.d = B, N, S, 64
    assert (route(dtype, p).backwards, route(dtype, p).ranked) == (backwards, ranked)
    api = capi.api()
    outs = []
    for order in (None, 0):
        out = dev_empty((N * 2, T, 32), np.int8, fill=55) if dtype == 2 else dev_empty((T, N * 64), np.float16, fill=-7)
        p.o_ptr = ptr(out)
        with tuning("TRTAMD_FMHA_RANKED", -1 if order is None else order):
            api.check(api.fused_mha_run(stream(), dtype, C.byref(p)))
            sync()
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1])
    units = outs[0].reshape(N, 2, T, 32).transpose(2, 0, 1, 3).reshape(T, N, 64) if dtype == 2 else outs[0].reshape(T, N, 64)
    assert (units != (55 if dtype == 2 else -7)).any(axis=2).all()


# launches that fill the chip: 768 workgroups of 128 queries, or of 64 with at most 64 keys; lengths on either side of a
# wavefront's 32 queries, a workgroup's 128, half a block and a block of keys; scores whose maximum grows from block to block and
# scores of one size
@pytest.mark.parametrize("S,B,N,kernel", [(64, 192, 4, TURNS), (128, 192, 4, STREAM), (384, 64, 4, STREAM), (512, 48, 4, STREAM)])
@pytest.mark.parametrize("growing", [False, True])
@pytest.mark.parametrize("ranked", [0, 1])
def test_fp16_attention_of_full_launches(S, B, N, kernel, growing, ranked):
    api = capi.api()
    r = rng(1600 + S)
    edges = [n for n in (1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 161, 255, 257, 383, 384, 449, 511, 512) if n <= S]
    lens = np.array([edges[i % len(edges)] for i in range(B)])
    lens[3] = 0
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv = r.standard_normal((T, N, 3, 64))
    if growing:
        for b in range(B):
            # scores up to about +-8 x 90 x 0.125: a block's largest is e^10 and more above the one before
            qkv[cu[b]:cu[b + 1], :, 1] *= (1 + np.arange(lens[b]) * 0.25)[:, None, None]
    qkv = qkv.astype(np.float16)
    d_qkv, d_cu = dev(qkv), dev(cu)
    out = dev_empty((T + 64, N * 64), np.float16, fill=-7)
    p = capi.FmhaParams()
    p.qkv_ptr, p.o_ptr, p.cu_seqlens = ptr(d_qkv), ptr(out), ptr(d_cu)
    p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * N * 64, 2 * N * 64
    p.b, p.h, p.s, p.d = B, N, S, 64
    p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(0.125), half2_bits(1.0), half2_bits(1.0)
    assert route(1, p).kernel == kernel and route(1, p).parts * B * N == 768
    with tuning("TRTAMD_FMHA_RANKED", ranked):
        api.check(api.fused_mha_run(stream(), 1, C.byref(p)))
        sync()
    got = host(out)
    assert (got[T:] == -7).all()
    for b in range(min(B, 2 * len(edges))):
        lo, hi = int(cu[b]), int(cu[b + 1])
        if lo == hi:
            continue
        n = b % N
        want = attention_f64(qkv[lo:hi, n, 0], qkv[lo:hi, n, 1], qkv[lo:hi, n, 2], 0.125)
        assert_fp_close(got[lo:hi, n * 64:(n + 1) * 64], want, what=f"sequence {b} of {hi - lo}, head {n}")


# one workgroup of 128 queries short of the lines between the two FP16 kernels, by blocks of keys, and on them; past one round
# of four per CU with two blocks
@pytest.mark.parametrize("B,N,S,kernel", [
    (1024, 1, 64, TURNS), (767, 1, 128, TURNS), (768, 1, 128, STREAM), (1024, 1, 100, STREAM), (205, 5, 100, TURNS),
    (383, 1, 192, TURNS), (384, 1, 192, STREAM), (271, 1, 200, TURNS), (272, 1, 200, STREAM), (179, 1, 260, TURNS),
    (180, 1, 260, STREAM), (167, 1, 384, TURNS), (168, 1, 321, STREAM), (95, 1, 400, TURNS), (96, 1, 448, STREAM),
    (89, 1, 512, TURNS), (90, 1, 449, STREAM)])
def test_fp16_attention_on_either_side_of_its_kernels_lines(B, N, S, kernel):
    api = capi.api()
    r = rng(1900 + B + S)
    edges = [n for n in (S, 1, 16, 63, 64, 65, 127, 128, 129, S - 1, 193, 257, 385) if n <= S]
    lens = np.array([edges[i % len(edges)] for i in range(B)])
    lens[7] = 0
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv = r.standard_normal((T, N, 3, 64)).astype(np.float16)
    d_qkv, d_cu = dev(qkv), dev(cu)
    out = dev_empty((T + 64, N * 64), np.float16, fill=-7)
    p = capi.FmhaParams()
    p.qkv_ptr, p.o_ptr, p.cu_seqlens = ptr(d_qkv), ptr(out), ptr(d_cu)
    p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * N * 64, 2 * N * 64
    p.b, p.h, p.s, p.d = B, N, S, 64
    p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(0.125), half2_bits(1.0), half2_bits(1.0)
    assert route(1, p).kernel == kernel
    api.check(api.fused_mha_run(stream(), 1, C.byref(p)))
    sync()
    got = host(out)
    assert (got[T:] == -7).all()
    for b in [*range(2 * len(edges)), *range(B - len(edges), B)]:
        lo, hi = int(cu[b]), int(cu[b + 1])
        if lo == hi:
            continue
        n = b % N
        want = attention_f64(qkv[lo:hi, n, 0], qkv[lo:hi, n, 1], qkv[lo:hi, n, 2], 0.125)
        assert_fp_close(got[lo:hi, n * 64:(n + 1) * 64], want, what=f"sequence {b} of {hi - lo}, head {n}")


# one unit short of the lines between the numbers of INT8 workgroups per unit, by blocks of keys, and on them
@pytest.mark.parametrize("layout,units,S,parts", [
    ("packed", 639, 128, 2), ("packed", 640, 128, 1), ("packed", 383, 192, 3), ("packed", 384, 192, 2), ("packed", 767, 130, 2),
    ("packed", 768, 192, 1), ("packed", 255, 256, 4), ("packed", 256, 256, 3), ("packed", 767, 256, 2), ("packed", 768, 200, 1),
    ("packed", 192, 260, 4), ("packed", 193, 320, 3), ("packed", 639, 320, 2), ("packed", 640, 260, 1), ("packed", 170, 384, 4),
    ("packed", 171, 330, 3), ("packed", 287, 330, 3), ("packed", 288, 384, 2), ("packed", 895, 384, 2), ("packed", 896, 330, 1),
    ("packed", 319, 400, 3), ("packed", 320, 512, 2), ("packed", 719, 448, 2), ("packed", 720, 400, 1), ("packed", 719, 512, 2),
    ("packed", 720, 460, 1),
    ("full", 193, 256, 3), ("full", 192, 384, 4), ("full", 193, 384, 3), ("full", 341, 384, 3), ("full", 342, 384, 2),
    ("full", 641, 192, 1), ("full", 800, 128, 2),
    ("padded", 640, 96, 2), ("padded", 641, 96, 1), ("padded", 641, 128, 2), ("padded", 255, 256, 4), ("padded", 256, 256, 3),
    ("padded", 192, 320, 4), ("padded", 193, 320, 3), ("padded", 341, 384, 3), ("padded", 342, 384, 2), ("padded", 256, 512, 3),
    ("masked", 640, 128, 2), ("masked", 641, 128, 1), ("masked", 192, 384, 4), ("masked", 193, 384, 3)])
def test_int8_attention_on_either_side_of_its_lines(layout, units, S, parts):
    """The bytes of one workgroup per unit, and of every unit."""
    r = rng(2000 + units + S)
    full = layout != "packed"
    lens = np.full(units, S) if full else np.concatenate([[S, S - 1, 0, 1, 64, 65], r.integers(1, 40, units - 6)])
    T = int(lens.sum())
    bits = lambda x: int(np.float32(x).view(np.uint32))
    p = capi.FmhaParams()
    p.b, p.h, p.s, p.d = units, 1, S, 64
    p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = bits(0.0009 * 0.125), bits(127.0), bits(0.75 / 127)
    q = np.clip(np.rint(33 * r.standard_normal((T, 192), np.float32)), -127, 127).astype(np.int8)
    if layout in ("packed", "full"):
        d_qkv, d_cu = dev(interleave(q)), dev(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
        p.cu_seqlens, p.interleaved = ptr(d_cu), 1
        p.qkv_stride_in_bytes = p.o_stride_in_bytes = T
        shape = (2, T, 32)
    else:
        d_qkv = dev(q.reshape(S, units, 192))
        p.qkv_stride_in_bytes, p.o_stride_in_bytes = 192 * units, 64 * units
        shape = (S, units, 64)
        if layout == "masked":
            mask = (np.arange(S)[:, None] < r.integers(1, S + 1, units)[None, :]).astype(np.int32)
            packed, _ = oracle.convert_mask(mask, *((1, 8) if S == 384 else (2, 2)))
            d_mask = dev(packed)
            p.packed_mask_ptr, p.packed_mask_stride_in_bytes = ptr(d_mask), packed.shape[1] * 4
    p.qkv_ptr = ptr(d_qkv)
    assert route(2, p).parts == parts
    api = capi.api()
    outs = []
    for forced in (-1, 1):
        out = dev_empty(shape, np.int8, fill=-128)
        p.o_ptr = ptr(out)
        with tuning("TRTAMD_FMHA_QSPLIT", forced):
            assert route(2, p).parts == (parts if forced < 0 else 1)
            api.check(api.fused_mha_run(stream(), 2, C.byref(p)))
            sync()
        outs.append(host(out))
    assert np.array_equal(outs[0], outs[1])
    assert (outs[0] != -128).all() # a result is a mean of values of at most 127, times 0.75


@pytest.mark.parametrize("scale", [0.125, 1.0])
def test_fp16_attention_of_full_launches_keeps_infinite_scores_apart(scale):
    """Keys with a score of -infinity weigh nothing, also where they are a whole block or the first one; an infinite V
    behind the last key of a sequence does not reach it.  Scales on either side of ln 2, from where on the scale times
    the largest binary32 value is infinite."""
    api = capi.api()
    r = rng(1700)
    B, N, S = 200, 4, 128
    lens = np.full(B, 100)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    T = int(cu[-1])
    qkv = r.standard_normal((T, N, 3, 64)).astype(np.float16)
    qkv[:, :, 0, 0] = np.abs(qkv[:, :, 0, 0]) + np.float16(0.5)
    qkv[cu[1]:cu[1] + 64, :, 1, 0] = -np.inf        # sequence 1: the first block
    qkv[cu[2] + 64:cu[2] + 100, :, 1, 0] = -np.inf  # sequence 2: the last one
    qkv[cu[4]:cu[5], :, 2, 5] = np.inf              # sequence 4: V, next to sequences 3 and 5
    d_qkv, d_cu = dev(qkv), dev(cu)
    out = dev_empty((T, N * 64), np.float16, fill=0)
    p = capi.FmhaParams()
    p.qkv_ptr, p.o_ptr, p.cu_seqlens = ptr(d_qkv), ptr(out), ptr(d_cu)
    p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * N * 64, 2 * N * 64
    p.b, p.h, p.s, p.d = B, N, S, 64
    p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(scale), half2_bits(1.0), half2_bits(1.0)
    api.check(api.fused_mha_run(stream(), 1, C.byref(p)))
    sync()
    got = host(out)
    for b, keys in ((0, slice(0, 100)), (1, slice(64, 100)), (2, slice(0, 64)), (3, slice(0, 100)), (5, slice(0, 100))):
        lo = int(cu[b])
        k, v = qkv[lo:lo + 100][keys], qkv[lo:lo + 100][keys]
        want = attention_f64(qkv[lo:lo + 100, 1, 0], k[:, 1, 1], v[:, 1, 2], scale)
        assert_fp_close(got[lo:lo + 100, 64:128], want, what=f"sequence {b}")
    # sequence 4 itself: infinite, or NaN where the weight of one of its keys is below the smallest binary16 value (scores of
    # standard deviation 8 at scale 1)
    own = got[cu[4]:cu[5], 64 + 5]
    assert np.isinf(own).all() if scale == 0.125 else not np.isfinite(own).any()


# packed masks: FP16 launches of few workgroups, of more of them with 64 queries, and with 128; and INT8
@pytest.mark.parametrize("dtype,scale", [(1, 0.125), (1, 1.0), (2, 0.125)])
@pytest.mark.parametrize("S,B,N,kernel", [(64, 9, 2, WHOLE), (96, 9, 2, WHOLE), (128, 9, 2, WHOLE), (384, 9, 2, WHOLE),
                                          (64, 150, 2, TURNS), (96, 72, 2, TURNS), (128, 99, 2, TURNS), (384, 30, 2, TURNS),
                                          (128, 200, 4, STREAM), (384, 70, 4, STREAM)])
def test_attention_with_packed_masks(dtype, scale, S, B, N, kernel):
    """Masks that are a prefix of every kind of length, that have holes in the first, a middle and the last block, that
    leave one key or none: the general kernel's results to the bar, zeros where no key is left.  FP16 scales on either side of
    ln 2, from where on the scale times the largest binary32 value is infinite."""
    api = capi.api()
    r = rng(1800 + S + B)
    mask = np.zeros((S, B), np.int32)
    for b in range(B):
        n = [S, 1, 0, S - 1, min(64, S), min(65, S - 1), S // 2 + 3, S, S][b % 9]
        mask[:n, b] = 1
        if b % 9 >= 7:
            mask[:, b] = r.integers(0, 2, S)
    mask[:, 8] = 0
    mask[S - 1, 8] = 1
    packed, _ = oracle.convert_mask(mask, *((1, 8) if S == 384 else (2, 2)))
    x = r.standard_normal((S, B, N, 3, 64))
    if dtype == 2:
        qkv, s_q = quantize_amax(x.astype(np.float32))
        bits = lambda v: int(np.float32(v).view(np.uint32))
        scales = bits(s_q * s_q * scale), bits(127.0), bits(s_q / 127.0 / 0.02)
    else:
        qkv, scales = x.astype(np.float16), (half2_bits(scale), half2_bits(1.0), half2_bits(1.0))
    size = qkv.itemsize
    d_qkv, d_mask = dev(qkv), dev(packed)

    def run():
        out = dev_empty((S, B, N * 64), qkv.dtype.type, fill=55)
        p = capi.FmhaParams()
        p.qkv_ptr, p.o_ptr, p.packed_mask_ptr = ptr(d_qkv), ptr(out), ptr(d_mask)
        p.qkv_stride_in_bytes, p.o_stride_in_bytes = size * 3 * B * N * 64, size * B * N * 64
        p.packed_mask_stride_in_bytes = packed.shape[1] * 4
        p.b, p.h, p.s, p.d = B, N, S, 64
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = scales
        assert dtype == 2 or route(1, p).kernel in (kernel, 0) # 0: the general kernel, asked for
        api.check(api.fused_mha_run(stream(), dtype, C.byref(p)))
        sync()
        return host(out)

    got = run()
    with tuning("TRTAMD_FMHA_GENERIC", 1):
        want = run()
    assert (got[:, 2] == 0).all()
    if dtype == 2:
        # the two kernels add a row's weights up in different orders: a unit in the last place of the sum turns one of
        # 384 quantised weights in 10^5 over, and the output by one where it was next to a tie
        assert_int8_close(got, want, what="general kernel", max_frac_off=1e-3)
    else:
        # at scale 1 a row has two or three keys that count, and the truncation of their weights (2^-10) no longer averages out:
        # a quarter of it times the distance of two values of V, 2^-9 where they are eight apart
        assert_fp_close(got, want, **(dict(atol=1e-3, rtol=2e-3) if scale == 0.125 else {}), what="general kernel")
        for b in (0, 1, 3, 5, 7, 8, B - 1):
            keep = mask[:, b] == 1
            if keep.any():
                ref = attention_f64(qkv[:, b, 1, 0], qkv[keep, b, 1, 1], qkv[keep, b, 1, 2], scale)
                assert_fp_close(got[:, b, 64:128], ref, what=f"sequence {b}")


@pytest.mark.parametrize("S,copies", [(64, 15), (96, 8), (128, 8), (384, 3)])
def test_masked_fp16_launches_of_few_workgroups_give_the_bytes_of_larger_ones(S, copies):
    """With all of K and V in LDS at once and in turns: masks that are a prefix, that have holes in the first, a middle and the
    last block, that leave one key or none."""
    api = capi.api()
    B, N = 9, 2
    r = rng(2100 + S)
    mask = np.ones((S, B), np.int32)
    for b in range(1, B):
        mask[:, b] = r.integers(0, 2, S) if b >= 5 else np.arange(S) < [S, 1, S - 1, min(65, S - 1), S // 2 + 3][b]
    mask[:min(64, S), 6] = 0
    mask[:, 7] = 0
    mask[S - 1, 8] = 1
    qkv = r.standard_normal((S, B, N, 3, 64)).astype(np.float16)
    got = []
    for n, kernel in ((1, WHOLE), (copies, TURNS)):
        packed, _ = oracle.convert_mask(np.tile(mask, (1, n)), *((1, 8) if S == 384 else (2, 2)))
        d_qkv, d_mask, out = dev(np.tile(qkv, (1, n, 1, 1, 1))), dev(packed), dev_empty((S, B * n, N * 64), np.float16, fill=55)
        p = capi.FmhaParams()
        p.qkv_ptr, p.o_ptr, p.packed_mask_ptr = ptr(d_qkv), ptr(out), ptr(d_mask)
        p.qkv_stride_in_bytes, p.o_stride_in_bytes = 2 * 3 * B * n * N * 64, 2 * B * n * N * 64
        p.packed_mask_stride_in_bytes = packed.shape[1] * 4
        p.b, p.h, p.s, p.d = B * n, N, S, 64
        p.scale_bmm1, p.scale_softmax, p.scale_bmm2 = half2_bits(0.125), half2_bits(1.0), half2_bits(1.0)
        assert route(1, p).kernel == kernel
        api.check(api.fused_mha_run(stream(), 1, C.byref(p)))
        sync()
        got.append(host(out))
    assert (got[0][:, 7] == 0).all()
    assert np.array_equal(np.tile(got[0], (1, copies, 1)), got[1])
