"""Which kernel, split and order a fused attention call leads to, asked of the launcher itself (include/trtamd_test_hooks.h); no
launch is made."""
import ctypes as C
from collections import namedtuple

import pytest

from tensorrt_amd import capi

FP16, INT8 = 1, 2
GENERAL, TURNS, STREAM, WHOLE = range(4)   # INT8 kernels count as GENERAL
Route = namedtuple("Route", "kernel parts ranked backwards")


def params(dtype, units, s, packed=True, masked=False, heads=1):
    """units (sequence, head) pairs; pointers that are only compared with NULL."""
    assert units % heads == 0
    p = capi.FmhaParams()
    p.b, p.h, p.s, p.d = units // heads, heads, s, 64
    size = 1 if dtype == INT8 else 2
    p.qkv_stride_in_bytes, p.o_stride_in_bytes = size * 3 * heads * 64, size * heads * 64
    if packed:
        p.cu_seqlens = 16
    else:
        p.qkv_stride_in_bytes *= p.b
        p.o_stride_in_bytes *= p.b
        p.packed_mask_ptr = 16 if masked else None
    return p


def decode(r):
    """backwards: the number of workgroups whose every other round of 256 goes backwards."""
    assert r >= 0
    return Route(r & 15, r >> 4 & 15, bool(r >> 8 & 1), (r >> 17) * 512)


def route(dtype, units, s, **layout):
    return decode(capi.api().test_fmha_route(dtype, C.byref(params(dtype, units, s, **layout))))


def test_parameters_without_a_kernel():
    api = capi.api()
    for dtype, units, s in ((0, 4, 64), (3, 4, 64), (FP16, 4, 513), (INT8, 4, 0), (INT8, 0, 64)):
        assert api.test_fmha_route(dtype, C.byref(params(dtype, units, s))) == -1
    p = params(FP16, 4, 64)
    p.d = 32
    assert api.test_fmha_route(FP16, C.byref(p)) == -1
    assert api.test_fmha_route(FP16, None) == -1


@pytest.mark.parametrize("dtype", [FP16, INT8])
@pytest.mark.parametrize("s", [1, 64, 96, 128, 192, 256, 257, 384, 400, 512])
@pytest.mark.parametrize("layout", [dict(), dict(packed=False), dict(packed=False, masked=True)])
def test_every_part_has_queries_and_every_round_is_whole(dtype, s, layout):
    """No more parts than tiles of 64 queries (of the capacity that the kernel has), at least one, and only whole pairs of rounds
    change places, of packed sequences only."""
    blocks = next(k for k in (1, 2, 3, 4, 6, 8) if s <= 64 * k)
    for units in [*range(1, 200, 7), *range(200, 1300, 23), 1 << 20]:
        r = route(dtype, units, s, **layout)
        assert 1 <= r.parts <= (blocks if dtype == FP16 else max(1, -(-s // 64)))
        assert r.backwards % 512 == 0 and r.backwards <= units * r.parts
        assert layout.get("packed", True) or r.backwards == 0
        if dtype == FP16:
            assert r.parts == {TURNS: blocks, WHOLE: blocks, STREAM: -(-blocks // 2)}[r.kernel]
            assert (r.kernel == WHOLE) == (r.kernel != STREAM and units * blocks <= 256 and s <= 384)


# either side of each line between the numbers of parts
@pytest.mark.parametrize("s,masked,parts", [
    (64, True, {200: 1, 1000: 1}),
    (96, True, {300: 2, 640: 2, 641: 1, 800: 1, 896: 1}), (96, False, {640: 2, 641: 1, 800: 1}),
    (128, True, {640: 2, 641: 1, 800: 1}), (128, False, {640: 2, 800: 2, 895: 2, 896: 1}),
    (192, False, {255: 3, 383: 3, 384: 2, 640: 2, 641: 1, 768: 1}),
    (256, False, {192: 4, 193: 4, 255: 4, 256: 3, 383: 3, 384: 2, 768: 2, 895: 2, 896: 1}),
    (320, False, {192: 4, 193: 3, 383: 3, 384: 2, 640: 2, 641: 1}),
    (384, True, {170: 4, 171: 4, 192: 4, 193: 3, 256: 3, 341: 3, 342: 2, 895: 2, 896: 1}), (384, False, {192: 4, 256: 3, 896: 1}),
    (448, False, {171: 4, 255: 4, 256: 3, 383: 3, 384: 2, 640: 2, 641: 1}),
    (512, False, {171: 4, 255: 4, 256: 3, 383: 3, 384: 2, 720: 2, 895: 2, 896: 1})])
def test_parts_of_padded_int8_units(s, masked, parts):
    assert {u: route(INT8, u, s, packed=False, masked=masked).parts for u in parts} == parts


@pytest.mark.parametrize("s,parts", [
    (128, {200: 2, 639: 2, 640: 1}), (192, {200: 3, 383: 3, 384: 2, 767: 2, 768: 1}),
    (256, {192: 4, 193: 4, 255: 4, 256: 3, 383: 3, 384: 2, 767: 2, 768: 1}), (320, {192: 4, 193: 3, 383: 3, 384: 2, 639: 2, 640: 1}),
    (384, {170: 4, 171: 3, 256: 3, 287: 3, 288: 2, 895: 2, 896: 1}),
    (448, {170: 4, 171: 3, 256: 3, 319: 3, 320: 2, 719: 2, 720: 1}), (512, {170: 4, 171: 3, 256: 3, 319: 3, 320: 2, 719: 2, 720: 1})])
def test_parts_of_packed_int8_units(s, parts):
    assert {u: route(INT8, u, s).parts for u in parts} == parts


# units, s: longest first, whether every other round goes backwards
@pytest.mark.parametrize("units,s,ranked,backwards", [
    (255, 192, False, False), (256, 192, True, False), (384, 192, True, True),
    (191, 256, False, False), (192, 256, True, True), (193, 256, False, True), (255, 256, False, True), (256, 256, True, False), (384, 256, True, True),
    (128, 384, False, False), (129, 384, True, True), (256, 384, True, False), (288, 384, True, True),
    (1024, 384, True, True), (1025, 384, True, False), (1200, 128, True, True)])
def test_order_of_packed_int8_units(units, s, ranked, backwards):
    r = route(INT8, units, s)
    assert (r.ranked, r.backwards) == (ranked, units * r.parts // 512 * 512 if backwards else 0)


@pytest.mark.parametrize("s", [128, 192, 256, 320, 384, 448, 512])
def test_packed_int8_units_that_fill_their_length_go_as_padded_ones(s):
    """The interleaved layout's strides are the number of tokens: from 15/16 of what the length allows on the split of the padded
    layout (of four blocks of keys one part less from 193 to 255 units), in natural order."""
    for units in (100, 200, 240, 256, 300, 352, 512, 700, 800, 1000, 1200):
        parts = 3 if s == 256 and 193 <= units <= 255 else route(INT8, units, s, packed=False).parts
        packed = route(INT8, units, s)
        most = units * s
        for tokens, full in ((most, True), (-(-most * 15 // 16), True), (-(-most * 15 // 16) - 1, False), (units, False)):
            p = params(INT8, units, s)
            p.interleaved, p.qkv_stride_in_bytes, p.o_stride_in_bytes = 1, tokens, tokens
            r = decode(capi.api().test_fmha_route(INT8, C.byref(p)))
            assert (r.parts == parts and not r.ranked) if full else r == packed, (units, tokens)


# units, s: kernel, longest first, whether every other round goes backwards
@pytest.mark.parametrize("units,s,kernel,ranked,backwards", [
    (383, 192, TURNS, False, False), (384, 192, STREAM, True, True), (767, 192, STREAM, True, True), (1600, 192, STREAM, False, True),   # two parts of three
    (128, 256, TURNS, False, True), (271, 256, TURNS, False, True), (272, 256, STREAM, True, True), (1536, 256, STREAM, False, True),
    (100, 320, TURNS, False, False), (200, 320, STREAM, True, True),
    (85, 384, TURNS, False, False), (86, 384, TURNS, True, True), (127, 384, TURNS, True, True), (128, 384, TURNS, False, False),
    (167, 384, TURNS, False, False), (168, 384, STREAM, True, False), (171, 384, STREAM, True, True), (255, 384, STREAM, True, True),
    (256, 384, STREAM, True, False), (341, 384, STREAM, True, False), (342, 384, STREAM, True, True), (1023, 384, STREAM, True, True),
    (1024, 384, STREAM, False, False),
    (64, 448, TURNS, False, True), (95, 448, TURNS, False, True), (96, 448, STREAM, True, False), (89, 512, TURNS, False, True), (128, 448, STREAM, True, True), (768, 512, STREAM, False, True)])
def test_order_of_packed_fp16_workgroups(units, s, kernel, ranked, backwards):
    r = route(FP16, units, s)
    assert (r.kernel, r.ranked, r.backwards) == (kernel, ranked, units * r.parts // 512 * 512 if backwards else 0)


@pytest.mark.parametrize("s,stream_from", [(64, None), (128, 768), (192, 384), (256, 384), (320, 180), (384, 144), (448, 96), (512, 90)])
@pytest.mark.parametrize("masked", [False, True])
def test_padded_fp16_sequences_change_kernels_where_they_are_faster(s, stream_from, masked):
    line = stream_from or 5000
    for units, kernel in ((line - 1, TURNS), (line, TURNS if stream_from is None else STREAM)):
        r = route(FP16, units, s, packed=False, masked=masked)
        assert (r.kernel, r.backwards) == (kernel, 0), units
