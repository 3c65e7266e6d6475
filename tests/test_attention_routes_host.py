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


def route(dtype, units, s, **layout):
    """backwards: the number of workgroups whose every other round of 256 goes backwards."""
    r = capi.api().test_fmha_route(dtype, C.byref(params(dtype, units, s, **layout)))
    assert r >= 0
    return Route(r & 15, r >> 4 & 15, bool(r >> 8 & 1), (r >> 17) * 512)


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
