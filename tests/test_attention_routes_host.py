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
