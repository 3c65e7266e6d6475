"""Which kernel a linear layer's sizes lead to, asked of the launcher itself (include/trtamd_test_hooks.h); no launch is made."""
import pytest

from tensorrt_amd import capi

INTERLEAVED, LINEAR = 1, 0
# the plans (TRTAMD_LINEAR_PLAN) that have a kernel: interleaved operands, linear ones whose rows are whole lines of 128
# bytes, linear ones whose rows end within a line
KERNELS = {(INTERLEAVED, 1024): {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12}, (LINEAR, 1536): {2, 4, 5, 8, 9, 10, 11, 12, 13, 14},
           (LINEAR, 1472): {1, 2, 3, 4, 8, 9}}


def plan(layout, T, row_bytes, N, gelu=0):
    return capi.api().test_linear_plan(layout, T, row_bytes, N, gelu)


@pytest.fixture
def forced():
    api = capi.api()
    yield lambda n: api.check(api.test_set_tuning(b"TRTAMD_LINEAR_PLAN", n))
    api.check(api.test_reset_tuning(b"TRTAMD_LINEAR_PLAN"))


def test_sizes_that_no_layer_has():
    for sizes in ((0, 64, 32), (1, 0, 32), (1, 96, 32), (1, 64, 0), (1, 64, 48), (-1, 64, 32)):
        assert plan(LINEAR, *sizes) == -1


@pytest.mark.parametrize("layout,row_bytes", KERNELS)
def test_a_plan_is_taken_where_it_has_a_kernel_and_passed_over_where_not(forced, layout, row_bytes):
    chosen = plan(layout, 130, row_bytes, 96)
    for n in range(0, 16):
        forced(n)
        assert plan(layout, 130, row_bytes, 96) == (n if n in KERNELS[layout, row_bytes] else chosen), n


@pytest.mark.parametrize("T,row_bytes,N", [(16384, 2112, 3168), (33289, 1472, 2208), (7765, 6208, 768), (2048, 4160, 1024)])
@pytest.mark.parametrize("gelu", [0, 1])
def test_many_tokens_with_rows_that_end_within_a_line(T, row_bytes, N, gelu):
    """The layers whose launches tiles of 128 x 256 shorten most against the 128 x 128 and 64 x 64 ones take them, or at 2048
    tokens something else than those two."""
    assert plan(LINEAR, T, row_bytes, N, gelu) in ({1} if T > 2048 else {1, 3})


@pytest.mark.parametrize("T,row_bytes,N,gelu", [(1200, 256, 512, 0), (2600, 256, 384, 0), (4000, 128, 256, 0), (1700, 384, 576, 0),
                                                (2100, 512, 256, 0), (800, 640, 960, 0), (600, 768, 1152, 0), (1400, 768, 384, 0),
                                                (384, 768, 1536, 1), (512, 1024, 1536, 0), (1200, 1024, 512, 0),
                                                (384, 1024, 2048, 1), (256, 1280, 2560, 0), (700, 1536, 768, 0)])
def test_short_rows_go_in_tiles(T, row_bytes, N, gelu):
    """Layers with short rows of whole lines, where 64 x 64 tiles take 5 to 30 % less than the pieces."""
    assert plan(LINEAR, T, row_bytes, N, gelu) in (4, 14)


@pytest.mark.parametrize("T", [97, 102, 128])
def test_the_smaller_pieces_where_both_are_even(T):
    """The first layers of a 768-channel FP16 encoder."""
    assert plan(LINEAR, T, 1536, 2304) == plan(LINEAR, T, 1536, 3072, 1) == 9


@pytest.mark.parametrize("T,row_bytes,N,want", [(1, 128, 256, 9), (65, 256, 512, 9), (102, 1536, 2304, 9),
                                                (448, 6144, 768, 8), (96, 8192, 1024, 9), (2100, 256, 32, 9)])
def test_few_tokens_go_in_pieces(T, row_bytes, N, want):
    assert plan(LINEAR, T, row_bytes, N) == want


def layers(layout, size, hidden, ffn):
    """The four linear layers of an encoder layer: row bytes, channels, GELU."""
    return [(layout, size * hidden, 3 * hidden, 0), (layout, size * hidden, hidden, 0), (layout, size * hidden, ffn, 1),
            (layout, size * ffn, hidden, 0)]


@pytest.mark.parametrize("T", [[1], [48], [255], [256], [600], [4096], [9084, 8231], [16384, 16640], [24000, 23999]])
@pytest.mark.parametrize("model", [(INTERLEAVED, 1, 1024, 4096), (LINEAR, 2, 768, 3072), (LINEAR, 2, 1024, 4096),
                                   (INTERLEAVED, 1, 768, 3072), (INTERLEAVED, 1, 512, 2048)])
def test_the_layers_of_a_pass_are_estimated_once(model, T):
    """One encoder layer after the other asks for the same few plans, as two halves of a batch do in turn: nothing is worked
    out again."""
    asked = [(layout, t, row_bytes, n, gelu) for t in T for layout, row_bytes, n, gelu in layers(*model)]
    first = [plan(*a) for a in asked]
    before = capi.api().test_linear_estimates()
    for _ in range(24):
        assert [plan(*a) for a in asked] == first
    assert capi.api().test_linear_estimates() == before


def test_plans_are_remembered_for_the_switches_that_they_were_made_under(forced):
    want = plan(LINEAR, 7000, 1536, 768)
    for n in (10, 14, 2):
        forced(n)
        assert plan(LINEAR, 7000, 1536, 768) == n
    forced(-1)
    assert plan(LINEAR, 7000, 1536, 768) == want
