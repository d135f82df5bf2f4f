"""Which form makes a fused prompt product and what workspace it asks for, on both sides of each line of the rule (on the
host: the plan needs no GPU)."""

import pytest

TILES, REGISTERS, BF16 = 0, 1, 2
SMALL, LARGE, HUGE = (4096, 4096), (4104, 4096), (16392, 8192)  # N, K: N K = 2^24, just past it, just past 2^27


def plan(M, N, K, swiglu=0, fmt=1):
    from lit_gpt import ops

    return ops.q4f_plan(M, N, K, swiglu, fmt)


@pytest.mark.parametrize("fmt", [0, 1, 3])
@pytest.mark.parametrize("M,size,swiglu,form", [
    (2, SMALL, 0, TILES), (32, SMALL, 0, TILES), (32, LARGE, 0, REGISTERS), (33, SMALL, 0, REGISTERS),
    (96, SMALL, 0, REGISTERS), (96, SMALL, 1, REGISTERS), (97, SMALL, 0, TILES), (97, LARGE, 0, REGISTERS),
    (97, LARGE, 1, TILES), (97, HUGE, 1, REGISTERS), (128, LARGE, 0, REGISTERS), (128, HUGE, 1, REGISTERS),
    (129, HUGE, 1, TILES), (129, HUGE, 0, TILES), (129, (16384, 8192), 0, REGISTERS), (256, (16384, 4096), 0, REGISTERS),
    (129, (16392, 4096), 0, TILES), (256, (28672, 4096), 0, TILES), (128, (28672, 4096), 0, REGISTERS), (129, LARGE, 0, REGISTERS), (129, SMALL, 0, REGISTERS), (256, SMALL, 0, REGISTERS),
    (257, SMALL, 0, TILES), (64, (4096, 4160), 0, TILES), (64, (4096, 192), 0, TILES), (64, (4096, 128), 0, REGISTERS)])
def test_four_bit_weights(fmt, M, size, swiglu, form):
    assert plan(M, *size, swiglu, fmt)[0] == form


@pytest.mark.parametrize("M,size,swiglu,form", [
    (32, (8184, 8192), 0, TILES), (32, (8192, 8192), 0, BF16), (32, (4096, 8192), 1, BF16), (33, SMALL, 0, BF16),
    (1024, (28672, 8192), 1, BF16), (1025, (28672, 8192), 1, TILES), (1025, (512, 4096), 0, BF16), (517, (4096, 4160), 0, BF16)])
def test_bf16_weights(M, size, swiglu, form):
    assert plan(M, *size, swiglu, 2)[0] == form


def test_workspaces_are_those_of_the_form():
    from lit_gpt import ops

    for M in (16, 64, 93, 128, 200, 300, 600, 1500):
        for N, K in ((4096, 11008), SMALL, (12288, 4096), (512, 4160)):
            for swiglu in (0, 1):
                most = ops.load_library().lga_q4f_workspace_bytes(M, N, K, swiglu)
                for fmt in (0, 1, 2, 3):
                    form, need, counters = plan(M, N, K, swiglu, fmt)
                    assert need <= most and counters == (form == TILES and need > 0)
    # the two formats' ranges of K differ: neither product asks for the other's partial sums
    most = ops.load_library().lga_q4f_workspace_bytes(600, 4096, 11008, 0)
    assert plan(600, 4096, 11008, 0, 1)[1:] == (4096 + 2 * 600 * 4096 * 4, True) and plan(600, 4096, 11008, 0, 2)[1:] == (most, False)


def test_refused_sizes_have_no_workspace():
    assert plan(0, 64, 64) == (TILES, 0, False) and plan(4, 64, 32) == (TILES, 0, False) and plan(4, 64, 64, 0, 7) == (TILES, 0, False)


@pytest.mark.parametrize("M,N,K,halves", [(1000, 4096, 11008, True), (517, 8192, 28672, True), (1400, 4096, 4096, False),
                                          (2048, 28672, 8192, False)])
def test_halves_of_long_rows(M, N, K, halves):
    """4-bit prompts past the tiles' own ranges of K ask for two ranges' sums where rows are long and tiles few."""
    assert plan(M, N, K) == (TILES, 4096 + 2 * M * N * 4 if halves else 0, halves)
