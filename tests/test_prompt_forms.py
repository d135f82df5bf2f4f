"""Which form makes a fused prompt product and what workspace it asks for, on both sides of each line of the rule (on the
host: the plan needs no GPU)."""

import pytest

TILES, REGISTERS, BF16, RING = 0, 1, 2, 3
SMALL, LARGE, HUGE = (4096, 4096), (4104, 4096), (16392, 8192)  # N, K: N K = 2^24, just past it, just past 2^27


def plan(M, N, K, swiglu=0, fmt=1):
    from lit_gpt import ops

    return ops.q4f_plan(M, N, K, swiglu, fmt)


@pytest.mark.parametrize("fmt", [0, 1, 3])
@pytest.mark.parametrize("M,size,swiglu,form", [
    (2, SMALL, 0, RING), (32, SMALL, 0, RING), (32, LARGE, 0, REGISTERS), (32, SMALL, 1, RING), (32, LARGE, 1, REGISTERS),
    (32, (8192, 8192), 1, REGISTERS), (32, (8200, 8192), 1, RING), (32, (11008, 4096), 1, RING), (33, LARGE, 1, RING), (65, SMALL, 0, RING),
    (96, LARGE, 0, REGISTERS), (96, (8192, 8064), 0, REGISTERS), (96, (8200, 4096), 0, RING), (97, LARGE, 0, RING),
    (33, (8192, 2048), 0, REGISTERS), (96, (8192, 1536), 0, REGISTERS), (97, (8192, 2048), 0, RING), (64, (8192, 2560), 1, REGISTERS),
    (65, (8192, 2560), 1, RING), (48, (8192, 2688), 1, RING), (64, (8184, 2048), 1, RING),
    (64, (8192, 8192), 0, RING), (96, SMALL, 0, RING), (96, SMALL, 1, RING), (97, SMALL, 0, RING), (97, LARGE, 1, RING),
    (97, HUGE, 1, RING), (128, LARGE, 0, RING), (128, HUGE, 1, RING), (129, HUGE, 1, RING), (129, HUGE, 0, RING),
    (256, (16384, 4096), 0, RING), (256, (28672, 4096), 0, RING), (129, SMALL, 0, RING), (257, SMALL, 0, RING),
    (257, (264, 256), 0, RING), (64, (4096, 4160), 0, TILES), (64, (4096, 192), 0, TILES), (300, (4096, 4160), 1, TILES)])
def test_four_bit_weights(fmt, M, size, swiglu, form):
    assert plan(M, *size, swiglu, fmt)[0] == form


@pytest.mark.parametrize("M,size,int4,nf4", [(33, SMALL, RING, REGISTERS), (64, SMALL, RING, REGISTERS), (64, LARGE, REGISTERS, REGISTERS),
                                             (64, (8200, 4096), RING, REGISTERS), (64, (4096, 128), RING, REGISTERS)])
def test_formats_apart(M, size, int4, nf4):
    """33 to 64 rows of one matrix below 2^26 values: codebooks stay in gemm_q4d.hip's form, int4 only between 2^24 and 2^26."""
    assert plan(M, *size, 0, 0)[0] == int4 and plan(M, *size, 0, 1)[0] == nf4 and plan(M, *size, 0, 3)[0] == nf4


@pytest.mark.parametrize("M,size,swiglu,form", [
    (32, (8184, 8192), 0, TILES), (32, (8192, 8192), 0, BF16), (32, (4096, 8192), 1, BF16), (33, SMALL, 0, BF16),
    (1024, (28672, 8192), 1, BF16), (1025, (28672, 8192), 1, BF16), (1025, (512, 4096), 0, BF16), (517, (4096, 4160), 0, BF16)])
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
    # the formats' ranges of K differ: neither product asks for the other's partial sums
    most = ops.load_library().lga_q4f_workspace_bytes(600, 4096, 11008, 0)
    assert plan(600, 4096, 11008, 0, 1)[1:] == (4096 + 3 * 600 * 4096 * 4, False) and plan(600, 4096, 11008, 0, 2)[1:] == (most, False)


def test_refused_sizes_have_no_workspace():
    assert plan(0, 64, 64) == (TILES, 0, False) and plan(4, 64, 32) == (TILES, 0, False) and plan(4, 64, 64, 0, 7) == (TILES, 0, False)


@pytest.mark.parametrize("M,N,K,ranges", [(1000, 4096, 11008, 4), (517, 8192, 28672, 2), (1400, 4096, 4096, 0), (2048, 28672, 8192, 0)])
def test_ranges_of_long_rows(M, N, K, ranges):
    """4-bit prompts ask for the sums of the ranges that they are made in, where rows are long and tiles few, and for no counters: their
    two launches share no buffer with another product's."""
    assert plan(M, N, K) == (RING, 4096 + ranges * M * N * 4 if ranges else 0, False)


@pytest.mark.parametrize("fmt", [0, 1, 3])
def test_two_launches_keep_no_buffer(fmt):
    """Only the one launch of the LDS image's tiles may use a buffer that other products of its stream use: whatever else sums over
    ranges of K takes its workspace from the allocator, bounded at 128 MB."""
    for M in (2, 31, 33, 64, 93, 128, 129, 257, 600, 1000, 2048):
        for N, K in ((4096, 11008), SMALL, (8192, 28672), (12288, 4096), (512, 1024)):
            for swiglu in (0, 1):
                form, need, counters = plan(M, N, K, swiglu, fmt)
                assert form != TILES and not counters and need <= 4096 + (128 << 20)
