"""Which systolic kernel a call runs (mxq_systolic_plan_of): the rule is host code, so these need no GPU."""
import pytest

from _util import systolic_plan

MXG = ("MXGEMMINI",)
LADDERS = {"hw_final": (MXG, None, 16), "e4m4": (MXG, [(4, 4)] * 16, 16), "e5m6": (MXG, [(5, 6)] * 16, 16),
           "mxquant": (("MXQUANT", 4, 3), None, 16), "mxquant_e5m10": (("MXQUANT", 5, 10), [(6, 9)] * 16, 16)}


def _plan(name, K, M, N, **kw):
    from mxq import matmul, schedule
    ar, ladder, size = LADDERS[name]
    return systolic_plan(K, M, N, getattr(matmul, ar[0])(*ar[1:]), ladder or schedule.HW_FINAL, size, **kw)


@pytest.mark.parametrize("block", [32, 64])
@pytest.mark.parametrize("name", LADDERS)
@pytest.mark.parametrize("M", [1, 4, 8, 16, 64])
def test_small_kernel_refuses_strides_its_offsets_cannot_hold(name, M, block):
    """k_systolic_small's threads reach 64 * waves / rows rows of A from one address by a 32-bit element offset; a
    row stride past that limit goes to a kernel of 64-bit offsets, whatever the shape."""
    for log in range(12, 34):
        for ld in (1 << log, (1 << log) - 1, (1 << log) + 5, 4_198_405):
            kernel, rows, cols, waves = _plan(name, 4096, M, 256, ld_a=max(ld, M), block_size=block)
            if kernel == "small":
                assert (64 * waves // rows) * max(ld, M) <= 1 << 32, f"{rows} rows, stride {ld}"
            if kernel == "tile":
                assert ld < 1 << 28 and block == 32
    assert _plan(name, 4096, M, 256, block_size=block)[0] == "small"     # (the shapes are the small kernel's)


@pytest.mark.parametrize("name", LADDERS)
@pytest.mark.parametrize("block", [32, 64])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 256, 1024, 4096])
def test_a_short_product_is_not_computed_for_padding(name, K, block):
    """A small kernel's workgroup computes a whole round of reductions, one for every wave and group of columns, however
    few K holds.  Where the outputs make more than a round of workgroups for the chip (256 CUs), the padded rows of K times
    the rounds of workgroups stay under twice what the tiles would compute (of 64 x 64, rounded up the same way)."""
    for M in (8, 16, 33, 64, 128, 200, 333, 512, 1024, 2048):
        for N in (64, 512, 1000, 2048, 4096):
            kernel, rows, cols, waves = _plan(name, K, M, N, block_size=block)
            wgs = -(-M // rows) * -(-N // cols)
            if kernel != "small" or wgs <= 256:
                continue
            at_once = waves * (64 // cols) * 16
            work = -(-K // at_once) * at_once * wgs * rows * cols
            assert work <= 2 * max(-(-K // 32) * 32, 128) * -(-M // 64) * -(-N // 64) * 4096, \
                f"{M} x {N}, K = {K}: {wgs} workgroups of {rows} x {cols}, {waves} waves"


# HW_FINAL on MI355X: K, M, N -> the tiles (rows, columns) within a tenth of the fastest's time
MEASURED = {(64, 4, 4096): [(8, 64), (8, 32)], (64, 333, 2048): [(32, 32)], (64, 512, 2048): [(64, 64), (32, 32)],
            (512, 16, 1024): [(4, 32)], (512, 256, 512): [(8, 64), (8, 32)], (2048, 4, 512): [(4, 16)],
            (2048, 4, 4096): [(4, 16), (4, 32)], (2048, 8, 4096): [(4, 32)], (2048, 16, 256): [(4, 16)],
            (2048, 16, 1024): [(4, 16)], (2048, 16, 4096): [(8, 32), (4, 64)], (2048, 24, 2048): [(8, 32)],
            (2048, 32, 4096): [(8, 64), (4, 64)], (2048, 128, 512): [(8, 32)], (2048, 64, 4096): [(8, 64), (8, 32)],
            (2048, 128, 4096): [(16, 64), (32, 32)], (2048, 200, 2048): [(16, 64)], (2048, 512, 1000): [(32, 32)],
            (2048, 333, 5632): [(32, 32)], (2048, 1024, 2048): [(64, 64)], (4096, 512, 4096): [(64, 64)]}


@pytest.mark.parametrize("K,M,N", MEASURED, ids=str)
def test_measured_choices(K, M, N):
    assert _plan("hw_final", K, M, N)[1:3] in MEASURED[K, M, N]


def test_measured_choice_mxquant():
    """MXQUANT(4, 3) under HW_FINAL, 512 x 2048 outputs of K = 2048: 32 x 32 tiles 625 us, 16-row tiles of few outputs 640."""
    assert _plan("mxquant", 2048, 512, 2048)[:3] == ("tile", 32, 32)
