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
