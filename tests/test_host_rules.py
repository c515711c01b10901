"""Host-side rules that need no GPU: how the exact recompute is split, which calls go straight to the kernels, and which
inputs the host module refuses before any launch."""
import pytest


@pytest.mark.parametrize("B, H, m, b, rt, splits", [
    (1, 12, 21, 1560, 1560, 2), (2, 12, 21, 1560, 1560, 2),   # fewer tiles than workgroup slots: two key ranges
    (2, 24, 21, 1560, 1560, 1), (1, 12, 21, 1560, 7800, 1), (1, 12, 21, 1560, 32760, 1), (4, 12, 21, 1560, 32760, 1)])
def test_paired_recompute_is_not_split_once_its_tiles_fill_the_chip(B, H, m, b, rt, splits):
    from vmonarch_amd.vmonarch import _OVERLAPS, _recompute_plan
    assert _recompute_plan(B, H, m * b, 128, 128, 2, rt) == (_OVERLAPS["with_r0"], splits)
