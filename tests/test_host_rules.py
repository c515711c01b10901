"""Host-side rules that need no GPU: how the exact recompute is split, which calls go straight to the kernels, and which
inputs the host module refuses before any launch."""
import pytest


@pytest.mark.parametrize("B, H, m, b, rt, splits", [
    (1, 12, 21, 1560, 1560, 2), (2, 12, 21, 1560, 1560, 2),   # fewer tiles than workgroup slots: two key ranges
    (2, 24, 21, 1560, 1560, 1), (1, 12, 21, 1560, 7800, 1), (1, 12, 21, 1560, 32760, 1), (4, 12, 21, 1560, 32760, 1)])
def test_paired_recompute_is_not_split_once_its_tiles_fill_the_chip(B, H, m, b, rt, splits):
    from vmonarch_amd.vmonarch import _OVERLAPS, _recompute_plan
    assert _recompute_plan(B, H, m * b, 128, 128, 2, rt) == (_OVERLAPS["with_r0"], splits)


def test_calls_that_something_records_take_the_autograd_function():
    import torch
    from vmonarch_amd.kernel import _recorded
    x, leaf, seen = torch.randn(1, 2, 8, 16), torch.randn(1, 2, 8, 16, requires_grad=True), []

    def note(t):
        seen.append(_recorded(x, t, x))
        return t * 2

    assert not _recorded(x, x, x) and _recorded(x, x, leaf)
    with torch.no_grad():
        assert not _recorded(x, x, leaf)
        torch.func.vmap(note)(x)
        with torch.autograd.forward_ad.dual_level():
            note(x)
        torch.jit.trace(note, (x,), check_trace=False)
    assert seen == [True, True, True]


@pytest.mark.parametrize("which", ["k", "v"])
@pytest.mark.parametrize("other", ["float32", "float16", "uint8"])
def test_inputs_of_another_dtype_are_refused(which, other):
    """The kernels read every input in q's type: a wider one would be read as other numbers, a narrower one past its end.
    Refused on the host before any launch, by the public entry and by the host module under it."""
    import torch
    from vmonarch_amd import _lib, flash_entropy_attention
    x = {n: torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16) for n in "qkv"}
    x[which] = x[which].to(getattr(torch, other))
    with pytest.raises(AssertionError, match="one dtype"):
        flash_entropy_attention(**x)
    host, (q, k, v) = _lib.host(), x.values()
    for call in (lambda: host.fea_attention(q, k, v, 1.0),
                 lambda: host.vmonarch_fwd(q, k, v, 2, 4, 2, 0, 0.01, 1.0, False, 1, 0, 0, None, None, None),
                 lambda: host.vmonarch_fwd_train(q, k, v, 2, 4, 2, 0, 0.01, 1.0, 1, 0, 0)):
        with pytest.raises(AssertionError, match="dtype"):
            call()


def test_inputs_elsewhere_are_refused():
    import torch
    from vmonarch_amd import _lib
    q, far = torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16), torch.zeros(1, 2, 8, 16, dtype=torch.bfloat16, device="meta")
    host = _lib.host()
    for k, v in ((far, q), (q, far)):
        with pytest.raises(AssertionError, match="device"):
            host.fea_attention(q, k, v, 1.0)
    with pytest.raises(ValueError, match="GPU"):
        host.fea_attention(q, q, q, 1.0)


def test_large_64_wide_grids_fork_the_recompute():
    """The shared launch takes 64-wide R-step 0 its third workgroup per CU; 128-wide heads have two either way."""
    from vmonarch_amd.vmonarch import _OVERLAPS, _recompute_plan
    plan = lambda H, m, b, D: _recompute_plan(1, H, m * b, D, D, 2, b)   # noqa: E731
    assert plan(12, 21, 1560, 64) == (_OVERLAPS["start"], 3) and plan(12, 4, 1560, 64) == (_OVERLAPS["start"], 3)
    assert plan(12, 4, 600, 64)[0] == plan(8, 4, 1024, 64)[0] == _OVERLAPS["with_r0"]
    assert plan(12, 21, 1560, 128)[0] == plan(12, 4, 1560, 128)[0] == _OVERLAPS["with_r0"]
