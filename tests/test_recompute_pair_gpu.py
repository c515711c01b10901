"""VMonarch's exact recompute in one launch with R-step 0 (vmo_fea_fwd_pair) against the two as launches of their own:
the same tiles, so z, and through the saved statistics the gradients, bit for bit; and the rule that picks the order."""
import pytest
import torch

from conftest import randn_lp

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# recompute tiles: one partial, several, none left over; key splits 1 (no merge) and more, down to a partial last stage
@pytest.mark.parametrize("B, H, m, b, rt, D, splits, dtype", [
    (1, 2, 4, 64, 64, 64, 1, torch.bfloat16), (2, 3, 5, 37, 37, 128, 2, torch.float16), (1, 5, 9, 130, 300, 64, 3, torch.float16),
    (1, 4, 21, 100, 1, 128, 8, torch.bfloat16), (1, 1, 33, 128, 256, 128, 2, torch.bfloat16)])
def test_pair_launch_is_bitwise_the_two_launches(monkeypatch, B, H, m, b, rt, D, splits, dtype):
    import vmonarch_amd.vmonarch as vm
    g = torch.Generator().manual_seed(m + b)
    q, k, v, dz = (randn_lp(g, B, H, m * b, D, scale=0.5, dtype=dtype).to(DEV) for _ in range(4))
    monkeypatch.setattr(vm, "_recompute_splits", lambda *a: splits)
    print(f"pair B={B} H={H} m={m} b={b} rt={rt} D={D} splits={splits} {dtype}", flush=True)
    out = []
    for order in ("off", "with_r0"):
        monkeypatch.setattr(vm, "_RECOMPUTE_OVERLAP", order)
        with torch.no_grad():
            z = vm.vmonarch_attention(q, k, v, m, b, 2, recompute_tokens=rt)
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        zg = vm.vmonarch_attention(*leaves, m, b, 2, recompute_tokens=rt)
        out.append([z, zg.detach(), *torch.autograd.grad(zg, leaves, dz)])
    for a, c in zip(*out):
        assert torch.equal(a, c)


def test_recompute_plan():
    from vmonarch_amd.vmonarch import _OVERLAPS, _recompute_plan
    assert _recompute_plan(1, 2, 256, 64, 64, 2, 0) == (0, 1)
    assert _recompute_plan(1, 2, 256, 64, 64, 2, 64) == (_OVERLAPS["with_r0"], 1)
    assert _recompute_plan(1, 12, 32760, 128, 128, 2, 1560) == (_OVERLAPS["with_r0"], 2)
    assert _recompute_plan(1, 2, 256, 64, 64, 1, 64)[0] == _OVERLAPS["off"]         # values [k | v]: no pair
    assert _recompute_plan(1, 12, 32760, 32, 32, 2, 1560)[0] == _OVERLAPS["start"]   # 32-wide heads: no pair
    fp8 = _recompute_plan(1, 12, 32760, 128, 128, 2, 1560, qk_fp8=True)              # R-step 0 with fp8 S: no pair
    assert fp8 == (_OVERLAPS["start"], 3)
