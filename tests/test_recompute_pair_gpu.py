"""VMonarch's exact recompute in one launch with R-step 0 (vmo_fea_fwd_pair) against the two as launches of their own:
where R-step 0 alone takes the 128-query kernel too (frames below 512 tokens, or many tiles), the same tiles, so z, and
through the saved statistics the gradients, bit for bit; and the rule that picks the order."""
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


# few tiles of 512 tokens and more: R-step 0 alone takes the key-group kernel, which adds in another order
@pytest.mark.parametrize("H, m, b, D, dtype, tol", [(2, 4, 1024, 64, torch.bfloat16, 1e-2), (1, 3, 520, 128, torch.float16, 1.2e-3)])
def test_pair_launch_where_the_two_launches_take_key_groups(monkeypatch, H, m, b, D, dtype, tol):
    """Each order's z and gradients are within 4.6e-3 (bf16) / 5.5e-4 (fp16) of float64 (u and the row outputs are stored in
    16 bits between the steps), so within twice that of each other, in the 2-norm; the exact rows, cut into the same key
    ranges either way, are equal bit for bit."""
    import vmonarch_amd.vmonarch as vm
    from test_fea_small_grid_gpu import _query_tile
    g = torch.Generator().manual_seed(m + b)
    q, k, v, dz = (randn_lp(g, 1, H, m * b, D, scale=0.5, dtype=dtype).to(DEV) for _ in range(4))
    assert _query_tile(q, k, k, None, m) in (32, 64)
    monkeypatch.setattr(vm, "_recompute_splits", lambda *a: 2)
    print(f"pair against key groups H={H} m={m} b={b} D={D} {dtype}", flush=True)
    out = []
    for order in ("off", "with_r0"):
        monkeypatch.setattr(vm, "_RECOMPUTE_OVERLAP", order)
        leaves = [t.clone().requires_grad_() for t in (q, k, v)]
        z = vm.vmonarch_attention(*leaves, m, b, 2, recompute_tokens=b)
        out.append([z.detach(), *torch.autograd.grad(z, leaves, dz)])
    assert torch.equal(out[0][0][:, :, :b], out[1][0][:, :, :b])
    for a, c in zip(*out):
        assert (a.double() - c.double()).norm() <= tol * c.double().norm()


def test_recompute_plan():
    from vmonarch_amd.vmonarch import _OVERLAPS, _recompute_plan
    assert _recompute_plan(1, 2, 256, 64, 64, 2, 0) == (0, 1)
    assert _recompute_plan(1, 2, 256, 64, 64, 2, 64) == (_OVERLAPS["with_r0"], 1)
    assert _recompute_plan(1, 12, 32760, 128, 128, 2, 1560) == (_OVERLAPS["with_r0"], 2)
    assert _recompute_plan(1, 2, 256, 64, 64, 1, 64)[0] == _OVERLAPS["off"]         # values [k | v]: no pair
    assert _recompute_plan(1, 12, 32760, 32, 32, 2, 1560)[0] == _OVERLAPS["start"]   # 32-wide heads: no pair
    fp8 = _recompute_plan(1, 12, 32760, 128, 128, 2, 1560, qk_fp8=True)              # R-step 0 with fp8 S: no pair
    assert fp8 == (_OVERLAPS["start"], 3)
