"""The one-block-per-wave multi-block L-step backward (csrc/lstep_mb.hip) around its row blocks: one row into the third
and fourth block, one short of them, in fp16, with an upstream gradient laid out as a (B, N, H, D) buffer; against the
oracle at the tolerance of the other L-step gradients (2e-2 of the largest element: operands rounded to 11 bits, sums
of at most 128 terms in fp32)."""
import pytest
import torch

from conftest import assert_close_ref, randn_lp
from oracle import lstep_grad

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("last", [False, True])
@pytest.mark.parametrize("m, d, dv", [(66, 128, 128), (95, 64, 64), (97, 128, 128), (127, 128, 64), (127, 64, 128),
                                      (31, 32, 32), (63, 16, 16), (95, 32, 64), (97, 16, 16)])
def test_lstep_backward_at_block_edges(m, d, dv, last):
    from vmonarch_amd.vmonarch import _lstep_bwd_launch
    g = torch.Generator().manual_seed(m + d + dv)
    B, H, b = 2, 2, 7
    N, wout, gw = m * b, d + (dv if last else 0), dv if last else d
    q = randn_lp(g, B, H, N, d, dtype=torch.float16)
    out = randn_lp(g, B, H, N, wout, scale=0.5, dtype=torch.float16)
    ent = torch.rand(B, H, N, generator=g) * 3.0
    grad = randn_lp(g, B, H, N, gw, dtype=torch.float16)
    skip = 2 * b + 3 if last else 0   # whole rows and part of the next
    dq0 = torch.randn(B, H, N, d, generator=g)
    dq, dout = dq0.to(DEV), torch.empty((B, H, N, wout), device=DEV, dtype=q.dtype)
    gd = grad.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)
    print(f"lstep_bwd blocks m={m} d={d} dv={dv} last={last}", flush=True)
    _lstep_bwd_launch(q.to(DEV), out.to(DEV), ent.to(DEV), gd, dq, dout, m, b, d ** -0.5, last, skip, 0.3)
    torch.cuda.synchronize()
    r5 = lambda t: t.float().numpy().reshape(B, H, m, b, -1)   # noqa: E731
    gg = grad.float().numpy().copy()
    gg[:, :, :skip] = 0.0
    dq_ref, dout_ref = lstep_grad(r5(q), r5(out), -ent.numpy().reshape(B, H, m, b), d ** -0.5, last,
                                  gg.reshape(B, H, m, b, -1), 0.3)
    assert_close_ref((dq.cpu() - dq0).numpy(), dq_ref.reshape(B, H, N, d), 2e-2)
    assert_close_ref(dout.float().cpu().numpy(), dout_ref.reshape(B, H, N, wout), 2e-2)


# the last step's delta = rowsum(out * d out): one block per wave up to three and four blocks, two blocks (whole and
# compact tiles), narrow heads (16-wide rows held twice) and unequal pairs; partial last blocks
@pytest.mark.parametrize("d, dv, m, dtype", [
    (128, 128, 33, torch.bfloat16), (128, 128, 41, torch.float16), (128, 128, 64, torch.bfloat16),
    (128, 128, 65, torch.bfloat16), (128, 128, 96, torch.float16), (128, 128, 97, torch.bfloat16),
    (128, 128, 128, torch.float16), (64, 64, 48, torch.float16), (64, 128, 70, torch.bfloat16),
    (128, 32, 50, torch.bfloat16), (32, 32, 7, torch.float16), (16, 16, 40, torch.bfloat16), (16, 16, 100, torch.float16)])
def test_multi_block_last_step_delta(d, dv, m, dtype):
    """Against the sum over the stored 16-bit d out in float64: at most d + dv fp32 steps of rounding 2^-24 each apart,
    256 x 2^-24 = 1.5e-5 of the sum of magnitudes; d out and dq as without it."""
    from vmonarch_amd.vmonarch import _lstep_bwd_launch
    g = torch.Generator().manual_seed(d + dv + m)
    B, H, b = 1, 2, 5
    N, skip = m * b, 7
    q, out = randn_lp(g, B, H, N, d, dtype=dtype).to(DEV), randn_lp(g, B, H, N, d + dv, dtype=dtype).to(DEV)
    ent, grad = (torch.rand(B, H, N, generator=g) * 3.0).to(DEV), randn_lp(g, B, H, N, dv, dtype=dtype).to(DEV)
    print(f"multi-block delta d={d} dv={dv} m={m} {dtype}", flush=True)
    res = []
    for delta in (None, torch.full((B, H, N), float("nan"), device=DEV)):
        dq, dout = torch.zeros(B, H, N, d, device=DEV), torch.empty_like(out)
        _lstep_bwd_launch(q, out, ent, grad, dq, dout, m, b, d ** -0.5, True, skip, 0.01, delta=delta)
        res.append((dq, dout))
    assert torch.equal(res[0][0], res[1][0]) and torch.equal(res[0][1], res[1][1])
    prod = out.double() * dout.double()
    assert bool(((delta.double() - prod.sum(-1)).abs() <= 256 * 2.0 ** -24 * prod.abs().sum(-1)).all())
