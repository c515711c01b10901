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
