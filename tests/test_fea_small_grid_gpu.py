"""The key-group flash-entropy forward (csrc/fea_fwd_ks.hip), taken by launches of at most 256 query tiles with at least
512 keys: the same problems as the first heads of a launch with many more (which the 128-query kernel takes), and
against the oracle.  The two kernels weigh the same p = 2^(s c - m) bit for bit and add them in another order: their
fp32 sums of n terms differ by a few n^0.5 2^-24 relative (n <= 1100: under 1e-5 for lse and entropy), and o by one
rounding to the 16-bit type where that moves it across a rounding boundary."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import randn_lp
from oracle import entropy_attention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# tiles of 32 or 64 queries; keys at the shortest taken, one more, a 32-key remainder and most of a stage
@pytest.mark.parametrize("D, Dv, values_k", [(64, 64, False), (64, 128, False), (128, 128, False), (64, 64, True),
                                             (64, 128, True), (128, 128, True), (128, 256, True)])
@pytest.mark.parametrize("H, nq, nk, dtype, planted", [(2, 77, 512, torch.bfloat16, False), (3, 513, 513, torch.float16, False),
                                                       (2, 1000, 799, torch.bfloat16, False), (4, 1100, 1024, torch.float16, False),
                                                       (2, 200, 700, torch.bfloat16, True), (2, 200, 700, torch.float16, True)])
def test_key_group_forward(D, Dv, values_k, H, nq, nk, dtype, planted):
    """`planted`: a key far into the row (another key group than the first) ~120 (bf16) / 38 (fp16) log2 units above
    the first 32 keys, which takes the exact two-pass path."""
    _key_group_forward(D, Dv, values_k, H, nq, nk, dtype, planted, 1, 256)


# several frames per head, each a problem of its own; 86 heads of them are more than 256 tiles
@pytest.mark.parametrize("D, Dv, values_k", [(64, 64, False), (128, 128, True), (64, 128, True)])
@pytest.mark.parametrize("H, nq, nk, dtype, planted", [(2, 77, 513, torch.bfloat16, False), (3, 200, 700, torch.float16, True)])
def test_key_group_forward_of_several_frames(D, Dv, values_k, H, nq, nk, dtype, planted):
    _key_group_forward(D, Dv, values_k, H, nq, nk, dtype, planted, 3, 86)


def _query_tile(q, k, w0, w1, frames):
    """Queries per workgroup of the kernel that fea_forward takes for these inputs (with the entropy)."""
    from vmonarch_amd import _lib
    a = _lib.FeaFwdArgs()
    a.dtype, a.batch, a.heads, a.frames = _lib.DTYPES[q.dtype], q.shape[0], q.shape[1], frames
    a.nq, a.nk = q.shape[2] // frames, k.shape[2] // frames
    a.d, a.dw0, a.dw1 = q.shape[3], w0.shape[3], 0 if w1 is None else w1.shape[3]
    a.q, a.k, a.w0, a.o = (_lib.view(t) for t in (q, k, w0, q))
    if w1 is not None:
        a.w1 = _lib.view(w1)
    a.ent, a.sm_scale, a.num_splits = q.data_ptr(), 1.0, 1
    return _lib.lib().vmo_fea_fwd_query_tile(ctypes.byref(a))


def _key_group_forward(D, Dv, values_k, H, nq, nk, dtype, planted, F, big):
    """big: heads of the launch that the 128-query kernel takes, more than 256 tiles of 64."""
    from vmonarch_amd.kernel import fea_forward
    g = torch.Generator().manual_seed(D + Dv + nk + H)
    q, k = (randn_lp(g, 1, big, F * n, D, scale=0.5, dtype=dtype) for n in (nq, nk))
    w1 = randn_lp(g, 1, big, F * nk, Dv - D if values_k else Dv, dtype=dtype) if Dv > D or not values_k else None
    sm = D ** -0.5
    if planted:
        kf = k.unflatten(2, (F, nk))
        kf[:, :, :, nk - 90] = 0
        kf[:, :, :, nk - 90, 0] = 16.0
        q[:, :, :, 0] = (120 if dtype == torch.bfloat16 else 38) * np.log(2) / (16.0 * sm)
        kf[:, :, :, :32, 0] = 0
    # (B, N, H, D) buffers viewed as (B, H, N, D): the small launch reads them with another batch's strides
    qd, kd = (t.to(DEV).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k))
    wd = None if w1 is None else w1.to(DEV).transpose(1, 2).contiguous().transpose(1, 2)
    args = lambda h: (qd[:, :h], kd[:, :h], kd[:, :h] if values_k else wd[:, :h],   # noqa: E731
                      wd[:, :h] if values_k and wd is not None else None, sm)
    print(f"key groups D={D} Dv={Dv} values_k={values_k} H={H} {F}x{nq}x{nk} {dtype} planted={planted}", flush=True)
    assert _query_tile(*args(H)[:4], F) in (32, 64) and _query_tile(*args(big)[:4], F) == 128
    o, lse, ent = fea_forward(*args(H), frames=F)
    o_big, lse_big, ent_big = (t[:, :H] for t in fea_forward(*args(big), frames=F))
    step = 2.0 ** (-7 if dtype == torch.bfloat16 else -10)
    assert ((o.float() - o_big.float()).abs() <= step * o_big.float().abs() + 1e-5).all()
    assert (o != o_big).float().mean() < 0.02
    torch.testing.assert_close(lse, lse_big, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(ent, ent_big, rtol=1e-5, atol=2e-4 if planted else 2e-5)
    w = k[:, :H] if values_k and w1 is None else torch.cat([k[:, :H], w1[:, :H]], -1) if values_k else w1[:, :H]
    o_ref, e_ref = entropy_attention(*(t.unflatten(2, (F, -1)).float().numpy() for t in (q[:, :H], k[:, :H], w)), sm)
    np.testing.assert_allclose(o.unflatten(2, (F, -1)).float().cpu().numpy(), o_ref, atol=2e-2, rtol=1e-2)
    np.testing.assert_allclose(ent.unflatten(2, (F, -1)).cpu().numpy(), e_ref, atol=2e-2, rtol=1e-2)
