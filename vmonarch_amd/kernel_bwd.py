"""Backward of the flash-entropy attention through the C ABI (vmo_fea_bwd).

Mirrors _FlashEntropyAttention.backward of the reference (kernel.py:360-381): given the saved
q, k, v, o, lse, ent and the upstream grads (do, de) it returns (dq, dk, dv) in q.dtype.  Rows
>= n_valid are padding: their gradients are zero.
"""
import torch

from . import _lib


def _pad_features(t, width):
    return t if t.shape[-1] == width else torch.nn.functional.pad(t, (0, width - t.shape[-1]))


def fea_backward_raw(q, k, v, o, lse, ent, do, de, sm_scale, dq=None, dk=None, dv=None, overwrite="", v1=None,
                     fold_k=False, dk_base=None, dv_base=None, frames=1, dq_route=None, dq_base=None, delta=None):
    """q: (B, H, F*nq, D); k: (B, H, F*nk, D); v: (B, H, F*nk, Dv); o, do: (B, H, F*nq, Dv);
    lse, ent, de: (B, H, F*nq) fp32 with unit token stride.  Returns (dq, dk, dv).

    `frames` = F splits every (b, h) into F independent problems of nq queries and nk keys (frame f:
    rows [f nq, (f + 1) nq) and [f nk, (f + 1) nk)), read in place whatever the memory order.

    With `v1` (same shape and strides as v) the values are [v | v1], 2 Dv wide, read in place.

    A gradient passed in as a float32 view is accumulated into (+= in the kernels), or overwritten
    when its letter ("q", "k", "v") is in `overwrite`; one passed in q's dtype (a 16-bit view, any
    strides with a contiguous feature dim) is written; one not passed is returned as a new tensor of
    q's dtype.

    `fold_k` (v is k, as the VMonarch R-steps pass it): dk receives k's whole gradient, as key and
    as the first value columns, and dv only v1's (None without v1).

    `dq_base` / `dk_base` / `dv_base` (float32, shaped like dq / dk / dv): dq / dk / dv, in q's dtype, are
    that base plus this call's gradient (the last of several calls summing one gradient).

    `delta` ((B, H, F*nq) fp32, unit token stride): rowsum(o * do) when the caller has it (the L-step
    backward forms it); otherwise the kernels form it from o and do.

    `dq_route` ("recompute" or "ds"; None lets the library choose) picks how dq is formed: a pass that
    recomputes S and dP, or a GEMM over dS^T stored by the dk / dv pass (the workspace then holds nk x nq
    16-bit values per problem)."""
    route = {None: 0, "recompute": _lib.BWD_RECOMPUTE_DQ, "ds": _lib.BWD_DS_DQ}[dq_route]
    return _lib.host().fea_bwd(q, k, v, o, lse, ent, do, de, sm_scale, dq, dk, dv, overwrite, v1, fold_k, dk_base, dv_base,
                               frames, route, dq_base, delta)


def fea_backward(q, k, v, o, lse, ent, do, de, sm_scale, n_valid):
    B, H, N, D = q.shape
    Dv = v.shape[-1]
    n = int(n_valid)
    from .kernel import _kernel_widths
    Dk, Dvk = _kernel_widths(D, Dv)
    if not ((Dk in (32, 64, 128) and Dvk in (32, 64, 128, 256)) or (Dk == 16 and Dvk in (16, 32, 64, 128, 256))
            or (Dk == 256 and Dvk == 256)):
        raise NotImplementedError(f"vmonarch_amd: backward for head dims ({D}, {Dv}) is not built")
    if de is None:
        de = torch.zeros((B, H, N), device=q.device, dtype=torch.float32)
    if do is None:
        do = torch.zeros_like(o)
    do = do.to(q.dtype)
    de = de.float()
    if de.stride(2) != 1:
        de = de.contiguous()
    if n == N and Dk == D and Dvk == Dv:
        # no padding rows, no padded features: the kernels write the gradients once, in the memory order
        # of the caller's q, k, v (a DiT block's (B, N, H, D) buffers need no copy afterwards)
        return _lib.host().fea_attention_bwd(q, k, v, o, lse, ent, do, de, sm_scale)
    dq = torch.zeros_like(q)
    dk = torch.zeros_like(k)
    dv = torch.zeros_like(v)
    if n == 0:
        return dq, dk, dv
    sl = slice(0, n)
    qx, kx = (_lib.row_aligned(_pad_features(t[:, :, sl], Dk)) for t in (q, k))
    vx, ox, dox = (_lib.row_aligned(_pad_features(t[:, :, sl], Dvk)) for t in (v, o, do))
    lse_x, ent_x = lse[:, :, sl], ent[:, :, sl]
    de_x = de[:, :, sl]
    gq, gk, gv = fea_backward_raw(qx, kx, vx, ox, lse_x, ent_x, dox, de_x, sm_scale)
    dq[:, :, sl] = gq[..., :D]
    dk[:, :, sl] = gk[..., :D]
    dv[:, :, sl] = gv[..., :Dv]
    return dq, dk, dv
