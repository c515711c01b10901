"""FlashEntropyAttention: attention that also returns the entropy of every attention row.

Drop-in for video_monarch_attention/kernel.py (reference).  Same public function and autograd
contract; the body calls the gfx950 HIP kernels through the host module (csrc/host_ops.cpp).

Differences from the reference that callers can observe: none in values (within bf16
tolerance).  Internally there is no padding to a multiple of 128 (kernel.py:399-400): tails are
masked in the kernel, so no padded copies of q / k / v are made.
"""
import torch

from . import _lib

SEQ_ALIGN = 128  # kept for API parity with the reference (kernel.py:12); no padding happens
_HEAD_DIMS = {16, 32, 64, 128, 256}  # accepted by the reference (kernel.py:324)


def _pad_features(t, width):
    """Zero-pad the feature dim to `width` (a zero feature changes neither q.k nor P.v)."""
    if t.shape[-1] == width:
        return t
    return torch.nn.functional.pad(t, (0, width - t.shape[-1]))


def _kernel_widths(d, dv):
    """Head dims of the flash-entropy kernels (forward and backward) that serve (d, dv): every pair the reference
    accepts (dv a multiple of d) as it is, 16-wide heads included (their kernels hold 16-wide rows in 32-wide LDS
    tiles); a 16-wide value head under wider q / k (beyond the reference) runs 32 wide, zero-padded."""
    return d, (32 if dv < 32 <= d else dv)


def fea_forward(q, k, w0, w1, sm_scale, frames=1, o=None, lse=None, ent=None, want_ent=True, want_lse=True,
                num_splits=1, qk_fp8=False):
    """Launch the flash-entropy forward.

    q: (B, H, F*nq, D); k, w0: (B, H, F*nk, .); w1: optional second value tensor (requires w0 is k).
    Returns (o, lse, ent): o (B, H, F*nq, Dw0 + Dw1) in q.dtype; lse (log2 units) and ent (nats)
    (B, H, F*nq) fp32, or None when not wanted.  o / lse / ent may be passed in as (strided) views
    to write into; lse / ent views need a unit token stride.  `qk_fp8`: S = q k^T in fp8 (the VMonarch
    R-step variants only; vmo_fea_fwd_args.qk_fp8).
    """
    return _lib.host().fea_fwd(q, k, w0, w1, sm_scale, frames, o, lse, ent, want_ent, want_lse, num_splits, bool(qk_fp8))


class _FlashEntropyAttention(torch.autograd.Function):
    """Autograd contract of the reference (kernel.py:316-381):
    forward(ctx, q, k, v, sm_scale, n_valid, warp_specialize) -> (o, E);
    backward(ctx, do, de) -> (dq, dk, dv, None, None, None).
    Rows >= n_valid are padding: they are masked as keys and their outputs are zero
    (kernel.py:352-353)."""

    @staticmethod
    def forward(ctx, q, k, v, sm_scale, n_valid, warp_specialize):
        B, H, N, D = q.shape
        Dv = v.shape[-1]
        assert q.dtype in _lib.DTYPES, f"unsupported dtype {q.dtype}"
        assert k.dtype == v.dtype == q.dtype, f"q, k and v of one dtype, got {q.dtype}, {k.dtype} and {v.dtype}"
        assert k.shape == q.shape and v.shape[:-1] == q.shape[:-1]
        assert D in _HEAD_DIMS and Dv in _HEAD_DIMS
        if D == 256 and Dv != 256:
            raise NotImplementedError("vmonarch_amd: head dim 256 for q/k is built with 256-wide values only")
        if not q.is_cuda:
            raise RuntimeError("vmonarch_amd: flash_entropy_attention needs GPU tensors (no CPU path)")
        assert k.device == v.device == q.device, f"q, k and v on one GPU, got {q.device}, {k.device} and {v.device}"
        n = int(n_valid)
        Dk, Dvk = _kernel_widths(D, Dv)
        ctx.sm_scale = sm_scale
        ctx.n_valid = n
        if n == N and Dvk == Dv:   # no padding rows, no padded features
            o, ent, lse = _lib.host().fea_attention(q, k, v, sm_scale)
            ctx.save_for_backward(q, k, v, o, lse, ent)
            return o, ent
        qx, kx, vx = (_lib.row_aligned(_pad_features(t[:, :, :n], w)) for t, w in ((q, Dk), (k, Dk), (v, Dvk)))
        ent = torch.empty((B, H, N), device=q.device, dtype=torch.float32)
        lse = torch.empty((B, H, N), device=q.device, dtype=torch.float32)
        if Dvk == Dv:
            o = _lib.empty_in_layout(q, Dv, q.dtype)   # o in the caller's layout (e.g. (B, N, H, Dv))
            if n > 0:
                fea_forward(qx, kx, vx, None, sm_scale, o=o[:, :, :n], lse=lse[:, :, :n], ent=ent[:, :, :n])
        else:
            o_k = torch.empty((B, H, N, Dvk), device=q.device, dtype=q.dtype)
            if n > 0:
                fea_forward(qx, kx, vx, None, sm_scale, o=o_k[:, :, :n], lse=lse[:, :, :n], ent=ent[:, :, :n])
            o = _lib.empty_in_layout(q, Dv, q.dtype).copy_(o_k[..., :Dv])   # the caller's layout, as above
        if n < N:   # padding rows (kernel.py:352-353)
            o[:, :, n:] = 0
            ent[:, :, n:] = 0
            lse[:, :, n:] = 0
        ctx.save_for_backward(q, k, v, o, lse, ent)
        return o, ent

    @staticmethod
    def backward(ctx, do, de):
        from .kernel_bwd import fea_backward
        q, k, v, o, lse, ent = ctx.saved_tensors
        dq, dk, dv = fea_backward(q, k, v, o, lse, ent, do, de, ctx.sm_scale, ctx.n_valid)
        return dq, dk, dv, None, None, None


def _recorded(*tensors):
    """Whether something records the call: autograd, a functorch transform, forward-mode AD or torch.jit's tracer (which
    would see the host module's allocations only)."""
    return ((torch.is_grad_enabled() and any(t.requires_grad for t in tensors))
            or torch._C._are_functorch_transforms_active() or torch.autograd.forward_ad._current_level >= 0
            or torch._C._get_tracing_state() is not None)


def _plain_call(q, k, v):
    """Whether flash_entropy_attention can go straight to the kernels: nothing records the call (autograd's function,
    ~12 us of host time, is then only passed through), and inputs that its forward takes as they are (the host module
    asks for one dtype and device itself)."""
    if _recorded(q, k, v):
        return False
    if not (type(q) is type(k) is type(v) is torch.Tensor and q.is_cuda and q.dim() == 4):
        return False
    D, Dv = q.shape[-1], v.shape[-1]
    return (q.dtype in _lib.DTYPES and k.shape == q.shape and v.shape[:-1] == q.shape[:-1] and D in _HEAD_DIMS
            and Dv in _HEAD_DIMS and not (D == 256 and Dv != 256) and _kernel_widths(D, Dv) == (D, Dv))


def flash_entropy_attention(q, k, v, sm_scale=None, warp_specialize=True):
    """
    Non-causal attention that also returns the entropy of every attention row
    (reference: kernel.py:384-402; `warp_specialize` is accepted and ignored).

    Args:
        q, k: (B, H, N, D)
        v: (B, H, N, Dv)
        sm_scale: softmax scale, defaults to 1 / sqrt(D)
    Returns:
        o: (B, H, N, Dv) = softmax(sm_scale * q k^T) v, in q.dtype
        e: (B, H, N) float32, e_i = -sum_j P_ij log P_ij
    """
    n = q.shape[-2]
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    if _plain_call(q, k, v):
        return _lib.host().fea_attention(q, k, v, sm_scale)[:2]
    return _FlashEntropyAttention.apply(q, k, v, sm_scale, n, warp_specialize)
